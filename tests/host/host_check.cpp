// Host-side rules of the library, driven from tests/test_host_rules.py: one
// command per line on stdin, one line of answer each.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <iostream>
#include <map>
#include <sstream>

#include "solvers.hpp"

using namespace cam;

// batches BYTES ITEMS VECTORS (M N)*: ends of the batches
static void batches(std::istringstream& in) {
  int64_t bytes, m, n;
  size_t items;
  int vectors;
  in >> bytes >> items >> vectors;
  std::vector<JacobiSize> s;
  while (in >> m >> n) s.push_back(JacobiSize{m, n});
  for (size_t e : jacobi_svd_batches(s, vectors != 0, bytes, items)) std::printf("%zu ", e);
  std::printf("\n");
}

// bytes VECTORS M N
static void bytes(std::istringstream& in) {
  int64_t m, n;
  int vectors;
  in >> vectors >> m >> n;
  std::printf("%lld\n", static_cast<long long>(jacobi_svd_bytes(m, n, vectors != 0)));
}

// inverse (CHARGE VALUE)*: inverses of a bond's values
static void inverse(std::istringstream& in) {
  QIndex bond;
  std::vector<double> v;
  int q;
  std::string x;
  while (in >> q >> x) {
    Charge c;
    c.q[0] = static_cast<int16_t>(q);
    bond.charges.push_back(c);
    v.push_back(std::strtod(x.c_str(), nullptr));
  }
  bond.size = static_cast<int64_t>(v.size());
  bond.build_sectors();
  for (double y : bond_inverse(bond, v)) std::printf("%.17g ", y);
  std::printf("\n");
}

// tridiagonal K A.. B..: lowest eigenvalue, then its vector
static void tridiagonal(std::istringstream& in) {
  size_t k;
  in >> k;
  auto read = [&](size_t n) {
    std::vector<double> v;
    std::string x;
    while (n--) {
      in >> x;
      v.push_back(std::strtod(x.c_str(), nullptr));
    }
    return v;
  };
  const std::vector<double> a = read(k), b = read(k - 1);
  std::vector<double> vec;
  std::printf("%.17g ", tridiagonal_lowest(a, b, vec));
  for (double x : vec) std::printf("%.17g ", x);
  std::printf("\n");
}

// Problems of a plan, "M N BATCH BETA NSEG K.." each: what computes its outputs
// (kernels in route order) and how often each output is computed at least and
// at most.  A problem after "+" is added when the lists have been built.
static void plan(std::istringstream& in) {
  GemmPlan p;
  std::string word;
  static char mem[1];
  int64_t at = 16;                          // addresses only name the operands here
  auto ptr = [&]() { return reinterpret_cast<char*>(mem) + (at += 16); };
  while (in >> word) {
    if (word == "+") {
      p.choose_tiles(1);
      p.build_tiles();
      continue;
    }
    int n, batch, beta, nseg, k;
    const int m = std::atoi(word.c_str());
    in >> n >> batch >> beta >> nseg;
    const int id = p.add_problem(ptr(), m, m, n, batch, int64_t(m) * n, beta);
    while (nseg--) {
      in >> k;
      p.add_segment(id, ptr(), m, int64_t(m) * k, ptr(), k, 0, k, 0);
    }
  }
  if (p.direct.empty()) {
    p.choose_tiles(1);
    p.build_tiles();
  }
  std::vector<std::vector<int>> times;
  for (const GemmProb& q : p.probs) times.emplace_back(static_cast<size_t>(q.M) * q.N * q.batch, 0);
  auto mark = [&](int prob, int b, int m0, int n0, int tm, int tn) {
    const GemmProb& q = p.probs[prob];
    for (int n = n0; n < std::min(q.N, n0 + tn); ++n)
      for (int m = m0; m < std::min(q.M, m0 + tm); ++m) times[prob][(size_t(b) * q.N + n) * q.M + m]++;
  };
  std::string route;
  if (!p.direct.empty()) {
    route = "direct";
    for (const GemmTile& t : p.direct) {
      int64_t steps = 0;
      const GemmProb& q = p.probs[t.prob];
      for (int s = q.seg0; s < q.seg0 + q.nseg; ++s) steps += (p.segs[s].K + 3) / 4;
      mark(t.prob, t.batch, t.m0, t.n0, 16, 16 * (steps <= 8 ? 8 : steps <= 16 ? 4 : steps <= 32 ? 2 : 1));
    }
  } else {
    for (int t = 0; t < kNumTileShapes; ++t)
      for (const GemmTile& g : p.tiles[1][t]) {
        route = "tiles";
        mark(g.prob, g.batch, g.m0, g.n0, kTileShapes[t].tm, kTileShapes[t].tn);
      }
    if (!p.rows.empty()) route += route.empty() ? "rows" : "+rows";
    for (const RowItem& it : p.rows)
      for (int n = it.out0; n < it.out0 + it.nout; ++n)
        for (int r = 0; r < it.rows; ++r) {
          const int64_t row = int64_t(it.m0) + r;
          const RowOut& o = p.row_out[n];
          for (size_t id = 0; id < p.probs.size(); ++id)
            if (reinterpret_cast<int64_t>(p.probs[id].C) == o.off)
              mark(static_cast<int>(id), static_cast<int>(it.batch0 + row / it.M), static_cast<int>(row % it.M), o.n, 1, 1);
        }
  }
  int lo = 1 << 30, hi = 0;
  for (const auto& v : times)
    for (int x : v) {
      lo = std::min(lo, x);
      hi = std::max(hi, x);
    }
  std::printf("%s %d %d\n", route.c_str(), lo, hi);
}

int main() {
  const std::map<std::string, void (*)(std::istringstream&)> commands = {{"batches", batches}, {"bytes", bytes},
                                                                              {"inverse", inverse},
                                                                              {"plan", plan},
                                                                              {"tridiagonal", tridiagonal}};
  std::string line, name;
  while (std::getline(std::cin, line)) {
    std::istringstream in(line);
    in >> name;
    try {
      commands.at(name)(in);
    } catch (const Error& e) {
      std::printf("error %s\n", e.what());
    }
  }
  return 0;
}
