// Host-side rules of the library, driven from tests/test_host_rules.py: one
// command per line on stdin, one line of answer each.
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

int main() {
  const std::map<std::string, void (*)(std::istringstream&)> commands = {{"batches", batches}, {"bytes", bytes},
                                                                              {"inverse", inverse}};
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
