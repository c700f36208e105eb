// The dense route of the eigensolver (H_eff of at most 1000 entries): the
// matrix itself and its lowest eigenpair.
//
// dense_heff: every element of H_eff straight from the environment and MPO
// blocks,
//   H[(a0', a2', s1', s2'), (a0, a2, s1, s2)] =
//     sum over bond values of L_b(a0', a0) W(s1', s1) W(s2', s2) R_c(a2', a2),
// in one launch (a job per pair of wavefunction blocks, its terms enumerated
// on the host).  The matvec applied to every unit vector took 4 launches and
// some 60 us for each of the n columns.
//
// hermitian_lowest: Lanczos with full reorthogonalisation and no restart on
// the dense matrix, to an invariant subspace if need be (at most n steps),
// until the lowest Ritz residual is at rounding level: only one pair is asked
// for, where rocSOLVER's zheevd computes n, fails its check on many of these
// matrices and leaves them to zheevj.  Two launches per step: the product (a
// wave per row, bound by reading the matrix from the caches) and the
// projections (one workgroup, bound by reading the basis twice).
// iDMRG growth of a spin chain to chi=48, eight steps of which seven take
// this route with up to 900 entries: 545 -> 23 ms.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <limits>

#include "solvers.hpp"

namespace cam {

namespace {

struct DenseTerm {
  const double2 *L, *W1, *W2, *R;
  int64_t ldl, ldw1, ldw2, ldr;
};
struct DenseJob {
  int64_t row, col;            // first element of the block pair
  int32_t m0, m3, n1, n2;      // row block: a0', a2', s1', s2'
  int32_t k0, k3, k1, k2;      // column block: a0, a2, s1, s2
  int32_t term0, nterm;
};

__device__ __forceinline__ double2 mul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

__global__ __launch_bounds__(256) void dense_heff_kernel(const DenseJob* __restrict__ jobs,
                                                         const DenseTerm* __restrict__ terms, int njobs,
                                                         double2* __restrict__ A, int64_t n) {
  for (int jb = blockIdx.y; jb < njobs; jb += gridDim.y) {
    const DenseJob J = jobs[jb];
    const int64_t rows = int64_t(J.m0) * J.m3 * J.n1 * J.n2, tot = rows * J.k0 * J.k3 * J.k1 * J.k2;
    for (int64_t e = blockIdx.x * int64_t(256) + threadIdx.x; e < tot; e += int64_t(gridDim.x) * 256) {
      const int64_t i = e % rows, j = e / rows;
      const int a0 = static_cast<int>(i % J.m0), a2 = static_cast<int>(i / J.m0 % J.m3);
      const int s1 = static_cast<int>(i / (int64_t(J.m0) * J.m3) % J.n1);
      const int s2 = static_cast<int>(i / (int64_t(J.m0) * J.m3 * J.n1));
      const int c0 = static_cast<int>(j % J.k0), c2 = static_cast<int>(j / J.k0 % J.k3);
      const int t1 = static_cast<int>(j / (int64_t(J.k0) * J.k3) % J.k1);
      const int t2 = static_cast<int>(j / (int64_t(J.k0) * J.k3 * J.k1));
      double2 s = make_double2(0.0, 0.0);
      for (int t = J.term0; t < J.term0 + J.nterm; ++t) {
        const DenseTerm T = terms[t];
        const double2 w = mul(T.W1[s1 + t1 * T.ldw1], T.W2[s2 + t2 * T.ldw2]);
        const double2 p = mul(mul(T.L[a0 + c0 * T.ldl], w), T.R[a2 + c2 * T.ldr]);
        s.x += p.x;
        s.y += p.y;
      }
      A[J.row + i + (J.col + j) * n] = s;
    }
  }
}

__device__ __forceinline__ double wsum(double x) {
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  return x;
}

// w = A v for Hermitian A: w_i = sum_k conj(A[k, i]) v_k, a wave per row
__global__ __launch_bounds__(256) void hermitian_matvec_kernel(const double2* __restrict__ A, int n,
                                                               const double2* __restrict__ v,
                                                               double2* __restrict__ w) {
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (i >= n) return;
  const double2* a = A + static_cast<int64_t>(i) * n;
  double re = 0, im = 0;
  for (int k = lane; k < n; k += 64) {
    const double2 x = a[k], y = v[k];
    re += x.x * y.x + x.y * y.y;
    im += x.x * y.y - x.y * y.x;
  }
  re = wsum(re);
  im = wsum(im);
  if (lane == 0) w[i] = make_double2(re, im);
}

constexpr int kOrthThreads = 1024;

// Step j of the recurrence: w (n entries) projected off v_{j-1}, v_j, then
// off the whole basis, and normalised into v_{j+1}.  ab[2 j] = alpha_j,
// ab[2 j + 1] = beta_j, zero when the space is invariant.
__global__ __launch_bounds__(kOrthThreads) void lanczos_step_kernel(double2* __restrict__ V, int n, int j,
                                                                    const double2* __restrict__ w0,
                                                                    double* __restrict__ ab) {
  __shared__ double2 w[kSparseThreshold], coef[kSparseThreshold];
  __shared__ double part[kOrthThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int r = tid; r < n; r += kOrthThreads) w[r] = w0[r];
  __syncthreads();
  double alpha = 0.0;
  for (int pass = 0; pass < 2; ++pass) {
    const int i0 = pass == 0 ? max(j - 1, 0) : 0;
    for (int i = i0 + wave; i <= j; i += kOrthThreads / 64) {
      const double2* v = V + static_cast<int64_t>(i) * n;
      double re = 0, im = 0;
      for (int r = lane; r < n; r += 64) {
        const double2 x = v[r], y = w[r];
        re += x.x * y.x + x.y * y.y;
        im += x.x * y.y - x.y * y.x;
      }
      re = wsum(re);
      im = wsum(im);
      if (lane == 0) coef[i] = make_double2(re, im);
    }
    __syncthreads();
    for (int r = tid; r < n; r += kOrthThreads) {
      double2 y = w[r];
      for (int i = i0; i <= j; ++i) {
        const double2 p = mul(V[r + static_cast<int64_t>(i) * n], coef[i]);
        y.x -= p.x;
        y.y -= p.y;
      }
      w[r] = y;
    }
    alpha += coef[j].x;
    __syncthreads();
  }
  double s = 0.0;
  for (int r = tid; r < n; r += kOrthThreads) s += w[r].x * w[r].x + w[r].y * w[r].y;
  s = wsum(s);
  if (lane == 0) part[wave] = s;
  __syncthreads();
  s = 0.0;
  for (int q = 0; q < kOrthThreads / 64; ++q) s += part[q];
  double beta = sqrt(s);
  const bool end = j + 1 >= n || beta <= 16 * 2.220446049250313e-16 * fmax(1.0, fabs(alpha));
  const double inv = end ? 0.0 : 1.0 / beta;
  if (tid == 0) {
    ab[2 * j] = alpha;
    ab[2 * j + 1] = end ? 0.0 : beta;
  }
  if (j + 1 < n)
    for (int r = tid; r < n; r += kOrthThreads)
      V[r + static_cast<int64_t>(j + 1) * n] = make_double2(w[r].x * inv, w[r].y * inv);
}

// x = V s over k basis vectors
__global__ void ritz_vector_kernel(const double2* __restrict__ V, int n, int k, const double* __restrict__ s,
                                   double2* __restrict__ x) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  double2 y = make_double2(0.0, 0.0);
  for (int i = 0; i < k; ++i) {
    const double2 v = V[r + static_cast<int64_t>(i) * n];
    y.x += s[i] * v.x;
    y.y += s[i] * v.y;
  }
  x[r] = y;
}

// |y - e x|^2, |x|^2 and <x, y> (one workgroup)
__global__ __launch_bounds__(1024) void residual_kernel(const double2* __restrict__ x, const double2* __restrict__ y,
                                                        int n, double e, double* __restrict__ out) {
  __shared__ double part[3][16];
  double a = 0, b = 0, c = 0;
  for (int r = threadIdx.x; r < n; r += 1024) {
    const double2 u = x[r], v = y[r];
    const double dx = v.x - e * u.x, dy = v.y - e * u.y;
    a += dx * dx + dy * dy;
    b += u.x * u.x + u.y * u.y;
    c += u.x * v.x + u.y * v.y;
  }
  a = wsum(a);
  b = wsum(b);
  c = wsum(c);
  if ((threadIdx.x & 63) == 0) {
    part[0][threadIdx.x >> 6] = a;
    part[1][threadIdx.x >> 6] = b;
    part[2][threadIdx.x >> 6] = c;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    double t = 0;
    for (int q = 0; q < 16; ++q) t += part[threadIdx.x][q];
    out[threadIdx.x] = t;
  }
}

}  // namespace

// Lowest eigenvalue of the symmetric tridiagonal matrix (a, b): bisection on
// the Sturm count, then its vector by inverse iteration with partial
// pivoting.
double tridiagonal_lowest(const std::vector<double>& a, const std::vector<double>& b, std::vector<double>& vec) {
  const int k = static_cast<int>(a.size());
  CAM_REQUIRE(k >= 1 && static_cast<int>(b.size()) >= k - 1, "tridiagonal eigenproblem: sizes");
  const double eps = std::numeric_limits<double>::epsilon();
  double lo = HUGE_VAL, hi = HUGE_VAL, nrm = 0.0;
  for (int i = 0; i < k; ++i) {
    const double r = (i ? std::fabs(b[i - 1]) : 0.0) + (i + 1 < k ? std::fabs(b[i]) : 0.0);
    CAM_REQUIRE(std::isfinite(a[i]) && std::isfinite(r), "tridiagonal eigenproblem: not finite");
    lo = std::min(lo, a[i] - r);
    hi = std::min(hi, a[i]);              // the lowest eigenvalue is at most every diagonal entry
    nrm = std::max(nrm, std::fabs(a[i]) + r);
  }
  // squares of the entries stay in range
  const int scale = nrm > 0.0 ? std::ilogb(nrm) : 0;
  if (std::abs(scale) > 400) {
    std::vector<double> sa(a), sb(b);
    for (double& x : sa) x = std::ldexp(x, -scale);
    for (double& x : sb) x = std::ldexp(x, -scale);
    return std::ldexp(tridiagonal_lowest(sa, sb, vec), scale);
  }
  const double tiny = std::max(eps * eps * nrm, std::numeric_limits<double>::min());
  auto below = [&](double x) {            // whether an eigenvalue is < x
    double d = a[0] - x;
    if (d < 0.0) return true;
    for (int i = 1; i < k; ++i) {
      d = a[i] - x - b[i - 1] * b[i - 1] / (std::fabs(d) < tiny ? tiny : d);
      if (d < 0.0) return true;
    }
    return false;
  };
  hi += 2 * eps * nrm + tiny;
  lo -= 2 * eps * nrm + tiny;
  while (true) {
    const double mid = 0.5 * (lo + hi);
    if (mid <= lo || mid >= hi) break;
    (below(mid) ? hi : lo) = mid;
  }
  const double th = 0.5 * (lo + hi);
  // inverse iteration: L U of T - th with row interchanges
  std::vector<double> d(a), u(k, 0.0), u2(k, 0.0), l(k, 0.0);
  std::vector<char> sw(k, 0);
  for (int i = 0; i < k; ++i) d[i] -= th;
  for (int i = 0; i + 1 < k; ++i) u[i] = b[i];
  for (int i = 0; i + 1 < k; ++i) {
    const double s = b[i];
    if (std::fabs(d[i]) >= std::fabs(s)) {
      if (std::fabs(d[i]) < tiny) d[i] = tiny;
      l[i] = s / d[i];
      d[i + 1] -= l[i] * u[i];
    } else {
      sw[i] = 1;
      l[i] = d[i] / s;
      const double t = u[i];
      d[i] = s;
      u[i] = d[i + 1];
      d[i + 1] = t - l[i] * d[i + 1];
      if (i + 2 < k) {
        u2[i] = u[i + 1];
        u[i + 1] = -l[i] * u[i + 1];
      }
    }
  }
  if (std::fabs(d[k - 1]) < tiny) d[k - 1] = tiny;
  vec.assign(k, 1.0);
  for (int i = 0; i < k; ++i) vec[i] = 1.0 + 0.5 * std::sin(1.7 * i);
  for (int it = 0; it < 4; ++it) {
    if (it)
      for (int i = 0; i + 1 < k; ++i) {
        if (sw[i]) std::swap(vec[i], vec[i + 1]);
        vec[i + 1] -= l[i] * vec[i];
      }
    for (int i = k - 1; i >= 0; --i) {
      double s = vec[i];
      if (i + 1 < k) s -= u[i] * vec[i + 1];
      if (i + 2 < k) s -= u2[i] * vec[i + 2];
      vec[i] = s / d[i];
      if (std::fabs(vec[i]) > 1e200)
        for (double& x : vec) x *= 1e-200;
    }
    double mx = 0.0;
    for (double x : vec) mx = std::max(mx, std::fabs(x));
    double nn = 0.0;
    for (double& x : vec) {
      x /= mx;
      nn += x * x;
    }
    for (double& x : vec) x /= std::sqrt(nn);
  }
  return th;
}

void dense_heff(Heff& H, cplx* A) {
  hipStream_t s = H.ctx->stream;
  const double2* Lb = reinterpret_cast<const double2*>(H.L->data.get());
  const double2* Wb = reinterpret_cast<const double2*>(H.W->data.get());
  const double2* Rb = reinterpret_cast<const double2*>(H.R->data.get());
  // MPO views by (left bond value, ket sector)
  struct WV { int64_t br; int sp; const WMat* m; };
  std::map<std::pair<int64_t, int64_t>, std::vector<WV>> wby;
  for (const auto& kv : H.Wv)
    wby[{kv.first[0], kv.first[3]}].push_back(WV{kv.first[1], static_cast<int>(kv.first[2]), &kv.second});
  std::map<std::pair<int, int>, std::vector<DenseTerm>> pairs;     // (row block, column block) -> terms
  for (size_t q = 0; q < H.pblocks.size(); ++q) {
    const Heff::PB& P = H.pblocks[q];
    for (int64_t b = 0; b < H.w; ++b) {
      const auto li = H.Lv.find({b, P.s0});
      if (li == H.Lv.end()) continue;
      const auto w1 = wby.find({b, P.s1});
      if (w1 == wby.end()) continue;
      for (const WV& u : w1->second) {
        const auto w2 = wby.find({u.br, P.s2});
        if (w2 == wby.end()) continue;
        for (const WV& v : w2->second) {
          const auto ri = H.Rv.find({v.br, P.s3});
          if (ri == H.Rv.end()) continue;
          const auto pit = H.pindex.find({li->second.sout, ri->second.sout, u.sp, v.sp});
          CAM_REQUIRE(pit != H.pindex.end(), "heff: output block outside the allowed space (flux)");
          pairs[{pit->second, static_cast<int>(q)}].push_back(
              DenseTerm{Lb + li->second.off, Wb + u.m->off, Wb + v.m->off, Rb + ri->second.off, li->second.ld,
                        u.m->ld, v.m->ld, ri->second.ld});
        }
      }
    }
  }
  std::vector<DenseJob> jobs;
  std::vector<DenseTerm> terms;
  for (const auto& kv : pairs) {
    const Heff::PB &O = H.pblocks[kv.first.first], &P = H.pblocks[kv.first.second];
    DenseJob j{};
    j.row = O.off;
    j.col = P.off;
    j.m0 = static_cast<int32_t>(O.m0);
    j.m3 = static_cast<int32_t>(O.m3);
    j.n1 = static_cast<int32_t>(O.n1);
    j.n2 = static_cast<int32_t>(O.n2);
    j.k0 = static_cast<int32_t>(P.m0);
    j.k3 = static_cast<int32_t>(P.m3);
    j.k1 = static_cast<int32_t>(P.n1);
    j.k2 = static_cast<int32_t>(P.n2);
    j.term0 = static_cast<int32_t>(terms.size());
    j.nterm = static_cast<int32_t>(kv.second.size());
    terms.insert(terms.end(), kv.second.begin(), kv.second.end());
    jobs.push_back(j);
  }
  launch_zero(A, H.n * H.n * static_cast<int64_t>(sizeof(cplx)), s);
  if (jobs.empty()) return;
  DevBuf<DenseJob> dj(jobs.size());
  DevBuf<DenseTerm> dt(terms.size());
  dj.upload(jobs.data(), jobs.size(), s);
  dt.upload(terms.data(), terms.size(), s);
  hipLaunchKernelGGL(dense_heff_kernel, dim3(32, static_cast<unsigned>(std::min<size_t>(jobs.size(), 4096))),
                     dim3(256), 0, s, dj.get(), dt.get(), static_cast<int>(jobs.size()),
                     reinterpret_cast<double2*>(A), H.n);
  HIP_CHECK(hipGetLastError());
  HIP_CHECK(hipStreamSynchronize(s));
}

bool hermitian_lowest(Ctx& ctx, const cplx* A, int64_t n64, double* e, cplx* x) {
  const int n = static_cast<int>(n64);
  CAM_REQUIRE(n64 >= 1 && n64 <= kSparseThreshold, "hermitian_lowest: size out of range");
  hipStream_t s = ctx.stream;
  constexpr int kCheck = 12;                 // steps between convergence tests
  const int kmax = n;
  DevBuf<cplx> V(static_cast<size_t>(n) * std::min(n, 64)), w(static_cast<size_t>(n));
  DevBuf<double> ab(static_cast<size_t>(2 * n)), sv(static_cast<size_t>(n)), out(3);
  int cap = std::min(n, 64);
  launch_random_fill(V.get(), n, 0x5eedull, s);
  hipLaunchKernelGGL(residual_kernel, dim3(1), dim3(1024), 0, s, reinterpret_cast<const double2*>(V.get()),
                     reinterpret_cast<const double2*>(V.get()), n, 0.0, out.get());
  double h[3];
  HIP_CHECK(hipMemcpyAsync(h, out.get(), sizeof(h), hipMemcpyDeviceToHost, s));
  HIP_CHECK(hipStreamSynchronize(s));
  launch_scale(cplx{1.0 / std::sqrt(h[1]), 0.0}, V.get(), n, s);
  std::vector<double> hab(static_cast<size_t>(2 * n)), vec;
  const double eps = std::numeric_limits<double>::epsilon();
  int k = 0;
  bool done = false;
  while (!done) {
    const int k1 = std::min(kmax, k + kCheck);
    if (k1 + 1 > cap && cap < n) {           // the step after k1 writes vector k1
      const int grown = std::min(n, 2 * cap + kCheck);
      DevBuf<cplx> bigger(static_cast<size_t>(n) * grown);
      launch_copy(V.get(), bigger.get(), static_cast<int64_t>(n) * cap, s);
      HIP_CHECK(hipStreamSynchronize(s));
      V = std::move(bigger);
      cap = grown;
    }
    for (int j = k; j < k1; ++j) {
      double2* vp = reinterpret_cast<double2*>(V.get());
      hipLaunchKernelGGL(hermitian_matvec_kernel, dim3((n + 3) / 4), dim3(256), 0, s,
                         reinterpret_cast<const double2*>(A), n, vp + static_cast<int64_t>(j) * n,
                         reinterpret_cast<double2*>(w.get()));
      hipLaunchKernelGGL(lanczos_step_kernel, dim3(1), dim3(kOrthThreads), 0, s, vp, n, j,
                         reinterpret_cast<const double2*>(w.get()), ab.get());
    }
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipMemcpyAsync(hab.data(), ab.get(), 2 * k1 * sizeof(double), hipMemcpyDeviceToHost, s));
    HIP_CHECK(hipStreamSynchronize(s));
    std::vector<double> al, be;
    double nrm = 0.0;
    for (int j = 0; j < k1; ++j) {
      if (!std::isfinite(hab[2 * j]) || !std::isfinite(hab[2 * j + 1])) return false;
      al.push_back(hab[2 * j]);
      be.push_back(hab[2 * j + 1]);
      nrm = std::max(nrm, std::fabs(hab[2 * j]) + hab[2 * j + 1]);
      if (hab[2 * j + 1] == 0.0) {           // invariant
        done = true;
        break;
      }
    }
    k = static_cast<int>(al.size());
    *e = tridiagonal_lowest(al, be, vec);
    if (be[k - 1] * std::fabs(vec[k - 1]) <= 0.5 * eps * nrm) done = true;
    if (k == kmax) done = true;
  }
  sv.upload(vec.data(), vec.size(), s);
  hipLaunchKernelGGL(ritz_vector_kernel, dim3((n + 255) / 256), dim3(256), 0, s,
                     reinterpret_cast<const double2*>(V.get()), n, k, sv.get(), reinterpret_cast<double2*>(x));
  hipLaunchKernelGGL(hermitian_matvec_kernel, dim3((n + 3) / 4), dim3(256), 0, s, reinterpret_cast<const double2*>(A),
                     n, reinterpret_cast<const double2*>(x), reinterpret_cast<double2*>(w.get()));
  hipLaunchKernelGGL(residual_kernel, dim3(1), dim3(1024), 0, s, reinterpret_cast<const double2*>(x),
                     reinterpret_cast<const double2*>(w.get()), n, *e, out.get());
  HIP_CHECK(hipGetLastError());
  HIP_CHECK(hipMemcpyAsync(h, out.get(), sizeof(h), hipMemcpyDeviceToHost, s));
  HIP_CHECK(hipStreamSynchronize(s));
  double nrm = 0.0;
  for (int j = 0; j < k; ++j) nrm = std::max(nrm, std::fabs(hab[2 * j]) + hab[2 * j + 1]);
  if (!(std::sqrt(h[0]) <= 1e-13 * std::sqrt(double(n)) * nrm && std::fabs(h[1] - 1.0) <= 1e-12)) return false;
  *e = h[2] / h[1];                          // Rayleigh quotient
  launch_scale(cplx{1.0 / std::sqrt(h[1]), 0.0}, x, n, s);
  return true;
}

}  // namespace cam
