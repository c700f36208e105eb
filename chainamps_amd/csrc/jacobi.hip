// One-sided Jacobi SVD of dense complex blocks, FP64 on the device.
//
// The full per-block decompositions of the blockwise SVD: A = U diag(S) Vh
// with min(m, n) triplets, S descending.  With B = A (or A^H when m < n),
// L x c, columns sorted by length:
//   B P = Q R          Householder QR
//   R^H V = W diag(S)  plane rotations from the right until the columns of
//                      X = R^H V are orthogonal
//   B = (Q V) diag(S) (P W)^H
// Every rotation is computed from the columns' current inner products, so
// the columns end orthogonal relative to their own lengths, however small.
// The QR step is there for the spectra of bond wavefunctions: on R^H the
// rotations need 6 to 9 sweeps, on B itself 15 to 33 (decaying or truncated
// spectra; blocks with repeated columns take a second QR, see kStallSweeps).
// A rotation's rounding drifts the columns' lengths by some 1e-16 each, so the
// singular values are |x_j| / |v_j| and both vectors are normalised at the end.
//
// Two forms:
//  - a block whose working set fits the 160 KB of LDS is decomposed by one
//    workgroup, all such blocks of a call in one launch.  16 lanes own a
//    column pair; a step (all disjoint pairs of a round-robin round) is
//    one pass over LDS and one barrier.  Bound by LDS bandwidth (X and V read
//    and written once per step) and the rotation's latency.
//  - a larger block goes through block Jacobi: column blocks of 16, a round
//    of disjoint block pairs at a time, all blocks of a call side by side.
//    Three launches per round: the pairs' 32 x 32 Gram matrices (MFMA, split
//    over row chunks), a two-sided rotation sweep over each in LDS, and the
//    update of X and V (MFMA).  Bound by the round's three launch latencies
//    and the rotation chain in LDS.
// rocSOLVER's zgesvd, which these replace, issues some 500 launches for a
// block of 60 columns and spends most of its time in a one-workgroup QR
// iteration.  Whole svd_truncate calls on one square block, decaying spectrum
// (random entries): 64 columns 9.0 -> 1.2 ms (15 -> 1.6), 100: 21 -> 2.9
// (35 -> 3.4), 384: 216 -> 12 (459 -> 15), 768: 609 -> 34 (1399 -> 44); the
// values' error at 384 falls from 1.8e-14 (8e-14) to 2e-15.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>
#include <numeric>

#include "solvers.hpp"

namespace cam {

namespace {

typedef double d4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// sum over the 16 lanes of a DPP row, in every lane of it
template <int kRor>
__device__ __forceinline__ double ror_add(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x120 + kRor, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x120 + kRor, 0xf, 0xf, true);
  return x + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double row_sum(double x) {
  x = ror_add<8>(x);
  x = ror_add<4>(x);
  x = ror_add<2>(x);
  return ror_add<1>(x);
}

// 1 / sqrt(x) and 1 / x from the hardware's approximation by two Newton steps
// (a few 1e-16; the library's versions spend several times the instructions
// on rounding the last bit, which the rotations do not need)
__device__ __forceinline__ double fast_rsqrt(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  double e = fma(-h, g, 0.5);
  g = fma(g, e, g);
  h = fma(h, e, h);
  e = fma(-h, g, 0.5);
  return 2.0 * fma(h, e, h);
}
__device__ __forceinline__ double fast_rcp(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = fma(fma(-x, y, 1.0), y, y);
  return fma(fma(-x, y, 1.0), y, y);
}

// The rotation that makes columns x_i, x_j with |x_i|^2 = a, |x_j|^2 = b and
// x_i^H x_j = g (h2 = |g|^2) orthogonal:
//   x_i' = c x_i - s e^{-i phi} x_j,   x_j' = s e^{i phi} x_i + c x_j
// (phi the phase of g); the longer result is to become column i.
struct Rot {
  double c;
  double2 s;     // s e^{i phi}
  bool swap;
};
__device__ __forceinline__ Rot rotation(double a, double b, double2 g, double h2) {
  const double ih = fast_rsqrt(h2);
  const double d = b - a, w = fma(d, d, 4.0 * h2);
  const double t = copysign(2.0 * h2 * ih, d) * fast_rcp(fabs(d) + w * fast_rsqrt(w));
  Rot r;
  r.c = fast_rsqrt(fma(t, t, 1.0));
  const double s = t * r.c * ih;
  r.s = make_double2(s * g.x, s * g.y);
  r.swap = b > a;
  return r;
}
// Columns of an exactly rank-deficient block fall by 1e-16 per reflector or
// rotation; squared lengths below kNull2 (the block's own is about one) count
// as zero, which keeps the products of two of them in range.
constexpr double kNull2 = 1e-120;
// whether a pair is not yet orthogonal to tol (tol2 = tol^2)
__device__ __forceinline__ bool needs_rotation(double a, double b, double h2, double tol2) {
  return h2 > tol2 * a * b && a > kNull2 && b > kNull2;
}
__device__ __forceinline__ void rotate(const Rot& r, double2& x, double2& y) {
  const double2 u = make_double2(r.c * x.x - (r.s.x * y.x + r.s.y * y.y), r.c * x.y - (r.s.x * y.y - r.s.y * y.x));
  const double2 v = make_double2(r.c * y.x + (r.s.x * x.x - r.s.y * x.y), r.c * y.y + (r.s.x * x.y + r.s.y * x.x));
  x = r.swap ? v : u;
  y = r.swap ? u : v;
}

// Orders the LDS accesses of a wave's lanes where one lane reads what another
// has just written: the hardware keeps a wave's LDS operations in order, this
// keeps the compiler from moving them (no instruction of its own).
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// round-robin: pair k of round `step` among n (even) players
__device__ __forceinline__ void round_robin(int n, int step, int k, int& lo, int& hi) {
  const int a = k == 0 ? n - 1 : (step + k) % (n - 1);
  const int b = (step - k + n - 1) % (n - 1);
  lo = min(a, b);
  hi = max(a, b);
}

// ---- blocks in LDS -----------------------------------------------------------

constexpr int kSmallThreads = 576;    // 16 lanes for each of up to 35 column pairs
constexpr int64_t kSmallLds = 152 * 1024;
constexpr int kSmallCols = 72;        // 2 c^2 entries of 16 bytes fit up to c = 69
constexpr int kSmallRows = 1024;
constexpr int kMaxSweeps = 40;
// Blocks (of the block form) whose rotations still meet scaled inner products
// above kStalled after this many sweeps start again from another QR.  They have
// columns that repeat others: the QR leaves some copies among the long columns
// of R^H, where the rotations shrink them by a digit a sweep (128 columns, 64
// different ones: 36 sweeps; 640 columns, 160 different ones: more than 40).
// The new QR takes the columns that the first one found dependent last, and
// entries changed in their last bit: equal columns would leave equal rounding
// errors, dependent again.  Then 8 to 10 sweeps do.  Other blocks end within 9.
constexpr int kStallSweeps = 12;
constexpr double kStalled = 1e-3;

struct SmallJob {
  const double2* A;      // m x n, column-major
  double2* U;            // m x k (null: values only)
  double2* Vh;           // k x n
  double2* work;         // L x c: R and the reflectors
  double* S;             // k
  int* info;
  int m, n;
  double scale;          // power of two applied to A
};

// One sweep over the column pairs: 16 lanes per pair, each holding up to R
// rows of both columns in registers between the inner products (over the
// first L of the ld rows) and the rotation.
template <int R>
__device__ void small_sweep(double2* sm, int L, int c, int ld, double tol2, int* rotated) {
  const int ce = c + (c & 1), np = ce / 2;
  const int grp = threadIdx.x >> 4, l = threadIdx.x & 15, ng = blockDim.x >> 4;
  for (int step = 0; step < ce - 1; ++step) {
    for (int k = grp; k < np; k += ng) {
      int p, q;
      round_robin(ce, step, k, p, q);
      if (q >= c) continue;
      double2* X = sm + p * ld;
      double2* Y = sm + q * ld;
      double2 x[R], y[R];
      double a = 0, b = 0, gr = 0, gi = 0;
#pragma unroll
      for (int t = 0; t < R; ++t) {
        const int r = l + 16 * t;
        if (r < ld) {
          x[t] = X[r];
          y[t] = Y[r];
        }
        if (r < L) {
          a += x[t].x * x[t].x + x[t].y * x[t].y;
          b += y[t].x * y[t].x + y[t].y * y[t].y;
          gr += x[t].x * y[t].x + x[t].y * y[t].y;
          gi += x[t].x * y[t].y - x[t].y * y[t].x;
        }
      }
      a = row_sum(a);
      b = row_sum(b);
      gr = row_sum(gr);
      gi = row_sum(gi);
      const double h2 = gr * gr + gi * gi;
      Rot rot;
      rot.c = 1.0;
      rot.s = make_double2(0.0, 0.0);
      rot.swap = b > a;
      const bool need = needs_rotation(a, b, h2, tol2);
      if (need) rot = rotation(a, b, make_double2(gr, gi), h2);
      if (need || rot.swap) {
#pragma unroll
        for (int t = 0; t < R; ++t) {
          const int r = l + 16 * t;
          if (r < ld) {
            rotate(rot, x[t], y[t]);
            X[r] = x[t];
            Y[r] = y[t];
          }
        }
        if (need && l == 0) *rotated = 1;
      }
    }
    __syncthreads();
  }
}

// Householder vector of column x (rows j.. of it, 16 lanes): x_j becomes
// v_j = x_j - beta, beta = -e^{i arg x_j} |x| goes to *diag, and *tau is such
// that (1 - tau v v^H) x = beta e_j.
__device__ __forceinline__ void householder(double2* x, int j, int L, int l, double2* diag, double* tau) {
  double w = 0.0;
  for (int r = j + l; r < L; r += 16) w += x[r].x * x[r].x + x[r].y * x[r].y;
  w = row_sum(w);
  const double2 al = x[j];
  const double nx = w > kNull2 ? sqrt(w) : 0.0, aa = w > kNull2 ? sqrt(al.x * al.x + al.y * al.y) : 0.0;
  const double2 ph = aa > 0.0 ? make_double2(al.x / aa, al.y / aa) : make_double2(1.0, 0.0);
  if (l == 0) {
    *diag = make_double2(-ph.x * nx, -ph.y * nx);
    *tau = nx > 0.0 ? 1.0 / (nx * (nx + aa)) : 0.0;
    x[j] = make_double2(ph.x * (aa + nx), ph.y * (aa + nx));
  }
}
// y <- (1 - tau v v^H) y over rows j.. (16 lanes); the caller may go on with
// rows of y that other lanes updated
__device__ __forceinline__ void reflect(const double2* v, double tau, double2* y, int j, int L, int l) {
  double gr = 0, gi = 0;
  for (int r = j + l; r < L; r += 16) {
    const double2 a = v[r], b = y[r];
    gr += a.x * b.x + a.y * b.y;
    gi += a.x * b.y - a.y * b.x;
  }
  gr = tau * row_sum(gr);
  gi = tau * row_sum(gi);
  for (int r = j + l; r < L; r += 16) {
    const double2 a = v[r];
    double2 b = y[r];
    b.x -= gr * a.x - gi * a.y;
    b.y -= gr * a.y + gi * a.x;
    y[r] = b;
  }
  wave_order();
}

constexpr int kRowsPerLane = 9;   // rows per lane of a pair the sweeps are compiled for

// entries of LDS the block needs: B, then X = R^H V with V below, then [V; 0]
__host__ __device__ inline int64_t small_entries(int64_t L, int64_t c) { return c * (L > 2 * c ? L : 2 * c); }

__global__ __launch_bounds__(kSmallThreads) void jacobi_small_kernel(const SmallJob* __restrict__ jobs) {
  extern __shared__ double2 sm[];
  __shared__ int rotated;
  __shared__ double sig[kSmallCols], rx[kSmallCols], rv[kSmallCols], tau[kSmallCols];
  __shared__ double2 diag[kSmallCols];
  __shared__ int rank[kSmallCols], perm[kSmallCols];
  const SmallJob J = jobs[blockIdx.x];
  const int tid = threadIdx.x, nt = blockDim.x;
  const bool tr = J.m < J.n;
  const int L = tr ? J.n : J.m, c = tr ? J.m : J.n;
  const int grp = tid >> 4, l = tid & 15, ng = nt >> 4;
  // B's columns by falling length
  for (int k = grp; k < c; k += ng) {
    double w = 0.0;
    for (int r = l; r < L; r += 16) {
      const double2 v = J.A[tr ? k + static_cast<int64_t>(r) * J.m : r + static_cast<int64_t>(k) * J.m];
      const double x = v.x * J.scale, y = v.y * J.scale;
      w += x * x + y * y;
    }
    w = row_sum(w);
    if (l == 0) sig[k] = w;
  }
  __syncthreads();
  for (int k = tid; k < c; k += nt) {
    int r = 0;
    for (int j = 0; j < c; ++j) r += sig[j] > sig[k] || (sig[j] == sig[k] && j < k);
    rank[k] = r;
    perm[r] = k;
  }
  __syncthreads();
  for (int e = tid; e < J.m * J.n; e += nt) {
    const int i = e % J.m, j = e / J.m;
    double2 v = J.A[e];
    v.x *= J.scale;
    v.y *= tr ? -J.scale : J.scale;
    if (tr) sm[j + rank[i] * L] = v;
    else sm[i + rank[j] * L] = v;
  }
  __syncthreads();
  // Householder QR, a group per column; one barrier per reflector (the next
  // column's owner makes its reflector right after updating it)
  if (grp == 0) householder(sm, 0, L, l, &diag[0], &tau[0]);
  __syncthreads();
  for (int j = 0; j + 1 < c; ++j) {
    for (int k = grp; k < c; k += ng) {
      if (k <= j) continue;
      reflect(sm + j * L, tau[j], sm + k * L, j, L, l);
      if (k == j + 1) householder(sm + k * L, k, L, l, &diag[k], &tau[k]);
    }
    __syncthreads();
  }
  for (int e = tid; e < L * c; e += nt) J.work[e] = sm[e];
  __threadfence_block();
  __syncthreads();
  // X = R^H and V = 1, column by column
  const int ld = 2 * c;
  for (int e = tid; e < c * c; e += nt) {
    const int r = e % c, i = e / c;           // X[r, i] = conj(R[i, r])
    double2 v = make_double2(0.0, 0.0);
    if (r == i) v = make_double2(diag[i].x, -diag[i].y);
    else if (r > i) {
      v = J.work[i + r * L];
      v.y = -v.y;
    }
    sm[r + i * ld] = v;
    sm[c + r + i * ld] = make_double2(r == i ? 1.0 : 0.0, 0.0);
  }
  __syncthreads();
  const double eps = 2.220446049250313e-16, tol2 = eps * eps * L;
  bool done = c < 2;
  for (int sweep = 0; !done && sweep < kMaxSweeps; ++sweep) {
    if (tid == 0) rotated = 0;
    __syncthreads();
    if (ld <= 64) small_sweep<4>(sm, c, c, ld, tol2, &rotated);
    else small_sweep<kRowsPerLane>(sm, c, c, ld, tol2, &rotated);
    done = !rotated;
    __syncthreads();
  }
  // singular values |x| / |v|
  for (int k = grp; k < c; k += ng) {
    double a = 0, b = 0;
    for (int r = l; r < ld; r += 16) {
      const double2 x = sm[k * ld + r];
      const double w = x.x * x.x + x.y * x.y;
      if (r < c) a += w;
      else b += w;
    }
    a = row_sum(a);
    a = a > kNull2 ? sqrt(a) : 0.0;
    b = sqrt(row_sum(b));
    if (l == 0) {
      sig[k] = a / b;
      rx[k] = a > 0.0 ? 1.0 / a : 0.0;
      rv[k] = 1.0 / b;
    }
  }
  __syncthreads();
  for (int k = tid; k < c; k += nt) {
    int r = 0;
    for (int j = 0; j < c; ++j) r += sig[j] > sig[k] || (sig[j] == sig[k] && j < k);
    rank[k] = r;
    J.S[r] = sig[k] / J.scale;
  }
  if (tid == 0) *J.info = done ? 0 : 1;
  __syncthreads();
  if (!J.U) return;
  for (int e = tid; e < c * ld; e += nt) {
    const int j = e / ld, r = e % ld;
    const double f = r < c ? rx[j] : rv[j];
    double2 v = sm[e];
    v.x *= f;
    v.y *= f;
    sm[e] = v;
  }
  __syncthreads();
  // Null columns (an exactly rank-deficient block) get
  // directions that complete the others: unit vectors, twice projected off
  // every column.
  int unit = 0;
  for (int k = 0; k < c; ++k) {
    if (rx[k] != 0.0) continue;               // uniform: rx is shared
    for (; unit < c; ++unit) {
      for (int r = tid; r < c; r += nt) sm[k * ld + r] = make_double2(r == unit ? 1.0 : 0.0, 0.0);
      __syncthreads();
      for (int pass = 0; pass < 2; ++pass) {
        // coefficients of this column on the others (later null columns are
        // still zero and drop out), kept in sig / rv
        for (int j = grp; j < c; j += ng) {
          double gr = 0, gi = 0;
          if (j != k)
            for (int r = l; r < c; r += 16) {
              const double2 x = sm[j * ld + r], y = sm[k * ld + r];
              gr += x.x * y.x + x.y * y.y;
              gi += x.x * y.y - x.y * y.x;
            }
          gr = row_sum(gr);
          gi = row_sum(gi);
          if (l == 0) {
            sig[j] = gr;
            rv[j] = gi;
          }
        }
        __syncthreads();
        for (int r = tid; r < c; r += nt) {
          double2 y = sm[k * ld + r];
          for (int j = 0; j < c; ++j) {
            if (j == k) continue;
            const double2 x = sm[j * ld + r];
            y.x -= x.x * sig[j] - x.y * rv[j];
            y.y -= x.x * rv[j] + x.y * sig[j];
          }
          sm[k * ld + r] = y;
        }
        __syncthreads();
      }
      double len2 = 0.0;
      for (int r = 0; r < c; ++r) {
        const double2 y = sm[k * ld + r];
        len2 += y.x * y.x + y.y * y.y;
      }
      __syncthreads();
      // (the unit vectors' residuals sum to the missing dimensions, so one of
      // them leaves at least 1 / c; a residual only falls as columns are added)
      if (len2 > 0.25 / c) {
        const double f = 1.0 / sqrt(len2);
        for (int r = tid; r < c; r += nt) {
          double2 y = sm[k * ld + r];
          y.x *= f;
          y.y *= f;
          sm[k * ld + r] = y;
        }
        if (tid == 0) rx[k] = 1.0;
        ++unit;
        __syncthreads();
        break;
      }
    }
  }
  // right vectors P W of B: rows of Vh (conjugated) for B = A, columns of U
  // for B = A^H
  for (int e = tid; e < c * c; e += nt) {
    const int i = e % c, j = e / c;
    const double2 v = sm[j * ld + i];
    if (tr) J.U[perm[i] + static_cast<int64_t>(rank[j]) * c] = v;
    else J.Vh[rank[j] + static_cast<int64_t>(perm[i]) * c] = make_double2(v.x, -v.y);
  }
  // left vectors Q [V; 0]: V moves to columns of L rows (through registers: a
  // group's columns are read before the barrier and written after it)
  constexpr int kCols = 2;                    // the launch has a group per column pair
  double2 keep[kCols][(kSmallCols + 15) / 16];
#pragma unroll
  for (int q = 0; q < kCols; ++q)
#pragma unroll
    for (int t = 0; t < (kSmallCols + 15) / 16; ++t) {
      const int k = grp + q * ng, r = l + 16 * t;
      if (k < c && r < c) keep[q][t] = sm[k * ld + c + r];
    }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kCols; ++q)
#pragma unroll
    for (int t = 0; t < (kSmallCols + 15) / 16; ++t) {
      const int k = grp + q * ng, r = l + 16 * t;
      if (k < c && r < c) sm[k * L + r] = keep[q][t];
    }
  for (int k = grp; k < c; k += ng)
    for (int r = c + l; r < L; r += 16) sm[k * L + r] = make_double2(0.0, 0.0);
  __syncthreads();
  for (int k = grp; k < c; k += ng)           // a group's own columns: no barriers
    for (int j = c - 1; j >= 0; --j) reflect(J.work + j * L, tau[j], sm + k * L, j, L, l);
  __syncthreads();
  for (int e = tid; e < c * L; e += nt) {
    if (tr) {
      const int j = e % c, i = e / c;
      const double2 v = sm[j * L + i];
      J.Vh[rank[j] + static_cast<int64_t>(i) * c] = make_double2(v.x, -v.y);
    } else {
      const int i = e % L, j = e / L;
      J.U[i + static_cast<int64_t>(rank[j]) * L] = sm[j * L + i];
    }
  }
}

// ---- block Jacobi ------------------------------------------------------------

constexpr int kB = 16;                // columns per block
constexpr int kP = 2 * kB;            // columns of a pair
constexpr int kRows = 64;             // rows per workgroup of the Gram and update kernels

struct BlockJob {
  double2* X;            // c x cp, columns past c zero
  double2* V;            // c x cp
  double2* G;            // per pair and row chunk: kP x kP partial Gram matrices
  double2* Q;            // per pair: kP x kP
  int* active;           // per pair
  unsigned long long* off;   // largest |x_i^H x_j| / (|x_i| |x_j|) met in a sweep (bits of a double)
  int c, nb;             // rows and columns, column blocks (even)
  int chunks;            // row chunks of X (and of V)
  int first_pair;        // this block's first pair among all blocks'
  int done;
};

__device__ __forceinline__ const BlockJob* find_job(const BlockJob* jobs, int njobs, int pair) {
  int j = 0;
  while (j + 1 < njobs && jobs[j + 1].first_pair <= pair) ++j;
  return jobs + j;
}

// first column of half h (0, 1) of pair k in round `step`
__device__ __forceinline__ void pair_cols(const BlockJob& J, int step, int k, int& c0, int& c1) {
  int p, q;
  round_robin(J.nb, step, k, p, q);
  c0 = p * kB;
  c1 = q * kB;
}

// Partial Gram matrices of a round's pairs: one workgroup per (pair, 64 rows
// of X), 16 rows per wave.  A lane reads four consecutive rows of its column
// (lane % 16); k step s of the MFMA takes row 4 (lane / 16) + s.
__global__ __launch_bounds__(256) void gram_kernel(const BlockJob* __restrict__ jobs, int njobs, int step) {
  __shared__ double2 red[3][kP * kP];
  const BlockJob J = *find_job(jobs, njobs, blockIdx.x);
  const int k = blockIdx.x - J.first_pair, chunk = blockIdx.y;
  if (J.done || step >= J.nb - 1 || chunk >= J.chunks) return;
  int c0, c1;
  pair_cols(J, step, k, c0, c1);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int fr = lane & 15, fk = lane >> 4;
  const int r0 = chunk * kRows + wave * 16 + fk * 4;
  double2 x[2][4];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const double2* col = J.X + static_cast<int64_t>((h ? c1 : c0) + fr) * J.c;
#pragma unroll
    for (int s = 0; s < 4; ++s) x[h][s] = r0 + s < J.c ? col[r0 + s] : make_double2(0.0, 0.0);
  }
  d4v re[2][2], im[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) re[a][b] = im[a][b] = d4v{0, 0, 0, 0};
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        if (a == 1 && b == 0) continue;       // Hermitian
        re[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[a][s].x, x[b][s].x, re[a][b], 0, 0, 0);
        im[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[a][s].x, x[b][s].y, im[a][b], 0, 0, 0);
        re[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[a][s].y, x[b][s].y, re[a][b], 0, 0, 0);
        im[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(-x[a][s].y, x[b][s].x, im[a][b], 0, 0, 0);
      }
  // D[row][col]: row = fk + 4 v (index of the first operand), col = fr
  double2* out = J.G + (static_cast<int64_t>(k) * J.chunks + chunk) * (kP * kP);
  if (wave) {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = a; b < 2; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          red[wave - 1][(a * kB + fk + 4 * v) * kP + b * kB + fr] = make_double2(re[a][b][v], im[a][b][v]);
  }
  __syncthreads();
  if (wave == 0) {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = a; b < 2; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int e = (a * kB + fk + 4 * v) * kP + b * kB + fr;
          double2 t = make_double2(re[a][b][v], im[a][b][v]);
          for (int w = 0; w < 3; ++w) {
            t.x += red[w][e].x;
            t.y += red[w][e].y;
          }
          out[e] = t;
        }
  }
}

// One rotation sweep over a pair's Gram matrix: Q with X_pair Q closer to
// orthogonal, columns by falling length.  Bound by the latency of its chain
// of 31 steps: a step has one barrier (the matrix alternates between two
// buffers), every wave computes all 16 rotations in its first lanes and
// shares them by lane shuffles, and a thread updates the 2 x 2 block of one
// pair of rotations from both sides, and two rows of one column pair of Q.
// (One sweep per visit: two or four need fewer rounds, 11 and 9 instead of 15
// for a graded 128-column block, but each costs more than the Gram and update
// launches it saves.)
__global__ __launch_bounds__(256) void pair_kernel(const BlockJob* __restrict__ jobs, int njobs, int step) {
  __shared__ double2 G[2][kP][kP + 1], Q[kP][kP + 1];   // [column][row]
  __shared__ double worst[4];
  const BlockJob J = *find_job(jobs, njobs, blockIdx.x);
  const int k = blockIdx.x - J.first_pair;
  if (J.done || step >= J.nb - 1) return;
  const int tid = threadIdx.x;
  // sum of the chunks; the lower triangle from the upper one
  const double2* part = J.G + static_cast<int64_t>(k) * J.chunks * (kP * kP);
  for (int e = tid; e < kP * kP; e += 256) {
    const int i = e / kP, j = e % kP;
    if (i / kB > j / kB) continue;
    double2 t = make_double2(0.0, 0.0);
    for (int s = 0; s < J.chunks; ++s) {
      const double2 v = part[static_cast<int64_t>(s) * (kP * kP) + e];
      t.x += v.x;
      t.y += v.y;
    }
    if (i == j) t.y = 0.0;
    G[0][j][i] = t;
    if (i / kB < j / kB) G[0][i][j] = make_double2(t.x, -t.y);
  }
  for (int e = tid; e < kP * kP; e += 256) Q[e / kP][e % kP] = make_double2(e / kP == e % kP ? 1.0 : 0.0, 0.0);
  __syncthreads();
  double w = 0.0;
  for (int e = tid; e < kP * kP; e += 256) {
    const int i = e / kP, j = e % kP;
    if (i >= j) continue;
    const double2 g = G[0][j][i];
    const double h = sqrt(g.x * g.x + g.y * g.y), d = sqrt(G[0][i][i].x) * sqrt(G[0][j][j].x);
    if (G[0][i][i].x > kNull2 && G[0][j][j].x > kNull2) w = fmax(w, h / d);
  }
  for (int o = 32; o > 0; o >>= 1) w = fmax(w, __shfl_down(w, o, 64));
  if ((tid & 63) == 0) worst[tid >> 6] = w;
  __syncthreads();
  w = fmax(fmax(worst[0], worst[1]), fmax(worst[2], worst[3]));
  const double eps = 2.220446049250313e-16, tol2 = eps * eps * J.c;
  const bool act = w * w > tol2;
  if (tid == 0) {
    J.active[k] = act;
    atomicMax(J.off, static_cast<unsigned long long>(__double_as_longlong(w)));
  }
  if (!act) return;
  const int gi = tid & 15, gj = tid >> 4;     // rotations of this thread's rows and columns
  for (int st = 0; st < kP - 1; ++st) {
    const double2(*S)[kP + 1] = G[st & 1];
    double2(*D)[kP + 1] = G[(st & 1) ^ 1];
    int pi, qi, pj, qj;
    round_robin(kP, st, gi, pi, qi);
    round_robin(kP, st, gj, pj, qj);
    double2 g00 = S[pj][pi], g10 = S[pj][qi], g01 = S[qj][pi], g11 = S[qj][qi];   // [column][row]
    double2 u[2], v[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      u[t] = Q[pj][gi + 16 * t];
      v[t] = Q[qj][gi + 16 * t];
    }
    // lane gi holds rotation gi (every wave has all of them)
    const double a = S[pi][pi].x, b = S[qi][qi].x;
    const double2 g = S[qi][pi];
    const double h2 = g.x * g.x + g.y * g.y;
    Rot R;
    R.c = 1.0;
    R.s = make_double2(0.0, 0.0);
    // (a column without length keeps its place: an updated diagonal entry can
    // round below zero, and padding must stay behind the block's columns)
    R.swap = b > a && b > kNull2;
    if (needs_rotation(a, b, h2, tol2)) R = rotation(a, b, g, h2);
    Rot T;                                     // rotation gj
    T.c = __shfl(R.c, gj, 64);
    T.s.x = __shfl(R.s.x, gj, 64);
    T.s.y = __shfl(R.s.y, gj, 64);
    T.swap = __shfl(static_cast<int>(R.swap), gj, 64);
    R.s.y = -R.s.y;                            // rows take the conjugate rotation
    rotate(T, g00, g01);
    rotate(T, g10, g11);
    rotate(R, g00, g10);
    rotate(R, g01, g11);
    D[pj][pi] = g00;
    D[pj][qi] = g10;
    D[qj][pi] = g01;
    D[qj][qi] = g11;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      rotate(T, u[t], v[t]);
      Q[pj][gi + 16 * t] = u[t];
      Q[qj][gi + 16 * t] = v[t];
    }
    __syncthreads();
  }
  double2* out = J.Q + static_cast<int64_t>(k) * (kP * kP);
  for (int e = tid; e < kP * kP; e += 256) out[e] = Q[e / kP][e % kP];   // out[row + kP * column]
}

// X_pair <- X_pair Q and V_pair <- V_pair Q: one workgroup per (pair, 64 rows
// of X or V), 16 rows per wave, Q's columns the MFMA's first operand (lanes
// along rows in the result).
__global__ __launch_bounds__(256) void update_kernel(const BlockJob* __restrict__ jobs, int njobs, int step) {
  const BlockJob J = *find_job(jobs, njobs, blockIdx.x);
  const int k = blockIdx.x - J.first_pair;
  if (J.done || step >= J.nb - 1 || static_cast<int>(blockIdx.y) >= 2 * J.chunks || !J.active[k]) return;
  const bool onv = static_cast<int>(blockIdx.y) >= J.chunks;
  double2* M = onv ? J.V : J.X;
  const int rows = J.c;
  int c0, c1;
  pair_cols(J, step, k, c0, c1);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int fr = lane & 15, fk = lane >> 4;
  const int r = (onv ? blockIdx.y - J.chunks : blockIdx.y) * kRows + wave * 16 + fr;
  const double2* Q = J.Q + static_cast<int64_t>(k) * (kP * kP);
  double2 x[kP / 4];
#pragma unroll
  for (int s = 0; s < kP / 4; ++s) {
    const int kk = s * 4 + fk;
    const int col = kk < kB ? c0 + kk : c1 + kk - kB;
    x[s] = r < rows ? M[r + static_cast<int64_t>(col) * rows] : make_double2(0.0, 0.0);
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    d4v re{0, 0, 0, 0}, im{0, 0, 0, 0};
    double2 q[kP / 4];
#pragma unroll
    for (int s = 0; s < kP / 4; ++s) q[s] = Q[(s * 4 + fk) + kP * (j * kB + fr)];
#pragma unroll
    for (int s = 0; s < kP / 4; ++s) {
      re = __builtin_amdgcn_mfma_f64_16x16x4f64(q[s].x, x[s].x, re, 0, 0, 0);
      im = __builtin_amdgcn_mfma_f64_16x16x4f64(q[s].x, x[s].y, im, 0, 0, 0);
      re = __builtin_amdgcn_mfma_f64_16x16x4f64(-q[s].y, x[s].y, re, 0, 0, 0);
      im = __builtin_amdgcn_mfma_f64_16x16x4f64(q[s].y, x[s].x, im, 0, 0, 0);
    }
    if (r < rows) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int n = fk + 4 * v;
        M[r + static_cast<int64_t>((j ? c1 : c0) + n) * rows] = make_double2(re[v], im[v]);
      }
    }
  }
}

// ---- Householder QR of the larger blocks -----------------------------------
// Panels of 16 columns (8 where 16 columns of B do not fit in LDS), one
// workgroup per block and panel, a wave per column; the trailing columns are
// updated 16 at a time by the panel's compact WY form H_0 .. H_{w-1} =
// 1 - V T V^H (T upper triangular), which also applies Q to the left vectors
// at the end.

struct QrJob {
  const double2* A;      // m x n
  double2* B;            // L x c: sorted A (A^H), then R above and the reflectors on and below the diagonal
  double2* T;            // per panel 16 x 16 (zero-padded)
  double2* diag;         // R's diagonal
  double2* X;            // c x cp
  double2* V;            // c x cp
  double2* Y;            // L x ny: columns that Q is applied to (left vectors)
  double* len2;          // column lengths of A (A^H), squared
  int* perm;             // sorted position -> column
  int m, n, L, c, cp, w, npan, ny;
  double scale;
  int last_bit;          // whether entries are changed in their last bit
};

__global__ __launch_bounds__(64) void column_lengths_kernel(const QrJob* __restrict__ jobs) {
  const QrJob J = jobs[blockIdx.y];
  const bool tr = J.m < J.n;
  for (int k = blockIdx.x; k < J.c; k += gridDim.x) {
    double a = 0;
    for (int r = threadIdx.x; r < J.L; r += 64) {
      const double2 v = J.A[tr ? k + static_cast<int64_t>(r) * J.m : r + static_cast<int64_t>(k) * J.m];
      const double x = v.x * J.scale, y = v.y * J.scale;
      a += x * x + y * y;
    }
    for (int o = 32; o > 0; o >>= 1) a += __shfl_down(a, o, 64);
    if (threadIdx.x == 0) J.len2[k] = a;
  }
}

__global__ __launch_bounds__(1024) void sort_columns_kernel(const QrJob* __restrict__ jobs) {
  const QrJob J = jobs[blockIdx.x];
  for (int k = threadIdx.x; k < J.c; k += 1024) {
    const double w = J.len2[k];
    int r = 0;
    for (int j = 0; j < J.c; ++j) r += J.len2[j] > w || (J.len2[j] == w && j < k);
    J.perm[r] = k;
  }
}

// x (1 + d), |d| <= eps, pseudorandom by entry
__device__ __forceinline__ double last_bit(double x, uint64_t e) {
  e = (e ^ (e >> 30)) * 0xbf58476d1ce4e5b9ull;       // splitmix64's finisher
  e = (e ^ (e >> 27)) * 0x94d049bb133111ebull;
  e ^= e >> 31;
  return x + x * (static_cast<double>(static_cast<int64_t>(e)) * 0x1p-115);
}

__global__ void load_kernel(const QrJob* __restrict__ jobs) {
  const QrJob J = jobs[blockIdx.y];
  const bool tr = J.m < J.n;
  for (int64_t e = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; e < static_cast<int64_t>(J.L) * J.c;
       e += int64_t(gridDim.x) * blockDim.x) {
    const int64_t i = e % J.L, k = J.perm[e / J.L];
    double2 v = J.A[tr ? k + i * J.m : i + k * J.m];
    v.x *= J.scale;
    v.y *= tr ? -J.scale : J.scale;
    if (J.last_bit) v = make_double2(last_bit(v.x, 2 * e + 1), last_bit(v.y, 2 * e + 2));
    J.B[e] = v;
  }
}

__device__ __forceinline__ double wave_sum(double x) {
  x = row_sum(x);
  x += __shfl_xor(x, 16, 64);
  return x + __shfl_xor(x, 32, 64);
}

constexpr int kPanelThreads = 1024;
constexpr int64_t kPanelLds = 150 * 1024;
constexpr int64_t kQrMaxRows = kPanelLds / (8 * 16);   // 8 columns of 16-byte entries

__global__ __launch_bounds__(kPanelThreads) void panel_kernel(const QrJob* __restrict__ jobs, int pan) {
  extern __shared__ double2 sp[];
  __shared__ double2 D[kB][kB + 1], T[kB][kB + 1], dg[kB];
  __shared__ double tau[kB];
  const QrJob J = jobs[blockIdx.x];
  if (pan >= J.npan) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int j0 = pan * J.w, w = min(J.w, J.c - j0), rows = J.L - j0;
  double2* const Bp = J.B + j0 + static_cast<int64_t>(j0) * J.L;
  for (int e = tid; e < rows * w; e += kPanelThreads) sp[e] = Bp[e % rows + static_cast<int64_t>(e / rows) * J.L];
  if (tid < kB) tau[tid] = 0.0;
  __syncthreads();
  auto make = [&](int j) {                    // one wave: column j's reflector
    double2* x = sp + j * rows;
    double s = 0.0;
    for (int r = j + lane; r < rows; r += 64) s += x[r].x * x[r].x + x[r].y * x[r].y;
    s = wave_sum(s);
    const double2 al = x[j];
    const double nx = s > kNull2 ? sqrt(s) : 0.0, aa = s > kNull2 ? sqrt(al.x * al.x + al.y * al.y) : 0.0;
    const double2 ph = aa > 0.0 ? make_double2(al.x / aa, al.y / aa) : make_double2(1.0, 0.0);
    if (lane == 0) {
      dg[j] = make_double2(-ph.x * nx, -ph.y * nx);
      tau[j] = nx > 0.0 ? 1.0 / (nx * (nx + aa)) : 0.0;
      x[j] = make_double2(ph.x * (aa + nx), ph.y * (aa + nx));
    }
  };
  auto dot = [&](const double2* v, const double2* y, int r0) {
    double gr = 0, gi = 0;
    for (int r = r0 + lane; r < rows; r += 64) {
      const double2 a = v[r], b = y[r];
      gr += a.x * b.x + a.y * b.y;
      gi += a.x * b.y - a.y * b.x;
    }
    return make_double2(wave_sum(gr), wave_sum(gi));
  };
  if (wave == 0) make(0);
  __syncthreads();
  for (int j = 0; j + 1 < w; ++j) {
    if (wave > j && wave < w) {
      const double2* v = sp + j * rows;
      double2* y = sp + wave * rows;
      double2 g = dot(v, y, j);
      g.x *= tau[j];
      g.y *= tau[j];
      for (int r = j + lane; r < rows; r += 64) {
        const double2 a = v[r];
        double2 b = y[r];
        b.x -= g.x * a.x - g.y * a.y;
        b.y -= g.x * a.y + g.y * a.x;
        y[r] = b;
      }
      wave_order();
      if (wave == j + 1) make(j + 1);
    }
    __syncthreads();
  }
  // T from the reflectors' inner products
  for (int e = wave; e < kB * kB; e += kPanelThreads / 64) {
    const int i = e / kB, j = e % kB;
    if (i < j && j < w) {
      const double2 g = dot(sp + i * rows, sp + j * rows, j);
      if (lane == 0) D[i][j] = g;
    }
  }
  if (tid < kB * kB) T[tid / kB][tid % kB] = make_double2(0.0, 0.0);
  __syncthreads();
  if (wave == 0) {
    for (int j = 0; j < w; ++j) {
      const int i = lane;
      double2 t = make_double2(0.0, 0.0);
      if (i < j)
        for (int q = i; q < j; ++q) {
          const double2 p = cmul(T[i][q], D[q][j]);
          t.x -= tau[j] * p.x;
          t.y -= tau[j] * p.y;
        }
      if (i == j) t.x = tau[j];
      wave_order();
      if (i <= j) T[i][j] = t;
      wave_order();
    }
  }
  __syncthreads();
  double2* out = J.T + static_cast<int64_t>(pan) * (kB * kB);
  for (int e = tid; e < kB * kB; e += kPanelThreads) out[e] = T[e / kB][e % kB];   // out[row * 16 + column]
  if (tid < w) J.diag[j0 + tid] = dg[tid];
  for (int e = tid; e < rows * w; e += kPanelThreads) Bp[e % rows + static_cast<int64_t>(e / rows) * J.L] = sp[e];
}

// Columns Y (16 per workgroup) <- (1 - V T' V^H) Y over rows j0.. of a panel:
// T' = T^H on the trailing columns of B (onq = 0), T on Y.
// MFMA for V^H Y (rows split over the four waves) and for V (T' V^H Y).
__global__ __launch_bounds__(256) void reflect_kernel(const QrJob* __restrict__ jobs, int pan, int onq) {
  __shared__ double2 red[4][kB][kB + 1], W[kB][kB + 1];
  const QrJob J = jobs[blockIdx.y];
  if (pan >= J.npan) return;
  const int j0 = pan * J.w, w = min(J.w, J.c - j0);
  const int c0 = (onq ? 0 : j0 + w) + blockIdx.x * kB, cols = onq ? J.ny : J.c;
  if (c0 >= cols || (onq && !J.Y)) return;
  double2* const Y = onq ? J.Y : J.B;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int fr = lane & 15, fk = lane >> 4;
  const int64_t L = J.L;
  // reflector t (column j0 + t of B) at row r: zero above row j0 + t
  auto vat = [&](int t, int64_t r) {
    return t < w && r >= j0 + t && r < L ? J.B[r + (j0 + t) * L] : make_double2(0.0, 0.0);
  };
  const bool cin = c0 + fr < cols;
  {
    d4v re{0, 0, 0, 0}, im{0, 0, 0, 0};
    for (int64_t r0 = j0 + wave * 16; r0 < L; r0 += 64) {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int64_t r = r0 + fk * 4 + s;
        const double2 v = vat(fr, r);
        const double2 y = cin && r < L ? Y[r + (c0 + fr) * L] : make_double2(0.0, 0.0);
        re = __builtin_amdgcn_mfma_f64_16x16x4f64(v.x, y.x, re, 0, 0, 0);
        im = __builtin_amdgcn_mfma_f64_16x16x4f64(v.x, y.y, im, 0, 0, 0);
        re = __builtin_amdgcn_mfma_f64_16x16x4f64(v.y, y.y, re, 0, 0, 0);
        im = __builtin_amdgcn_mfma_f64_16x16x4f64(-v.y, y.x, im, 0, 0, 0);
      }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) red[wave][fk + 4 * v][fr] = make_double2(re[v], im[v]);
  }
  __syncthreads();
  {
    const int i = threadIdx.x >> 4, j = threadIdx.x & 15;
    const double2* T = J.T + static_cast<int64_t>(pan) * (kB * kB);
    double2 z = make_double2(0.0, 0.0);
    for (int q = 0; q < kB; ++q) {
      double2 t = onq ? T[i * kB + q] : T[q * kB + i];
      if (!onq) t.y = -t.y;
      double2 x = red[0][q][j];
#pragma unroll
      for (int u = 1; u < 4; ++u) {
        x.x += red[u][q][j].x;
        x.y += red[u][q][j].y;
      }
      const double2 p = cmul(t, x);
      z.x += p.x;
      z.y += p.y;
    }
    W[i][j] = z;
  }
  __syncthreads();
  // Y -= V W: lanes along rows (the first operand holds W's columns)
  for (int64_t r0 = j0 + wave * 16; r0 < L; r0 += 64) {
    const int64_t r = r0 + fr;
    d4v re{0, 0, 0, 0}, im{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int t = s * 4 + fk;
      const double2 v = vat(t, r), z = W[t][fr];
      re = __builtin_amdgcn_mfma_f64_16x16x4f64(z.x, v.x, re, 0, 0, 0);
      im = __builtin_amdgcn_mfma_f64_16x16x4f64(z.x, v.y, im, 0, 0, 0);
      re = __builtin_amdgcn_mfma_f64_16x16x4f64(-z.y, v.y, re, 0, 0, 0);
      im = __builtin_amdgcn_mfma_f64_16x16x4f64(z.y, v.x, im, 0, 0, 0);
    }
    if (r < L) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int k = c0 + fk + 4 * v;
        if (k < cols) {
          double2 y = Y[r + k * L];
          y.x -= re[v];
          y.y -= im[v];
          Y[r + k * L] = y;
        }
      }
    }
  }
}

// X = R^H, V = 1; padding columns zero
__global__ void start_kernel(const QrJob* __restrict__ jobs) {
  const QrJob J = jobs[blockIdx.y];
  const int64_t c = J.c;
  for (int64_t e = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; e < c * J.cp; e += int64_t(gridDim.x) * blockDim.x) {
    const int64_t r = e % c, i = e / c;
    double2 v = make_double2(0.0, 0.0);
    if (i < c && r == i) v = make_double2(J.diag[i].x, -J.diag[i].y);
    else if (i < c && r > i) {
      v = J.B[i + r * static_cast<int64_t>(J.L)];
      v.y = -v.y;
    }
    J.X[e] = v;
    J.V[e] = make_double2(i < c && r == i ? 1.0 : 0.0, 0.0);
  }
}

// nrm[2 j] = |x_j|, nrm[2 j + 1] = |v_j|; one wave per column
__global__ __launch_bounds__(64) void norms_kernel(const QrJob* __restrict__ jobs, double* const* __restrict__ nrm) {
  const QrJob J = jobs[blockIdx.y];
  for (int j = blockIdx.x; j < J.c; j += gridDim.x) {
    double a = 0, b = 0;
    for (int r = threadIdx.x; r < J.c; r += 64) {
      const double2 x = J.X[r + static_cast<int64_t>(j) * J.c], v = J.V[r + static_cast<int64_t>(j) * J.c];
      a += x.x * x.x + x.y * x.y;
      b += v.x * v.x + v.y * v.y;
    }
    for (int o = 32; o > 0; o >>= 1) {
      a += __shfl_down(a, o, 64);
      b += __shfl_down(b, o, 64);
    }
    if (threadIdx.x == 0) {
      nrm[blockIdx.y][2 * j] = sqrt(a);
      nrm[blockIdx.y][2 * j + 1] = sqrt(b);
    }
  }
}

// Null columns of X (an exactly rank-deficient block) are replaced by unit
// vectors that complete the others: with the r others, normalised, as B = Q R,
// the last c - r columns of Q.  On the panel kernels this takes about what the
// block's own QR does; unit vectors projected off every column one after
// another by one workgroup took 788 ms of the 798 ms of a 1024-column block of
// rank one (zgesvd: 328 ms).
struct NullJob {
  double2* X;            // c x c
  double2* B;            // c x r
  double2* Y;            // c x (c - r)
  const double* rx;      // 1 / |x|, by column
  const int* col;        // the r other columns, then the null ones
  int c, r;
};
__global__ void null_load_kernel(const NullJob* __restrict__ jobs) {
  const NullJob J = jobs[blockIdx.y];
  const int64_t c = J.c;
  for (int64_t e = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; e < c * c; e += int64_t(gridDim.x) * blockDim.x) {
    const int64_t i = e % c, k = e / c;
    if (k < J.r) {
      const double f = J.rx[J.col[k]];
      const double2 x = J.X[i + J.col[k] * c];
      J.B[e] = make_double2(x.x * f, x.y * f);
    } else {
      J.Y[i + (k - J.r) * c] = make_double2(i == k ? 1.0 : 0.0, 0.0);
    }
  }
}
__global__ void null_store_kernel(const NullJob* __restrict__ jobs) {
  const NullJob J = jobs[blockIdx.y];
  const int64_t c = J.c;
  for (int64_t e = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; e < c * (c - J.r);
       e += int64_t(gridDim.x) * blockDim.x)
    J.X[e % c + J.col[J.r + e / c] * c] = J.Y[e];
}

// singular vectors in falling order: the right ones P W (into Vh or, for
// B = A^H, U) and [V; 0], to which Q is still to be applied
struct OutJob {
  double2* U;
  double2* Vh;
  const int* src;        // singular index -> column
  const double* f;       // 1 / |x|, then 1 / |v|, by singular index
};
__global__ void vectors_kernel(const QrJob* __restrict__ jobs, const OutJob* __restrict__ outs) {
  const QrJob J = jobs[blockIdx.y];
  const OutJob O = outs[blockIdx.y];
  if (!O.U) return;
  const bool tr = J.m < J.n;
  const int64_t c = J.c, L = J.L;
  for (int64_t e = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; e < L * c; e += int64_t(gridDim.x) * blockDim.x) {
    const int64_t r = e % L, j = e / L;
    double2 v = make_double2(0.0, 0.0);
    if (r < c) {
      v = J.V[r + O.src[j] * c];
      v.x *= O.f[c + j];
      v.y *= O.f[c + j];
      double2 x = J.X[r + O.src[j] * c];
      x.x *= O.f[j];
      x.y *= O.f[j];
      if (tr) O.U[J.perm[r] + j * c] = x;
      else O.Vh[j + J.perm[r] * c] = make_double2(x.x, -x.y);
    }
    J.Y[e] = v;
  }
}
// Vh = Y^H for B = A^H (otherwise Y is U itself)
__global__ void adjoint_kernel(const QrJob* __restrict__ jobs, const OutJob* __restrict__ outs) {
  const QrJob J = jobs[blockIdx.y];
  const OutJob O = outs[blockIdx.y];
  if (!O.U || J.m >= J.n) return;
  for (int64_t e = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; e < static_cast<int64_t>(J.L) * J.c;
       e += int64_t(gridDim.x) * blockDim.x) {
    const int64_t j = e % J.c, r = e / J.c;
    const double2 v = J.Y[r + j * J.L];
    O.Vh[e] = make_double2(v.x, -v.y);
  }
}

}  // namespace

bool jacobi_svd_small(int64_t m, int64_t n) {
  const int64_t L = std::max(m, n), c = std::min(m, n);
  return c <= kSmallCols && L <= kSmallRows && small_entries(L, c) * static_cast<int64_t>(sizeof(double2)) <= kSmallLds;
}

bool jacobi_svd_fits(int64_t m, int64_t n) {
  return jacobi_svd_small(m, n) || (std::min(m, n) <= kJacobiMaxCols && std::max(m, n) <= kQrMaxRows);
}

// columns of a QR panel that fit in LDS, from their rows
static int panel_width(int64_t rows) {
  return rows * kB * static_cast<int64_t>(sizeof(double2)) <= kPanelLds ? kB : kB / 2;
}

// U and Vh, and the work that jacobi_svd allocates for a block (with the
// completion of null columns)
int64_t jacobi_svd_bytes(int64_t m, int64_t n, bool vectors) {
  const int64_t L = std::max(m, n), c = std::min(m, n), uv = vectors ? (m + n) * c : 0;
  constexpr int64_t es = sizeof(double2);
  if (jacobi_svd_small(m, n)) return es * (uv + L * c + c);
  const int64_t nb = (c + kB - 1) / kB + 1, chunks = (c + kRows - 1) / kRows, pan = c / panel_width(L) + 1;
  return es * (uv + 2 * L * c + pan * kB * kB + 6 * c + 2 * c * nb * kB + nb / 2 * (chunks + 1) * kP * kP +
               (vectors ? c * c + pan * kB * kB : 0));
}

std::vector<size_t> jacobi_svd_batches(const std::vector<JacobiSize>& blocks, bool vectors, int64_t bytes,
                                       size_t items) {
  std::vector<size_t> ends;
  int64_t sum = 0;
  size_t first = 0;
  for (size_t i = 0; i < blocks.size(); ++i) {
    const int64_t b = jacobi_svd_bytes(blocks[i].m, blocks[i].n, vectors);
    if (i > first && (sum + b > bytes || i - first >= items)) {
      ends.push_back(i);
      first = i;
      sum = 0;
    }
    sum += b;
  }
  if (first < blocks.size()) ends.push_back(blocks.size());
  return ends;
}

std::vector<char> jacobi_svd(Ctx& ctx, const std::vector<JacobiItem>& items) {
  hipStream_t s = ctx.stream;
  std::vector<char> ok(items.size(), 0);
  std::vector<size_t> small, big;
  for (size_t i = 0; i < items.size(); ++i) (jacobi_svd_small(items[i].m, items[i].n) ? small : big).push_back(i);
  auto scale_of = [](double weight) { return std::ldexp(1.0, -std::ilogb(std::sqrt(weight))); };

  if (!small.empty()) {
    size_t stot = 0;
    int64_t lds = 0, threads = 64, wtot = 0;
    for (size_t i : small) {
      const JacobiItem& it = items[i];
      const int64_t L = std::max(it.m, it.n), c = std::min(it.m, it.n);
      stot += static_cast<size_t>(c);
      lds = std::max<int64_t>(lds, small_entries(L, c) * static_cast<int64_t>(sizeof(double2)));
      // 16 lanes per column pair
      threads = std::max(threads, std::min<int64_t>(kSmallThreads, ((c + 1) / 2 * 16 + 63) / 64 * 64));
      wtot += L * c;
    }
    DevBuf<double> S(stot);
    DevBuf<int> info(small.size());
    DevBuf<cplx> work(static_cast<size_t>(wtot));
    wtot = 0;
    std::vector<SmallJob> jobs;
    size_t at = 0;
    for (size_t q = 0; q < small.size(); ++q) {
      const JacobiItem& it = items[small[q]];
      jobs.push_back(SmallJob{reinterpret_cast<const double2*>(it.A), reinterpret_cast<double2*>(it.U),
                              reinterpret_cast<double2*>(it.Vh), reinterpret_cast<double2*>(work.get() + wtot),
                              S.get() + at, info.get() + q, static_cast<int>(it.m), static_cast<int>(it.n),
                              scale_of(it.weight)});
      wtot += it.m * it.n;
      at += static_cast<size_t>(std::min(it.m, it.n));
    }
    DevBuf<SmallJob> dj(jobs.size());
    dj.upload(jobs.data(), jobs.size(), s);
    HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(jacobi_small_kernel),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, kSmallLds));
    hipLaunchKernelGGL(jacobi_small_kernel, dim3(jobs.size()), dim3(threads), static_cast<size_t>(lds), s,
                       dj.get());
    HIP_CHECK(hipGetLastError());
    std::vector<double> hs(stot);
    std::vector<int> hi(small.size());
    HIP_CHECK(hipMemcpyAsync(hs.data(), S.get(), stot * sizeof(double), hipMemcpyDeviceToHost, s));
    HIP_CHECK(hipMemcpyAsync(hi.data(), info.get(), hi.size() * sizeof(int), hipMemcpyDeviceToHost, s));
    HIP_CHECK(hipStreamSynchronize(s));
    at = 0;
    for (size_t q = 0; q < small.size(); ++q) {
      const JacobiItem& it = items[small[q]];
      const size_t c = static_cast<size_t>(std::min(it.m, it.n));
      it.S->assign(hs.begin() + at, hs.begin() + at + c);
      ok[small[q]] = hi[q] == 0;
      at += c;
    }
  }
  if (big.empty()) return ok;

  // ---- block Jacobi ----------------------------------------------------------
  const int nj = static_cast<int>(big.size());
  struct Sz { int64_t L, c, cp, npan; int w, nb, chunks; };
  std::vector<Sz> sz;
  int64_t xtot = 0, gtot = 0, ctot = 0, lds = 0;
  int pairs = 0, maxch = 0, npan = 0;
  for (size_t i : big) {
    const JacobiItem& it = items[i];
    Sz z;
    z.L = std::max(it.m, it.n);
    z.c = std::min(it.m, it.n);
    z.w = panel_width(z.L);
    z.npan = (z.c + z.w - 1) / z.w;
    z.nb = static_cast<int>((z.c + kB - 1) / kB);
    z.nb += z.nb & 1;
    z.cp = static_cast<int64_t>(z.nb) * kB;
    z.chunks = static_cast<int>((z.c + kRows - 1) / kRows);
    // B, T, diag, X, V and, for B = A^H, Y
    xtot += z.L * z.c + z.npan * kB * kB + z.c + 2 * z.c * z.cp + (it.m < it.n && it.U ? z.L * z.c : 0);
    gtot += static_cast<int64_t>(z.nb / 2) * (z.chunks + 1) * kP * kP;
    ctot += z.c;
    lds = std::max(lds, z.L * z.w * static_cast<int64_t>(sizeof(double2)));
    pairs += z.nb / 2;
    maxch = std::max(maxch, z.chunks);
    npan = std::max(npan, static_cast<int>(z.npan));
    sz.push_back(z);
  }
  DevBuf<cplx> work(static_cast<size_t>(xtot)), G(static_cast<size_t>(gtot));
  DevBuf<int> active(pairs), perm(static_cast<size_t>(ctot)), src(static_cast<size_t>(ctot));
  DevBuf<unsigned long long> off(big.size());
  DevBuf<double> dbl(static_cast<size_t>(5 * ctot));   // len2, then |x|, |v| pairs, then their inverses
  std::vector<BlockJob> jobs;
  std::vector<QrJob> qr;
  std::vector<double*> nrm;
  {
    double2* x = reinterpret_cast<double2*>(work.get());
    double2* g = reinterpret_cast<double2*>(G.get());
    auto take = [&](int64_t n) {
      double2* p = x;
      x += n;
      return p;
    };
    int pair = 0;
    int64_t cc = 0;
    for (int q = 0; q < nj; ++q) {
      const JacobiItem& it = items[big[q]];
      const Sz& z = sz[q];
      QrJob j{};
      j.A = reinterpret_cast<const double2*>(it.A);
      j.B = take(z.L * z.c);
      j.T = take(z.npan * kB * kB);
      j.diag = take(z.c);
      j.X = take(z.c * z.cp);
      j.V = take(z.c * z.cp);
      j.Y = !it.U ? nullptr : it.m < it.n ? take(z.L * z.c) : reinterpret_cast<double2*>(it.U);
      j.len2 = dbl.get() + cc;
      j.perm = perm.get() + cc;
      j.m = static_cast<int>(it.m);
      j.n = static_cast<int>(it.n);
      j.L = static_cast<int>(z.L);
      j.c = static_cast<int>(z.c);
      j.cp = static_cast<int>(z.cp);
      j.w = z.w;
      j.npan = static_cast<int>(z.npan);
      j.ny = j.c;
      j.scale = scale_of(it.weight);
      qr.push_back(j);
      BlockJob b{};
      b.X = j.X;
      b.V = j.V;
      b.G = g;
      b.Q = g + static_cast<int64_t>(z.nb / 2) * z.chunks * kP * kP;
      b.active = active.get() + pair;
      b.off = off.get() + q;
      b.c = j.c;
      b.nb = z.nb;
      b.chunks = z.chunks;
      b.first_pair = pair;
      jobs.push_back(b);
      nrm.push_back(dbl.get() + ctot + 2 * cc);
      g += static_cast<int64_t>(z.nb / 2) * (z.chunks + 1) * kP * kP;
      pair += z.nb / 2;
      cc += z.c;
    }
  }
  DevBuf<QrJob> dq(qr.size());
  dq.upload(qr.data(), qr.size(), s);
  DevBuf<BlockJob> dj(jobs.size());
  dj.upload(jobs.data(), jobs.size(), s);
  DevBuf<double*> dn(nrm.size());
  dn.upload(nrm.data(), nrm.size(), s);
  int64_t cmax = 0;
  for (const Sz& z : sz) cmax = std::max(cmax, z.c);
  HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(panel_kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize, kPanelLds));
  hipLaunchKernelGGL(column_lengths_kernel, dim3(static_cast<unsigned>(cmax), nj), dim3(64), 0, s, dq.get());
  hipLaunchKernelGGL(sort_columns_kernel, dim3(nj), dim3(1024), 0, s, dq.get());
  const unsigned cchunks = static_cast<unsigned>((cmax + kB - 1) / kB);
  auto factorise = [&](const QrJob* d, int count) {
    hipLaunchKernelGGL(load_kernel, dim3(256, count), dim3(256), 0, s, d);
    for (int p = 0; p < npan; ++p) {
      hipLaunchKernelGGL(panel_kernel, dim3(count), dim3(kPanelThreads), static_cast<size_t>(lds), s, d, p);
      hipLaunchKernelGGL(reflect_kernel, dim3(cchunks, count), dim3(256), 0, s, d, p, 0);
    }
    hipLaunchKernelGGL(start_kernel, dim3(256, count), dim3(256), 0, s, d);
    HIP_CHECK(hipGetLastError());
  };
  factorise(dq.get(), nj);
  std::vector<unsigned long long> hoff(jobs.size());
  for (int sweep = 0; sweep < kMaxSweeps; ++sweep) {
    launch_zero(off.get(), static_cast<int64_t>(jobs.size() * sizeof(unsigned long long)), s);
    int nsteps = 0, mch = 0;
    for (const BlockJob& b : jobs)
      if (!b.done) {
        nsteps = std::max(nsteps, b.nb - 1);
        mch = std::max(mch, b.chunks);
      }
    for (int st = 0; st < nsteps; ++st) {
      hipLaunchKernelGGL(gram_kernel, dim3(pairs, mch), dim3(256), 0, s, dj.get(), nj, st);
      hipLaunchKernelGGL(pair_kernel, dim3(pairs), dim3(256), 0, s, dj.get(), nj, st);
      hipLaunchKernelGGL(update_kernel, dim3(pairs, 2 * mch), dim3(256), 0, s, dj.get(), nj, st);
    }
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipMemcpyAsync(hoff.data(), off.get(), hoff.size() * sizeof(unsigned long long), hipMemcpyDeviceToHost, s));
    HIP_CHECK(hipStreamSynchronize(s));
    bool all = true;
    std::vector<QrJob> again;
    for (size_t q = 0; q < jobs.size(); ++q) {
      if (jobs[q].done) continue;
      double w;
      static_assert(sizeof(w) == sizeof(hoff[q]), "bits of a double");
      std::memcpy(&w, &hoff[q], sizeof(w));
      // the columns' scaled inner products at the sweep's start: at rounding
      // level nothing was left to rotate
      if (w <= 4.0 * std::numeric_limits<double>::epsilon() * std::sqrt(double(jobs[q].c))) jobs[q].done = 1;
      else all = false;
      if (sweep + 1 == kStallSweeps && w > kStalled) again.push_back(qr[q]);
    }
    if (all) break;
    dj.upload(jobs.data(), jobs.size(), s);
    if (again.empty()) continue;
    for (QrJob& j : again) {
      const size_t c = static_cast<size_t>(j.c);
      std::vector<cplx> diag(c);
      std::vector<int> old(c), order;
      HIP_CHECK(hipMemcpyAsync(diag.data(), j.diag, c * sizeof(cplx), hipMemcpyDeviceToHost, s));
      HIP_CHECK(hipMemcpyAsync(old.data(), j.perm, c * sizeof(int), hipMemcpyDeviceToHost, s));
      HIP_CHECK(hipStreamSynchronize(s));
      double longest = 0.0;
      for (const cplx& d : diag) longest = std::max(longest, std::hypot(d.re, d.im));
      auto dependent = [&](size_t k) {
        return std::hypot(diag[k].re, diag[k].im) <= double(c) * std::numeric_limits<double>::epsilon() * longest;
      };
      for (size_t k = 0; k < c; ++k)
        if (!dependent(k)) order.push_back(old[k]);
      for (size_t k = 0; k < c; ++k)
        if (dependent(k)) order.push_back(old[k]);
      HIP_CHECK(hipMemcpyAsync(j.perm, order.data(), c * sizeof(int), hipMemcpyHostToDevice, s));
      HIP_CHECK(hipStreamSynchronize(s));
      j.last_bit = 1;
    }
    DevBuf<QrJob> da(again.size());
    da.upload(again.data(), again.size(), s);
    factorise(da.get(), static_cast<int>(again.size()));
    HIP_CHECK(hipStreamSynchronize(s));
  }
  hipLaunchKernelGGL(norms_kernel, dim3(static_cast<unsigned>(cmax), nj), dim3(64), 0, s, dq.get(), dn.get());
  HIP_CHECK(hipGetLastError());
  std::vector<double> hn(static_cast<size_t>(2 * ctot));
  HIP_CHECK(hipMemcpyAsync(hn.data(), dbl.get() + ctot, hn.size() * sizeof(double), hipMemcpyDeviceToHost, s));
  HIP_CHECK(hipStreamSynchronize(s));
  std::vector<int> hsrc(static_cast<size_t>(ctot));
  std::vector<double> hfac(static_cast<size_t>(2 * ctot));
  std::vector<OutJob> outs(big.size());
  std::vector<std::vector<int>> null_cols(big.size());
  std::vector<double> hrx(static_cast<size_t>(ctot), 0.0);
  bool vectors = false;
  int64_t cc = 0;
  for (int q = 0; q < nj; ++q) {
    const JacobiItem& it = items[big[q]];
    const Sz& z = sz[q];
    std::vector<int> ord(static_cast<size_t>(z.c));
    std::iota(ord.begin(), ord.end(), 0);
    const double* nn = hn.data() + 2 * cc;
    ok[big[q]] = jobs[q].done;
    if (jobs[q].done) {
      std::vector<double> sg(static_cast<size_t>(z.c));
      for (int64_t j = 0; j < z.c; ++j) {
        const bool null = !(nn[2 * j] * nn[2 * j] > kNull2);
        sg[j] = null ? 0.0 : nn[2 * j] / nn[2 * j + 1];
        hrx[cc + j] = null ? 0.0 : 1.0 / nn[2 * j];
        if (null && it.U) null_cols[q].push_back(static_cast<int>(j));
      }
      std::stable_sort(ord.begin(), ord.end(), [&](int a, int b) { return sg[a] > sg[b]; });
      it.S->resize(static_cast<size_t>(z.c));
      for (int64_t j = 0; j < z.c; ++j) {
        (*it.S)[j] = sg[ord[j]] / qr[q].scale;
        hsrc[cc + j] = ord[j];
        hfac[2 * cc + j] = hrx[cc + ord[j]] != 0.0 ? hrx[cc + ord[j]] : 1.0;   // completed columns have length 1
        hfac[2 * cc + z.c + j] = 1.0 / nn[2 * ord[j] + 1];
      }
      if (it.U) {
        outs[q] = OutJob{reinterpret_cast<double2*>(it.U), reinterpret_cast<double2*>(it.Vh), src.get() + cc,
                         dbl.get() + 3 * ctot + 2 * cc};
        vectors = true;
      }
    }
    cc += z.c;
  }
  if (vectors) {
    src.upload(hsrc.data(), hsrc.size(), s);
    HIP_CHECK(hipMemcpyAsync(dbl.get() + 3 * ctot, hfac.data(), hfac.size() * sizeof(double), hipMemcpyHostToDevice, s));
    DevBuf<OutJob> dout(outs.size());
    dout.upload(outs.data(), outs.size(), s);
    std::vector<DevBuf<cplx>> completion;
    DevBuf<NullJob> dz;
    DevBuf<QrJob> dzq;
    DevBuf<int> dcol;
    std::vector<NullJob> nulls;
    std::vector<QrJob> nqr;
    std::vector<int> ncol;
    cc = 0;
    for (int q = 0; q < nj; ++q) {
      const int c = qr[q].c, z = static_cast<int>(null_cols[q].size());
      if (z) {
        QrJob j{};
        j.L = c;
        j.c = c - z;
        j.w = panel_width(c);
        j.npan = (j.c + j.w - 1) / j.w;
        j.ny = z;
        completion.emplace_back(static_cast<size_t>(c) * c + static_cast<size_t>(j.npan) * kB * kB + j.c);
        double2* at = reinterpret_cast<double2*>(completion.back().get());
        j.B = at;
        j.Y = at + static_cast<int64_t>(c) * j.c;
        j.T = at + static_cast<int64_t>(c) * c;
        j.diag = j.T + static_cast<int64_t>(j.npan) * (kB * kB);
        nqr.push_back(j);
        // (the column lengths' array is free by now and takes 1 / |x|)
        nulls.push_back(NullJob{qr[q].X, j.B, j.Y, dbl.get() + cc, nullptr, c, j.c});
        for (int k = 0, next = 0; k < c; ++k) {
          if (next < z && null_cols[q][next] == k) ++next;
          else ncol.push_back(k);
        }
        ncol.insert(ncol.end(), null_cols[q].begin(), null_cols[q].end());
      }
      cc += c;
    }
    if (!nulls.empty()) {
      const int nn = static_cast<int>(nulls.size());
      HIP_CHECK(hipMemcpyAsync(dbl.get(), hrx.data(), hrx.size() * sizeof(double), hipMemcpyHostToDevice, s));
      dcol.alloc(ncol.size());
      dcol.upload(ncol.data(), ncol.size(), s);
      int pans = 0, off = 0;
      int64_t nlds = 0;
      for (int q = 0; q < nn; ++q) {
        nulls[q].col = dcol.get() + off;
        off += nulls[q].c;
        pans = std::max(pans, nqr[q].npan);
        nlds = std::max(nlds, static_cast<int64_t>(nqr[q].L) * nqr[q].w * static_cast<int64_t>(sizeof(double2)));
      }
      dz.alloc(nulls.size());
      dz.upload(nulls.data(), nulls.size(), s);
      dzq.alloc(nqr.size());
      dzq.upload(nqr.data(), nqr.size(), s);
      hipLaunchKernelGGL(null_load_kernel, dim3(256, nn), dim3(256), 0, s, dz.get());
      for (int p = 0; p < pans; ++p) {
        hipLaunchKernelGGL(panel_kernel, dim3(nn), dim3(kPanelThreads), static_cast<size_t>(nlds), s, dzq.get(), p);
        hipLaunchKernelGGL(reflect_kernel, dim3(cchunks, nn), dim3(256), 0, s, dzq.get(), p, 0);
      }
      for (int p = pans - 1; p >= 0; --p)
        hipLaunchKernelGGL(reflect_kernel, dim3(cchunks, nn), dim3(256), 0, s, dzq.get(), p, 1);
      hipLaunchKernelGGL(null_store_kernel, dim3(256, nn), dim3(256), 0, s, dz.get());
      HIP_CHECK(hipGetLastError());
    }
    hipLaunchKernelGGL(vectors_kernel, dim3(256, nj), dim3(256), 0, s, dq.get(), dout.get());
    for (int p = npan - 1; p >= 0; --p)
      hipLaunchKernelGGL(reflect_kernel, dim3(cchunks, nj), dim3(256), 0, s, dq.get(), p, 1);
    hipLaunchKernelGGL(adjoint_kernel, dim3(256, nj), dim3(256), 0, s, dq.get(), dout.get());
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipStreamSynchronize(s));
  }
  return ok;
}

}  // namespace cam
