// Grouped persistent complex GEMM kernels (gfx950 MFMA).
//
// Workgroup = 4 wave64s arranged 2x2 (8 for the widest FP64 tiles); a TM x TN
// output tile per workgroup, each wave owning a sub-tile made of 16x16 MFMA
// fragments.  K is consumed in chunks of KC (16 or 8) staged through LDS
// as interleaved (re, im) pairs (one LDS read gives both parts of a fragment);
// the next chunk is prefetched into registers while the current one is
// multiplied.  A complex product is four real MFMAs,
//   Cre += Are*Bre + (-Aim)*Bim,   Cim += Are*Bim + Aim*Bre,
// or three (Gauss): P1 = Are*Bre, P2 = Aim*Bim, P3 = (Are+Aim)*(Bre+Bim),
//   Cre = P1 - P2,   Cim = P3 - P1 - P2.
//
// MFMA 16x16x4 operand layout (wave64): lane l supplies A[l%16][l/16] and
// B[l/16][l%16].  Accumulator element v of lane l is D[row][l%16] with
// row = l/16 + 4v for the f64 instruction and row = 4(l/16) + v for f32
// (measured on gfx950).  The kernel passes its B as the first operand, so D
// is the transposed tile: row = column n, l%16 = row m.
#include <algorithm>
#include <array>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <memory>
#include <mutex>
#include <numeric>
#include <type_traits>
#include <unordered_map>

#include "gemm.hpp"

namespace cam {

namespace {

constexpr int KCmax = 16;  // largest K chunk staged in LDS
constexpr int kXcds = 8;   // MI355X accelerator complex dies (one L2 each)

// global-address-space access (global_load / global_store rather than
// flat) through native vector types: HIP's double2/float2 have reference
// constructors that would cast the address back to the flat space
typedef double d2v __attribute__((ext_vector_type(2)));
typedef float f2v __attribute__((ext_vector_type(2)));
template <typename T> struct NV;
template <> struct NV<double2> { using T = d2v; };
template <> struct NV<float2> { using T = f2v; };
template <typename T>
__device__ __forceinline__ T gload(const T* p) {
  using V = typename NV<T>::T;
  const V v = *(const __attribute__((address_space(1))) V*)(p);
  T r;
  r.x = v.x;
  r.y = v.y;
  return r;
}
template <typename T>
__device__ __forceinline__ void gstore(T* p, const T& a) {
  using V = typename NV<T>::T;
  V v;
  v.x = a.x;
  v.y = a.y;
  *(__attribute__((address_space(1))) V*)(p) = v;
}

// The plan (tiles, problems, segments) is read-only for the whole launch:
// reading it through the constant address space lets the compiler use
// scalar loads, whose waits (lgkmcnt) do not also wait for the operand
// prefetch in flight (vmcnt).
template <typename T>
__device__ __forceinline__ T cload(const T* p) {
  static_assert(sizeof(T) % 4 == 0, "plan records are word-sized");
  using W = const __attribute__((address_space(4))) uint32_t*;
  const W q = (W)(p);
  union {
    T t;
    uint32_t w[sizeof(T) / 4];
  } u;
#pragma unroll
  for (int i = 0; i < static_cast<int>(sizeof(T) / 4); ++i) u.w[i] = q[i];
  return u.t;
}

template <typename R> struct CT;
template <> struct CT<double> { using T = double2; };
template <> struct CT<float> { using T = float2; };

template <typename R> struct Mf;
template <> struct Mf<double> {
  typedef double acc __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc mma(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int fk, int v) { return fk + 4 * v; }
};
template <> struct Mf<float> {
  typedef float acc __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc mma(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int fk, int v) { return 4 * fk + v; }
};

// Raw buffer access: wave-uniform 64-bit base in scalar registers plus a
// 32-bit per-lane byte offset.  An offset at or past the record limit reads
// zero without touching memory, which is how elements outside a problem are
// padded.
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));
constexpr uint32_t kBufRecords = 0x7ffffff0u;
constexpr uint32_t kBufOutside = 0x80000000u;
constexpr int kBufFlags = 0x00020000;   // raw 32-bit data format

template <typename R> struct BufRaw;
template <> struct BufRaw<double> {
  using V = d2v;
  static __device__ __forceinline__ V load(const char* base, uint32_t records, uint32_t off) {
    __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, records, kBufFlags);
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
  }
};
template <> struct BufRaw<float> {
  using V = f2v;
  static __device__ __forceinline__ V load(const char* base, uint32_t records, uint32_t off) {
    __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, records, kBufFlags);
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
  }
};

// Waves of a workgroup over its tile: 2 x 2, or eight of them for the wide
// FP64 tiles (a wave's accumulators for more than 32 x 32 FP64 outputs would
// leave one wave per SIMD).
template <typename R, int TM, int TN> struct Waves {
  static constexpr bool kWide = sizeof(R) == 8 && TM * TN > 4096;
  static constexpr int kM = kWide && TM > TN ? 4 : 2;
  static constexpr int kN = kWide && TN > TM ? 4 : 2;
  static constexpr int kThreads = 64 * kM * kN;
};

// G3: complex products with three real MFMAs (P1 = Ar Br, P2 = Ai Bi,
// P3 = (Ar + Ai)(Br + Bi); re = P1 - P2, im = P3 - P1 - P2) instead of four;
// the error stays O(eps |A||B|) per product, as for the four-product form.
// KC = 8 halves the LDS footprint and the prefetch registers (more resident
// workgroups where registers allow) at one barrier per 8 instead of 16 k.
//
// Bound by MFMA issue: a vector instruction of either resident wave stalls the
// matrix pipe for about three cycles (v_add_f64: six or more; an FP64 MFMA
// takes 64, an FP32 one 32; an MFMA-only loop reaches 75.8 TFLOP/s in FP64,
// four 32-bit adds per MFMA 65, eight 56), and two waves per SIMD do not
// cover a wave's staging, barrier and first LDS reads.  So
//  - operands come in through buffer loads with a scalar base advanced by
//    scalar adds and one lane offset per operand; padding is cut off by the
//    record length;
//  - LDS holds interleaved (re, im) pairs: a staged element is one store and
//    a fragment (both parts) one load, without packing or selects;
//  - staging, cursor and loads stand between the MFMA passes of a chunk's
//    first k step, the barrier before its last one.
// About 30 vector instructions per 48 MFMAs are left (16 of them the Gauss
// sums), from over 200.  Coupled chain, d=64, chi=500: FP64 stages L and R
// 49.2 / 48.6 -> 39.1 / 39.6 ms (62.5 -> 78.5 TFLOP/s, pipe busy 0.63 -> 0.79),
// W stages 15.1 / 15.0 -> 12.6 / 12.0 ms (49 GB each: near the copy rate);
// chi=256 FP32 matvec 12.2 -> 9.4 ms.
template <typename R, int TM, int TN, bool G3, int KC>
__global__ __launch_bounds__((Waves<R, TM, TN>::kThreads)) void grouped_gemm_kernel(
    const GemmProb* __restrict__ probs, const GemmSeg* __restrict__ segs, const GemmTile* __restrict__ tiles,
    int ntiles, GemmBases bases) {
  using C = typename CT<R>::T;
  using V = typename BufRaw<R>::V;
  using acc_t = typename Mf<R>::acc;
  constexpr int ES = sizeof(C);
  // one element of padding: the rows of a K-contiguous operand, written at
  // one k per lane, then fall on different banks
  constexpr int LDA = TM + 1;
  constexpr int LDB = TN + 1;
  using WG = Waves<R, TM, TN>;
  constexpr int NT = WG::kThreads;
  constexpr int PA = TM * KC / NT;    // A elements per thread per chunk
  constexpr int PB = TN * KC / NT;    // B elements per thread per chunk
  constexpr int WTM = TM / WG::kM;    // a wave's sub-tile
  constexpr int WTN = TN / WG::kN;
  constexpr int FM = WTM / 16;        // 16-row fragments per wave
  constexpr int FN = WTN / 16;
  static_assert(PA * NT == TM * KC && PB * NT == TN * KC, "a chunk divides evenly over the threads");
  // two LDS buffers: chunk c+1 is stored while chunk c is multiplied, so one
  // barrier per chunk suffices
  __shared__ alignas(16) V sA[2][KC * LDA];
  __shared__ alignas(16) V sB[2][KC * LDB];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WG::kM, wn = wave / WG::kM;
  const int fr = lane & 15, fk = lane >> 4;

  // XCD-aware order: workgroup b runs on XCD b % 8, so consecutive tiles
  // (the M-tiles of one output column block, which read the same B columns)
  // are given to workgroups of the same XCD and share its L2
  const int G = gridDim.x;
  const int v0 = (G % kXcds == 0) ? (blockIdx.x % kXcds) * (G / kXcds) + blockIdx.x / kXcds : blockIdx.x;
  for (int t = v0; t < ntiles; t += G) {
    const GemmTile tl = cload(tiles + t);
    const GemmProb P = cload(probs + tl.prob);
    const int M = P.M, N = P.N;
    const int m0 = tl.m0, n0 = tl.n0;

    // four-product form: accr = re, acci = im; G3: accr = P1, acci = P2,
    // accs = P3
    acc_t accr[FM][FN], acci[FM][FN], accs[G3 ? FM : 1][G3 ? FN : 1];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        accr[i][j] = acc_t{0, 0, 0, 0};
        acci[i][j] = acc_t{0, 0, 0, 0};
        if (G3) accs[G3 ? i : 0][G3 ? j : 0] = acc_t{0, 0, 0, 0};
      }

    // prefetched operands of one chunk
    V ra[PA], rb[PB];
    const int send = P.seg0 + P.nseg;
    // layout of the operands (the same for every segment of a problem)
    const int32_t lay = P.nseg ? cload(segs + P.seg0).flags : 0;
    const bool akc = lay & kSegAKContig, bnc = lay & kSegBNContig;

    // Load cursor: segment, k offset in it, its K and its operands.  A wave's
    // load p covers the 64 consecutive elements 64 wave + kThreads p of the
    // chunk: M-contiguous A runs over the rows of a k, a K-contiguous operand
    // over the k of a row.  A lane's byte offset from the load's scalar base
    // does not depend on p; it spans at most 7 strides (KC = 8, K-contiguous)
    // of less than 2^24 elements, below 2^31 bytes.  Elements outside the
    // problem are cut off by the record length: of a K-contiguous operand the
    // rows past the edge, of an M-contiguous one the k past the segment's end
    // (its rows past the edge have their lane offset outside).
    int cs = P.seg0, ck = 0, csK = 0;
    uint32_t aoff = 0, boff = 0;
    const char* pa = nullptr;           // this wave's load 0 of the chunk
    const char* pb = nullptr;
    int64_t sap = 0, sbp = 0;           // bytes from load p to p + 1
    int64_t sak = 0, sbk = 0;           // bytes from a chunk to the next
    uint32_t lda = 0, ldb = 0;          // bytes of a stride
    const int lk = lane % KC, lr = lane / KC;
    auto setup = [&]() {
      const GemmSeg S = cload(segs + cs);
      csK = S.K;
      const int asp = (S.flags >> 8) & 15, bsp = (S.flags >> 12) & 15;
      const C* A = (asp ? reinterpret_cast<const C*>(bases.p[asp]) + reinterpret_cast<intptr_t>(S.A)
                        : reinterpret_cast<const C*>(S.A)) +
                   static_cast<int64_t>(tl.batch) * S.bsA;
      const C* B = (bsp ? reinterpret_cast<const C*>(bases.p[bsp]) + reinterpret_cast<intptr_t>(S.B)
                        : reinterpret_cast<const C*>(S.B)) +
                   static_cast<int64_t>(tl.batch) * S.bsB;
      const int64_t sA = S.csA * ES, sB = S.ldB * ES;
      lda = static_cast<uint32_t>(sA);
      ldb = static_cast<uint32_t>(sB);
      if (akc) {
        pa = reinterpret_cast<const char*>(A) + (m0 + wave * (64 / KC)) * sA;
        sap = (NT / KC) * sA;
        sak = KC * ES;
        aoff = lr * lda + lk * ES;
      } else {
        pa = reinterpret_cast<const char*>(A + m0 + wave * 64 % TM) + (wave * 64 / TM) * sA;
        sap = (NT / TM) * sA;
        sak = KC * sA;
        aoff = m0 + tid % TM < M ? (TM < 64 ? lane % TM * ES + (lane / TM) * lda : lane * ES) : kBufOutside;
      }
      if (bnc) {
        pb = reinterpret_cast<const char*>(B + n0 + wave * 64 % TN) + (wave * 64 / TN) * sB;
        sbp = (NT / TN) * sB;
        sbk = KC * sB;
        boff = n0 + tid % TN < N ? (TN < 64 ? lane % TN * ES + (lane / TN) * ldb : lane * ES) : kBufOutside;
      } else {
        pb = reinterpret_cast<const char*>(B) + (n0 + wave * (64 / KC)) * sB;
        sbp = (NT / KC) * sB;
        sbk = KC * ES;
        boff = lr * ldb + lk * ES;
      }
    };
    // steps the cursor to the next chunk; false (and K = 0) past the last one
    auto advance = [&]() {
      ck += KC;
      pa += sak;
      pb += sbk;
      if (ck < csK) return true;
      ck = 0;
      csK = 0;
      if (cs + 1 >= send) return false;
      ++cs;
      setup();
      return true;
    };
    // K-contiguous operands: rows (columns) of load p inside the problem
    int arows[PA], bcols[PB];
#pragma unroll
    for (int p = 0; p < PA; ++p)
      arows[p] = __builtin_amdgcn_readfirstlane(min(max(M - m0 - (wave * 64 + p * NT) / KC, 0), 64 / KC));
#pragma unroll
    for (int p = 0; p < PB; ++p)
      bcols[p] = __builtin_amdgcn_readfirstlane(min(max(N - n0 - (wave * 64 + p * NT) / KC, 0), 64 / KC));
    // record length of load p of an operand with T rows (columns) a chunk,
    // `in` of the load's inside the problem, at stride ld
    auto records = [&](bool kc, int T, int in, uint32_t ld, int p, int kleft) -> uint32_t {
      const int k = (wave * 64 + p * NT) / T;
      const uint32_t rk = kleft > 0 ? in * ld : 0;
      const uint32_t rm = k < kleft ? (T < 64 && k + 1 >= kleft ? ld : kBufRecords) : 0;
      return __builtin_amdgcn_readfirstlane(kc ? rk : rm);
    };
    // loads of the chunk at the cursor (past the last one: nothing)
    auto load = [&]() {
      const int kleft = csK - ck;
      const uint32_t ao = akc && lk >= kleft ? kBufOutside : aoff;
      const uint32_t bo = !bnc && lk >= kleft ? kBufOutside : boff;
#pragma unroll
      for (int p = 0; p < PA; ++p)
        ra[p] = BufRaw<R>::load(pa + p * sap, records(akc, TM, arows[p], lda, p, kleft), ao);
#pragma unroll
      for (int p = 0; p < PB; ++p)
        rb[p] = BufRaw<R>::load(pb + p * sbp, records(!bnc, TN, bcols[p], ldb, p, kleft), bo);
    };
    // stages the loaded chunk, conjugated where the problem asks for it (H_eff
    // problems do not)
    auto stage = [&](int buf, auto conj) {
      const bool cA = decltype(conj)::value && (lay & kSegConjA), cB = decltype(conj)::value && (lay & kSegConjB);
      V* __restrict__ dA = sA[buf];
      V* __restrict__ dB = sB[buf];
      if (akc) {
#pragma unroll
        for (int p = 0; p < PA; ++p)
          dA[(tid % KC) * LDA + tid / KC + p * (NT / KC)] = V{ra[p].x, cA ? -ra[p].y : ra[p].y};
      } else {
#pragma unroll
        for (int p = 0; p < PA; ++p)
          dA[(tid / TM + p * (NT / TM)) * LDA + tid % TM] = V{ra[p].x, cA ? -ra[p].y : ra[p].y};
      }
      if (bnc) {
#pragma unroll
        for (int p = 0; p < PB; ++p)
          dB[(tid / TN + p * (NT / TN)) * LDB + tid % TN] = V{rb[p].x, cB ? -rb[p].y : rb[p].y};
      } else {
#pragma unroll
        for (int p = 0; p < PB; ++p)
          dB[(tid % KC) * LDB + tid / KC + p * (NT / KC)] = V{rb[p].x, cB ? -rb[p].y : rb[p].y};
      }
    };
    auto store = [&](int buf) {
      if (lay & (kSegConjA | kSegConjB)) stage(buf, std::true_type{});
      else stage(buf, std::false_type{});
    };

    // fragments of one k step (four k), double buffered in registers
    V fa[2][FM], fb[2][FN];
    auto frag = [&](int buf, int ks, int slot) {
      const int kr = ks * 4 + fk;
#pragma unroll
      for (int i = 0; i < FM; ++i) fa[slot][i] = sA[buf][kr * LDA + wm * WTM + fr + i * 16];
#pragma unroll
      for (int j = 0; j < FN; ++j) fb[slot][j] = sB[buf][kr * LDB + wn * WTN + fr + j * 16];
    };
    // One pass of a k step's MFMAs over the fragments, FM*FN of them on
    // different accumulators (three passes with G3, else four).  B is the
    // instruction's first operand: the accumulator's lanes then run along m,
    // and a store instruction writes 16 consecutive rows.
    auto pass = [&](int slot, int w) {
      R sb[FN];
#pragma unroll
      for (int j = 0; j < FN; ++j) sb[j] = fb[slot][j].x + fb[slot][j].y;
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const V a = fa[slot][i];
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const V b = fb[slot][j];
          if constexpr (G3) {
            if (w == 0) accr[i][j] = Mf<R>::mma(b.x, a.x, accr[i][j]);
            if (w == 1) acci[i][j] = Mf<R>::mma(b.y, a.y, acci[i][j]);
            if (w == 2) accs[i][j] = Mf<R>::mma(sb[j], a.x + a.y, accs[i][j]);
          } else {
            if (w == 0) accr[i][j] = Mf<R>::mma(b.x, a.x, accr[i][j]);
            if (w == 1) acci[i][j] = Mf<R>::mma(b.y, a.x, acci[i][j]);
            if (w == 2) accr[i][j] = Mf<R>::mma(b.y, -a.y, accr[i][j]);
            if (w == 3) acci[i][j] = Mf<R>::mma(b.x, a.y, acci[i][j]);
          }
        }
      }
    };
    constexpr int kPasses = G3 ? 3 : 4;
    constexpr int KS = KC / 4;
    if (cs < send) {
      setup();
      load();
      store(0);
      bool more = advance();            // whether the registers hold a chunk
      load();
      __syncthreads();
      frag(0, 0, 0);
      // While chunk c is multiplied, chunk c + 1 (in the registers) is staged
      // into the other LDS buffer and chunk c + 2 loaded; both stand between
      // MFMA passes.  The barrier stands before the last k step, whose
      // fragments are in registers by then, and the next chunk's first
      // fragments are read ahead of that step's MFMAs, so that neither wait
      // leaves the pipe idle.  Nothing here is conditional: past the last
      // chunk the loads read nothing, and what they stage is not used.
      for (int buf = 0;; buf ^= 1) {
        bool next = false;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const int cur = ks & 1;
          if (ks + 1 < KS) {
            frag(buf, ks + 1, cur ^ 1);
          } else {
            // (the scheduler would move the step's MFMAs ahead of the barrier)
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            frag(buf ^ 1, 0, cur ^ 1);
            __builtin_amdgcn_sched_barrier(0);
          }
          pass(cur, 0);
          // the other LDS buffer was last read before the previous barrier
          if (ks == 0) store(buf ^ 1);
          pass(cur, 1);
          if (ks == 0) next = advance();
          pass(cur, 2);
          if (ks == 0) load();
          if (kPasses == 4) pass(cur, 3);
        }
        if (!more) break;
        more = next;
      }
    }

    // epilogue
    C* Cp = (P.cspace ? reinterpret_cast<C*>(const_cast<void*>(bases.p[P.cspace])) +
                            reinterpret_cast<intptr_t>(P.C)
                      : reinterpret_cast<C*>(P.C)) +
            static_cast<int64_t>(tl.batch) * P.bsC;
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int n = n0 + wn * WTN + j * 16 + Mf<R>::row(fk, v);
        if (n >= N) continue;
        C* col = Cp + static_cast<int64_t>(n) * P.csC;
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          const int m = m0 + wm * WTM + i * 16 + fr;
          if (m < M) {
            C val;
            if constexpr (G3) {
              const R p1 = accr[i][j][v], p2 = acci[i][j][v];
              val.x = p1 - p2;
              val.y = accs[i][j][v] - p1 - p2;
            } else {
              val.x = accr[i][j][v];
              val.y = acci[i][j][v];
            }
            if (P.beta) {
              const C old = gload(col + m);
              val.x += old.x;
              val.y += old.y;
            }
            gstore(col + m, val);
          }
        }
      }
    // the next tile's first chunk overwrites an LDS buffer of this one
    __syncthreads();
  }
}

// Row pass: `rows` rows of nin input columns times an nin x nout matrix, for
// N <= 16 problems with short segments (the W stages and environments of
// small QN sectors), where an output tile per problem would be mostly padding
// and every output channel would read the input rows again.
// Bound by HBM: per row (nin + nout) elements move for at most 64 x 64
// complex products, which take as long on the matrix cores; so all problems
// that read the same columns share a pass (a U(1) MPO with six channels and
// sectors of 4-5 levels: one pass of 27 x 27 instead of six problems of
// 27 x 5), and a wave streams 16 rows at a time from memory straight into
// MFMA operands, eight k steps (8 KB in FP64) in flight, without LDS or
// barriers.  The matrix is staged in LDS once per item, gathered by all
// threads at once through the pass's tables; rows run on over the batch
// members (they share B), so small row counts still fill the wave.
// U(1) chain, d=32, chi=1024: W stages 9.6 / 9.2 ms with one thread per row
// and problem -> 3.63 / 3.55 ms (12.9 GB to move each: 3.6 TB/s; a large copy
// reaches 4.8); chain d=64, chi=32: stage R (16 x 16 blocks, 1024 batch
// members) 0.74 -> 0.035 ms; spin chain chi=16: matvec 31 -> 21 us.
constexpr int kRowThreads = 256;
constexpr int kRowWaves = kRowThreads / 64;

template <typename R, int NT>
__device__ __forceinline__ void row_pass(const RowItem& it, const typename CT<R>::T* sB,
                                         const typename CT<R>::T* const* sInP, const int64_t* sInS,
                                         typename CT<R>::T* const* sOutP, const int64_t* sOutS) {
  using C = typename CT<R>::T;
  using V = typename NV<C>::T;
  using acc_t = typename Mf<R>::acc;
  constexpr int NP = 16 * NT, U = 8;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int fr = lane & 15, fk = lane >> 4;
  const int nks = (it.nin + 3) / 4;
  for (int c0 = wave * 16; c0 < it.rows; c0 += kRowWaves * 16) {
    // rows past the item repeat its last one and are not stored
    const bool live = c0 + fr < it.rows;
    const uint32_t t = static_cast<uint32_t>(it.m0) + static_cast<uint32_t>(min(c0 + fr, it.rows - 1));
    const uint32_t q = t / static_cast<uint32_t>(it.M);
    const int64_t b = it.batch0 + static_cast<int64_t>(q);
    const int64_t m = t - q * static_cast<uint32_t>(it.M);
    acc_t cr[NT], ci[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) cr[j][v] = ci[j][v] = R(0);
    for (int k0 = 0; k0 < nks; k0 += U) {
      V a[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = min((k0 + u) * 4 + fk, it.nin - 1);
        a[u] = *(const __attribute__((address_space(1))) V*)(sInP[k] + (b * sInS[k] + m));
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (k0 + u >= nks) break;
        const int k = (k0 + u) * 4 + fk;
        const bool in = k < it.nin;
        const R ar = in ? a[u].x : R(0);
        const R ai = in ? (it.conjA ? -a[u].y : a[u].y) : R(0);
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const C bv = sB[k * NP + j * 16 + fr];
          cr[j] = Mf<R>::mma(bv.x, ar, cr[j]);
          ci[j] = Mf<R>::mma(bv.x, ai, ci[j]);
          cr[j] = Mf<R>::mma(-bv.y, ai, cr[j]);
          ci[j] = Mf<R>::mma(bv.y, ar, ci[j]);
        }
      }
    }
    if (live) {
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int n = j * 16 + Mf<R>::row(fk, v);
          if (n >= it.nout) continue;
          C* dst = sOutP[n] + (b * sOutS[n] + m);
          C val;
          val.x = cr[j][v];
          val.y = ci[j][v];
          if (it.beta) {
            const C old = gload(dst);
            val.x += old.x;
            val.y += old.y;
          }
          gstore(dst, val);
        }
    }
  }
}

template <typename R>
__global__ __launch_bounds__(kRowThreads) void row_gemm_kernel(const RowItem* __restrict__ items, int nitems,
                                                               const RowIn* __restrict__ ins,
                                                               const RowOut* __restrict__ outs,
                                                               const RowBlk* __restrict__ blks, GemmBases bases) {
  using C = typename CT<R>::T;
  extern __shared__ __align__(16) char smem[];
  C* sB = reinterpret_cast<C*>(smem);          // [padded nin][16 NT]
  __shared__ const C* sInP[kRowIn];
  __shared__ int64_t sInS[kRowIn];
  __shared__ int sInB[kRowIn];                 // first block of the column's segment
  __shared__ int sInK[kRowIn];
  __shared__ C* sOutP[kRowOut];
  __shared__ int64_t sOutS[kRowOut];
  __shared__ int sOutB[kRowOut], sOutN[kRowOut];
  const int tid = threadIdx.x;
  // XCD-aware order, as for the tiles: consecutive items (passes over the
  // same rows) go to workgroups of one XCD, whose L2 serves repeated reads
  const int Gd = gridDim.x;
  const int v0 = (Gd % kXcds == 0) ? (blockIdx.x % kXcds) * (Gd / kXcds) + blockIdx.x / kXcds : blockIdx.x;
  for (int i = v0; i < nitems; i += Gd) {
    const RowItem it = cload(items + i);
    const C* ab = it.aspace ? reinterpret_cast<const C*>(bases.p[it.aspace]) : nullptr;
    const C* bb = it.bspace ? reinterpret_cast<const C*>(bases.p[it.bspace]) : nullptr;
    C* cb = it.cspace ? reinterpret_cast<C*>(const_cast<void*>(bases.p[it.cspace])) : nullptr;
    if (i != v0) __syncthreads();              // the previous item's tables are no longer read
    if (tid < it.nin) {
      const RowIn e = ins[it.in0 + tid];
      sInP[tid] = (it.aspace ? ab + e.off : reinterpret_cast<const C*>(e.off)) + e.kcs;
      sInS[tid] = e.bs;
      sInB[tid] = it.blk0 + e.seg * it.nprob;
      sInK[tid] = e.k;
    } else if (tid >= kRowThreads - kRowOut && tid - (kRowThreads - kRowOut) < it.nout) {
      const int n = tid - (kRowThreads - kRowOut);
      const RowOut e = outs[it.out0 + n];
      sOutP[n] = (it.cspace ? cb + e.off : reinterpret_cast<C*>(e.off)) + e.ncs;
      sOutS[n] = e.bs;
      sOutB[n] = e.prob;
      sOutN[n] = e.n;
    }
    __syncthreads();
    const int nt = (it.nout + 15) / 16, np = 16 * nt;
    const int tot = (it.nin + 3) / 4 * 4 * np;
    for (int e = tid; e < tot; e += kRowThreads) {
      const int k = e / np, n = e % np;
      C v;
      v.x = v.y = R(0);
      if (k < it.nin && n < it.nout) {
        const RowBlk B = blks[sInB[k] + sOutB[n]];
        const C* Bp = it.bspace ? bb + B.off : reinterpret_cast<const C*>(B.off);
        const int64_t kk = sInK[k], nn = sOutN[n];
        v = gload(Bp + ((B.flags & kSegBNContig) ? kk * B.ld + nn : kk + nn * B.ld));
        if (B.flags & kSegConjB) v.y = -v.y;
      }
      sB[e] = v;
    }
    __syncthreads();
    if (nt == 1) row_pass<R, 1>(it, sB, sInP, sInS, sOutP, sOutS);
    else if (nt == 2) row_pass<R, 2>(it, sB, sInP, sInS, sOutP, sOutS);
    else if (nt == 3) row_pass<R, 3>(it, sB, sInP, sInS, sOutP, sOutS);
    else row_pass<R, 4>(it, sB, sInP, sInS, sOutP, sOutS);
  }
}

template <typename R>
void launch_rows(const GemmPlan& plan, hipStream_t s, int grid_limit, const GemmBases& bases) {
  const int n = static_cast<int>(plan.rows.size());
  if (!n) return;
  static int cus = device_cu_count();
  int grid = std::min(n, cus * 8);
  if (grid_limit > 0) grid = std::min(grid, grid_limit);
  const size_t lds = static_cast<size_t>(plan.row_lds) * sizeof(typename CT<R>::T);
  hipLaunchKernelGGL((row_gemm_kernel<R>), dim3(grid), dim3(kRowThreads), lds, s, plan.d_rows, n, plan.d_row_in,
                     plan.d_row_out, plan.d_row_blk, bases);
  HIP_CHECK(hipGetLastError());
}

// Small plans: a workgroup's eight waves split the k steps of a 16 x 16 tile
// of outputs, or of two, four or eight of them next to each other where K is
// short.  Bound by latency: a tile of the persistent
// kernel walks K in chunks of 16, each a memory round trip and a barrier that
// nothing else on the compute unit covers when there are few tiles, and the
// tile shapes and row passes are separate launches.  Here every wave has all
// operands of eight k steps (16 KB) in flight straight into MFMA operands, and
// the partial sums meet in LDS once.  Without operand reuse it reads
// 32 elements per k of a tile, from L2 while the plan is small.
// Spin chain, chi=200: stages L and R 34 and 72 us in up to four launches each
// -> 15 and 10 us, matvec 115 -> 32 us.
constexpr int kDirectWaves = 8;

// waves that share the k steps of a tile: eight steps each while there are
// enough waves
__host__ __device__ inline int direct_split(int64_t steps) {
  return steps <= 8 ? 1 : steps <= 16 ? 2 : steps <= 32 ? 4 : kDirectWaves;
}

template <typename R>
__global__ __launch_bounds__(64 * kDirectWaves) void direct_gemm_kernel(const GemmProb* __restrict__ probs,
                                                                        const GemmSeg* __restrict__ segs,
                                                                        const GemmTile* __restrict__ tiles, int ntiles,
                                                                        GemmBases bases) {
  using C = typename CT<R>::T;
  using acc_t = typename Mf<R>::acc;
  constexpr int U = 8;
  __shared__ const C* sA[kDirectSegs];
  __shared__ const C* sB[kDirectSegs];
  __shared__ int64_t sLa[kDirectSegs], sLb[kDirectSegs];
  __shared__ int sK[kDirectSegs], sStep[kDirectSegs + 1];
  __shared__ C sum[kDirectWaves][256];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fk = lane >> 4;
  const int Gd = gridDim.x;
  const int v0 = (Gd % kXcds == 0) ? (blockIdx.x % kXcds) * (Gd / kXcds) + blockIdx.x / kXcds : blockIdx.x;
  for (int t = v0; t < ntiles; t += Gd) {
    const GemmTile tl = cload(tiles + t);
    const GemmProb P = cload(probs + tl.prob);
    if (t != v0) __syncthreads();              // the previous tile's tables and sums are no longer read
    if (tid < 64) {
      int k = 0;
      if (tid < P.nseg) {
        const GemmSeg S = segs[P.seg0 + tid];
        const int asp = (S.flags >> 8) & 15, bsp = (S.flags >> 12) & 15;
        sA[tid] = (asp ? reinterpret_cast<const C*>(bases.p[asp]) + reinterpret_cast<intptr_t>(S.A)
                       : reinterpret_cast<const C*>(S.A)) +
                  static_cast<int64_t>(tl.batch) * S.bsA;
        sB[tid] = (bsp ? reinterpret_cast<const C*>(bases.p[bsp]) + reinterpret_cast<intptr_t>(S.B)
                       : reinterpret_cast<const C*>(S.B)) +
                  static_cast<int64_t>(tl.batch) * S.bsB;
        sLa[tid] = S.csA;
        sLb[tid] = S.ldB;
        sK[tid] = k = S.K;
      }
      int st = (k + 3) / 4;                    // inclusive scan of the segments' k steps
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(st, o, 64);
        if (lane >= o) st += v;
      }
      sStep[tid + 1] = st;
      if (tid == 0) sStep[0] = 0;
    }
    const int32_t lay = P.nseg ? cload(segs + P.seg0).flags : 0;
    const bool akc = lay & kSegAKContig, bnc = lay & kSegBNContig;
    __syncthreads();
    const int total = P.nseg ? sStep[P.nseg] : 0;
    const int split = direct_split(total), share = wave % split;
    const int nt = tl.n0 + wave / split * 16;  // this wave's tile
    const int s_end = nt < P.N ? static_cast<int>(int64_t(total) * (share + 1) / split) : 0;
    // rows and columns past the edge repeat the last one and are not stored
    const int64_t m = min(tl.m0 + fr, P.M - 1), n = min(nt + fr, P.N - 1);
    acc_t re{0, 0, 0, 0}, im{0, 0, 0, 0};
    for (int s0 = static_cast<int>(int64_t(total) * share / split); s0 < s_end; s0 += U) {
      // lane u finds the segment of step s0 + u
      const int mine = min(s0 + (lane & (U - 1)), s_end - 1);
      int lo = 0, hi = P.nseg - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (sStep[mid] <= mine) lo = mid;
        else hi = mid - 1;
      }
      const int kk = (mine - sStep[lo]) * 4;
      C a[U], b[U];
      bool in[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = __builtin_amdgcn_readlane(lo, u);
        const int k0 = __builtin_amdgcn_readlane(kk, u) + fk, K = sK[j];
        const int64_t k = min(k0, K - 1);
        in[u] = k0 < K && s0 + u < s_end;
        a[u] = gload(sA[j] + (akc ? k + m * sLa[j] : m + k * sLa[j]));
        b[u] = gload(sB[j] + (bnc ? n + k * sLb[j] : k + n * sLb[j]));
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const R ar = in[u] ? a[u].x : R(0), br = in[u] ? b[u].x : R(0);
        R ai = in[u] ? a[u].y : R(0), bi = in[u] ? b[u].y : R(0);
        if (lay & kSegConjA) ai = -ai;
        if (lay & kSegConjB) bi = -bi;
        re = Mf<R>::mma(br, ar, re);
        im = Mf<R>::mma(br, ai, im);
        re = Mf<R>::mma(-bi, ai, re);
        im = Mf<R>::mma(bi, ar, im);
      }
    }
    // element v of a lane is column row(fk, v), row fr
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      C c;
      c.x = re[v];
      c.y = im[v];
      sum[wave][Mf<R>::row(fk, v) * 16 + fr] = c;
    }
    __syncthreads();
    for (int e = tid; e < 256 * (kDirectWaves / split); e += 64 * kDirectWaves) {
      const int g = e >> 8, o = e & 255;
      const int mm = tl.m0 + (o & 15), nn = tl.n0 + g * 16 + (o >> 4);
      if (mm >= P.M || nn >= P.N) continue;
      C c = sum[g * split][o];
      for (int w = 1; w < split; ++w) {
        c.x += sum[g * split + w][o].x;
        c.y += sum[g * split + w][o].y;
      }
      C* dst = (P.cspace ? reinterpret_cast<C*>(const_cast<void*>(bases.p[P.cspace])) + reinterpret_cast<intptr_t>(P.C)
                         : reinterpret_cast<C*>(P.C)) +
               (static_cast<int64_t>(tl.batch) * P.bsC + mm + static_cast<int64_t>(nn) * P.csC);
      if (P.beta) {
        const C old = gload(dst);
        c.x += old.x;
        c.y += old.y;
      }
      gstore(dst, c);
    }
  }
}

template <typename R>
void launch_direct(const GemmPlan& plan, hipStream_t s, int grid_limit, const GemmBases& bases) {
  const int n = static_cast<int>(plan.direct.size());
  static int cus = device_cu_count();
  int grid = std::min(n, cus * 4);
  if (grid_limit > 0) grid = std::min(grid, grid_limit);
  hipLaunchKernelGGL((direct_gemm_kernel<R>), dim3(grid), dim3(64 * kDirectWaves), 0, s, plan.d_probs,
                     plan.d_segs, plan.d_direct, n, bases);
  HIP_CHECK(hipGetLastError());
}

template <typename R, int TM, int TN>
void launch_shape(const GemmPlan& plan, const LaunchCfg& c, int shape, hipStream_t s, int grid_limit,
                  const GemmBases& bases) {
  const int nt = static_cast<int>(plan.tiles[c.tile_mode][shape].size());
  if (!nt) return;
  static int cus = device_cu_count();
  int grid = std::min(nt, cus * std::max(1, c.wg_per_cu));
  if (grid_limit > 0) grid = std::min(grid, grid_limit);
  const GemmTile* tiles = plan.d_tiles[c.tile_mode][shape];
  const GemmProb* P = plan.d_probs;
  const GemmSeg* S = plan.d_segs;
  auto go = [&](auto g3, auto kc) {
    hipLaunchKernelGGL((grouped_gemm_kernel<R, TM, TN, decltype(g3)::value, decltype(kc)::value>), dim3(grid),
                       dim3(Waves<R, TM, TN>::kThreads), 0, s, P, S, tiles, nt, bases);
  };
  using K8 = std::integral_constant<int, 8>;
  using K16 = std::integral_constant<int, 16>;
  if (c.algo == kAlgo3M) c.kc == 8 ? go(std::true_type{}, K8{}) : go(std::true_type{}, K16{});
  else c.kc == 8 ? go(std::false_type{}, K8{}) : go(std::false_type{}, K16{});
  HIP_CHECK(hipGetLastError());
}

}  // namespace

int device_cu_count() {
  int dev = 0;
  HIP_CHECK(hipGetDevice(&dev));
  hipDeviceProp_t prop;
  HIP_CHECK(hipGetDeviceProperties(&prop, dev));
  return prop.multiProcessorCount;
}

int GemmPlan::add_problem(void* C, int64_t csC, int M, int N, int batch, int64_t bsC, int beta,
                          int cspace) {
  GemmProb p{};
  p.C = C;
  p.csC = csC;
  p.bsC = bsC;
  p.M = M;
  p.N = N;
  p.seg0 = static_cast<int32_t>(segs.size());
  p.nseg = 0;
  p.batch = batch;
  p.beta = beta;
  p.cspace = cspace;
  probs.push_back(p);
  group.push_back(-1);
  uploaded = false;
  changed();
  return static_cast<int>(probs.size()) - 1;
}

void GemmPlan::changed() {
  rows_built = direct_uploaded = false;
  direct.clear();
  for (int m = 0; m < kTileModes; ++m) built[m] = tiles_uploaded[m] = false;
}

void GemmPlan::set_group(int prob, int64_t g) {
  CAM_REQUIRE(prob >= 0 && prob < static_cast<int>(probs.size()), "set_group: no such problem");
  group[prob] = g;
  changed();
}

void GemmPlan::add_segment(int prob, const void* A, int64_t csA, int64_t bsA, const void* B,
                           int64_t ldB, int64_t bsB, int K, int flags) {
  if (K <= 0) return;   // contributes nothing; the kernels assume K >= 1
  GemmProb& p = probs[prob];
  CAM_REQUIRE(p.seg0 + p.nseg == static_cast<int32_t>(segs.size()),
              "segments of a problem must be added contiguously");
  // the kernels address an element of a load by a 32-bit byte offset (at most
  // seven strides of 16-byte elements) and cut padding off by record lengths
  // that count whole strides
  constexpr int64_t kStrideLimit = (int64_t(1) << 24) - 2;
  CAM_REQUIRE(csA >= 0 && ldB >= 0 && csA <= kStrideLimit && ldB <= kStrideLimit,
              "add_segment: operand stride too large for 32-bit tile offsets");
  CAM_REQUIRE(csA >= ((flags & kSegAKContig) ? K : p.M) && ldB >= ((flags & kSegBNContig) ? p.N : K),
              "add_segment: operand stride below the contiguous extent");
  GemmSeg g{};
  g.A = A;
  g.B = B;
  g.csA = csA;
  g.ldB = ldB;
  g.bsA = bsA;
  g.bsB = bsB;
  g.K = K;
  g.flags = flags;
  // the kernels read layout and conjugation once per problem
  CAM_REQUIRE(p.nseg == 0 || ((segs[p.seg0].flags ^ g.flags) & 0xff) == 0,
              "segments of a problem must share their layout and conjugation flags");
  segs.push_back(g);
  p.nseg++;
  flops += 8.0 * double(p.M) * double(p.N) * double(K) * double(p.batch);
  uploaded = false;
  changed();
}

void GemmPlan::choose_tiles(int mode) {
  CAM_REQUIRE(mode >= 0 && mode < kTileModes, "unknown tile mode");
  cfg[0].tile_mode = cfg[1].tile_mode = mode;
}

// Row pass or tiles: N <= 16 and K <= 32 per segment (see GemmPlan::rows).
// Below the line the tiles lose: U(1) chi=1024 W stages 15.4 ms against 3.6,
// spin chain chi=200 W stages 50 us against 9, chain d=64 chi=32 stage R 0.128
// ms against 0.035.  Above it the passes do: they take four products where
// the tiles take three and re-read B per 16 rows; with N up to 32 the W stages
// of the d=64 chain run at 24 TFLOP/s against 44-55 (chi=64, 97, 500), FP32 54
// against 90 (chi=256).
static bool row_eligible(const GemmPlan& plan, const GemmProb& p) {
  static const bool off = [] {
    const char* e = std::getenv("CAM_SKINNY");
    return e && *e == '0';
  }();
  if (off || p.N > kRowN || p.nseg == 0 || p.M <= 0 || p.N <= 0) return false;
  int64_t k = 0;
  const GemmSeg& g0 = plan.segs[p.seg0];
  for (int s = p.seg0; s < p.seg0 + p.nseg; ++s) {
    const GemmSeg& g = plan.segs[s];
    if (g.K > kRowK || (g.flags & kSegAKContig) || ((g.flags ^ g0.flags) >> 8)) return false;
    if (g.bsB && p.batch > 1) return false;   // one matrix for all rows
    k += g.K;
  }
  return k <= kRowIn;
}

// tile shape of a problem under a policy
static int tile_shape(const GemmProb& p, int mode) {
  int shape = 0;
  if (mode == 0) return shape;
  double best = 1e300;
  const int t_end = mode == 3 ? kNumTileShapes : kNumSmallShapes;
  for (int t = (mode == 2 ? 1 : 0); t < t_end; ++t) {
    const double tm = kTileShapes[t].tm, tn = kTileShapes[t].tn;
    const double pm = std::ceil(p.M / tm) * tm, pn = std::ceil(p.N / tn) * tn;
    // padded area, with a small per-tile overhead so bigger tiles win ties
    const double c = pm * pn * (1.0 + 0.02 * (4096.0 / (tm * tn)));
    if (c < best) { best = c; shape = t; }
  }
  return shape;
}

// Small plan, or tiles and row passes: whichever the latencies measured on
// small spin and coupled chains make shorter (microseconds).  A tile launch
// takes 5 and 1.4 per chunk of its longest K, a row pass 5; the direct kernel 7
// for the first 1024 work items (what the chip holds) and 4 for every further
// 1024, 2 per eight k steps of its longest wave, and 0.2 per 1000 k steps of all
// tiles (operands from L2); a tenth must be gained.  Stage L / R of the spin chain, tiles against
// direct: chi=50 10.6 / 13.0 and 10.7 / 13.1, 100 14.5 / 25.0 and 9.2 / 9.7, 200
// 34.3 / 71.7 and 15.4 / 10.2, 400 57 / 139 and 41 / 26, 800 114 / 213 and 186 /
// 150; 8-level chain chi=24 7.9 and 10.5 (L), 64 14.0 and 11.7 (R); 8-level U(1)
// chain chi=64 (thousands of tiny problems) 14 and 48 (L).
bool GemmPlan::build_direct() {
  direct.clear();
  direct_uploaded = false;
  static const bool off = [] {
    const char* e = std::getenv("CAM_DIRECT");
    return e && *e == '0';
  }();
  if (off) return false;
  auto steps_of = [&](const GemmProb& p) {
    int64_t st = 0;
    for (int q = p.seg0; q < p.seg0 + p.nseg; ++q) st += (segs[q].K + 3) / 4;
    return st;
  };
  int64_t items = 0, steps = 0, wave_steps = 0, chunks[kNumTileShapes];
  std::fill(std::begin(chunks), std::end(chunks), int64_t(-1));
  bool rows_any = false, tiles_any = false;
  for (const GemmProb& p : probs) {
    if (p.M <= 0 || p.N <= 0 || p.batch <= 0) continue;
    if (p.nseg > kDirectSegs) return false;
    const int64_t st = steps_of(p);
    const int split = direct_split(st), tn = 16 * (kDirectWaves / split);
    const int64_t tm = (p.M + 15) / 16;
    items += p.batch * tm * ((p.N + tn - 1) / tn);
    steps += p.batch * tm * ((p.N + 15) / 16) * st;
    wave_steps = std::max(wave_steps, (st + split - 1) / split);
    if (row_eligible(*this, p)) {
      rows_any = true;
    } else {
      tiles_any = true;
      int64_t& c = chunks[tile_shape(p, 1)];
      int64_t n = 0;
      for (int q = p.seg0; q < p.seg0 + p.nseg; ++q) n += (segs[q].K + KCmax - 1) / KCmax;
      c = std::max(c, n);
    }
    if (items > (1 << 16)) return false;
  }
  if (!tiles_any) return false;
  double tiled = rows_any ? 5.0 : 0.0;
  for (int64_t c : chunks)
    if (c >= 0) tiled += 5.0 + 1.4 * static_cast<double>(c);
  const double one = 7.0 + 4.0 * static_cast<double>((items - 1) / 1024) + 2.0 * static_cast<double>((wave_steps + 7) / 8) +
                     2e-4 * static_cast<double>(steps);
  if (1.1 * one >= tiled) return false;
  direct.reserve(static_cast<size_t>(items));
  for (size_t pi = 0; pi < probs.size(); ++pi) {
    const GemmProb& p = probs[pi];
    if (!p.nseg && p.beta) continue;   // nothing to add
    const int tn = 16 * (kDirectWaves / direct_split(steps_of(p)));
    for (int b = 0; b < p.batch; ++b)
      for (int n0 = 0; n0 < p.N; n0 += tn)
        for (int m0 = 0; m0 < p.M; m0 += 16) direct.push_back(GemmTile{static_cast<int32_t>(pi), b, m0, n0});
  }
  return !direct.empty();
}

void GemmPlan::build_tiles() {
  if (build_direct()) return;
  build_tiles_mode(cfg[0].tile_mode);
  if (cfg[1].tile_mode != cfg[0].tile_mode) build_tiles_mode(cfg[1].tile_mode);
}

// Passes: problems with the same rows and the same input columns, up to
// kRowOut output columns and kRowB matrix elements each.  (Problems with
// different inputs are not merged: a channel that an output does not read
// must not reach it, not even as zero times infinity.)
void GemmPlan::build_rows(const std::vector<int>& eligible) {
  row_in.clear();
  row_out.clear();
  row_blk.clear();
  rows.clear();
  row_lds = 0;
  rows_built = true;
  rows_uploaded = false;
  if (eligible.empty()) return;
  struct Pass { std::vector<int> probs; int nout = 0; };
  std::vector<Pass> passes;
  constexpr int32_t kPerProblem = kSegConjB | kSegBNContig;   // B's layout may differ within a pass
  auto same_inputs = [&](const GemmProb& x, const GemmProb& y) {
    if (x.M != y.M || x.batch != y.batch || x.beta != y.beta || x.cspace != y.cspace || x.nseg != y.nseg) return false;
    for (int j = 0; j < x.nseg; ++j) {
      const GemmSeg &f = segs[x.seg0 + j], &g = segs[y.seg0 + j];
      if (f.A != g.A || f.csA != g.csA || f.bsA != g.bsA || f.K != g.K || ((f.flags ^ g.flags) & ~kPerProblem))
        return false;
    }
    return true;
  };
  std::unordered_multimap<uint64_t, int> open;   // hash of the inputs -> pass still being filled
  open.reserve(eligible.size());
  for (int pi : eligible) {
    const GemmProb& p = probs[pi];
    uint64_t h = 1469598103934665603ull;
    auto mix = [&h](uint64_t v) { h = (h ^ v) * 1099511628211ull; };
    mix(static_cast<uint64_t>(p.M));
    mix(static_cast<uint64_t>(p.batch));
    int nin = 0;
    for (int s = p.seg0; s < p.seg0 + p.nseg; ++s) {
      mix(reinterpret_cast<uint64_t>(segs[s].A));
      nin += segs[s].K;
    }
    const int kp = (nin + 3) / 4 * 4;
    const auto range = open.equal_range(h);
    auto it = range.first;
    while (it != range.second && !same_inputs(p, probs[passes[it->second].probs[0]])) ++it;
    if (it == range.second) {
      it = open.emplace(h, static_cast<int>(passes.size()));
      passes.emplace_back();
    } else {
      const int no = passes[it->second].nout + p.N;
      if (no > kRowOut || kp * ((no + 15) / 16 * 16) > kRowB) {
        it->second = static_cast<int>(passes.size());
        passes.emplace_back();
      }
    }
    passes[it->second].probs.push_back(pi);
    passes[it->second].nout += p.N;
  }
  // rows per item: long enough to pay for staging the matrix, short enough
  // for several items per compute unit
  int64_t total = 0;
  for (const Pass& q : passes) total += int64_t(probs[q.probs[0]].M) * probs[q.probs[0]].batch;
  int per = 1024;
  while (per > 16 * kRowWaves && total / per < 2048) per /= 2;
  size_t nins = 0, nouts = 0, nblks = 0;
  for (const Pass& q : passes) {
    const GemmProb& p0 = probs[q.probs[0]];
    for (int j = 0; j < p0.nseg; ++j) nins += static_cast<size_t>(segs[p0.seg0 + j].K);
    nouts += static_cast<size_t>(q.nout);
    nblks += q.probs.size() * static_cast<size_t>(p0.nseg);
  }
  row_in.reserve(nins);
  row_out.reserve(nouts);
  row_blk.reserve(nblks);
  std::vector<RowItem> first(passes.size());     // a pass's tables, without rows
  for (size_t qi = 0; qi < passes.size(); ++qi) {
    const Pass& q = passes[qi];
    const GemmProb& p0 = probs[q.probs[0]];
    const GemmSeg& g0 = segs[p0.seg0];
    RowItem it{};
    it.in0 = static_cast<int>(row_in.size());
    it.out0 = static_cast<int>(row_out.size());
    it.blk0 = static_cast<int>(row_blk.size());
    for (int j = 0; j < p0.nseg; ++j) {
      const GemmSeg& g = segs[p0.seg0 + j];
      for (int k = 0; k < g.K; ++k)
        row_in.push_back(RowIn{reinterpret_cast<int64_t>(g.A), k * g.csA, g.bsA, j, k});
      for (int pi : q.probs) {
        const GemmSeg& gp = segs[probs[pi].seg0 + j];
        row_blk.push_back(RowBlk{reinterpret_cast<int64_t>(gp.B), static_cast<int32_t>(gp.ldB), gp.flags});
      }
    }
    for (size_t j = 0; j < q.probs.size(); ++j) {
      const GemmProb& p = probs[q.probs[j]];
      for (int n = 0; n < p.N; ++n)
        row_out.push_back(RowOut{reinterpret_cast<int64_t>(p.C), n * p.csC, p.bsC, static_cast<int32_t>(j), n});
    }
    it.nin = static_cast<int>(row_in.size()) - it.in0;
    it.nout = q.nout;
    it.nprob = static_cast<int>(q.probs.size());
    it.M = p0.M;
    it.aspace = (g0.flags >> 8) & 15;
    it.bspace = (g0.flags >> 12) & 15;
    it.cspace = p0.cspace;
    it.conjA = (g0.flags & kSegConjA) ? 1 : 0;
    it.beta = p0.beta;
    row_lds = std::max(row_lds, (it.nin + 3) / 4 * 4 * ((it.nout + 15) / 16 * 16));
    first[qi] = it;
  }
  // passes of one row group next to each other at equal rows: they read the
  // same operand (from one XCD's L2 the second time)
  auto group_of = [&](size_t qi) {
    const int pi = passes[qi].probs[0];
    return group[pi] >= 0 ? group[pi] : -1 - int64_t(pi);
  };
  std::vector<std::pair<int64_t, int>> order(passes.size());
  for (size_t qi = 0; qi < passes.size(); ++qi) order[qi] = {group_of(qi), static_cast<int>(qi)};
  std::sort(order.begin(), order.end());
  for (size_t i0 = 0, i1; i0 < order.size(); i0 = i1) {
    int64_t most = 0;
    for (i1 = i0; i1 < order.size() && order[i1].first == order[i0].first; ++i1) {
      const GemmProb& p = probs[passes[order[i1].second].probs[0]];
      most = std::max(most, int64_t(p.M) * p.batch);
    }
    for (int64_t r0 = 0; r0 < most; r0 += per)
      for (size_t i = i0; i < i1; ++i) {
        const int qi = order[i].second;
        const GemmProb& p = probs[passes[qi].probs[0]];
        const int64_t all = int64_t(p.M) * p.batch;
        if (r0 >= all) continue;
        RowItem it = first[qi];
        it.batch0 = static_cast<int32_t>(r0 / p.M);
        it.m0 = static_cast<int32_t>(r0 % p.M);
        it.rows = static_cast<int32_t>(std::min<int64_t>(per, all - r0));
        rows.push_back(it);
      }
  }
}

void GemmPlan::build_tiles_mode(int mode) {
  auto& T = tiles[mode];
  for (int t = 0; t < kNumTileShapes; ++t) T[t].clear();
  std::vector<double> cost[kNumTileShapes];
  std::vector<int> row_probs;
  for (size_t pi = 0; pi < probs.size(); ++pi) {
    const GemmProb& p = probs[pi];
    if (row_eligible(*this, p)) {
      row_probs.push_back(static_cast<int>(pi));
      continue;
    }
    const int shape = tile_shape(p, mode);
    int64_t ktot = 0;
    for (int s = p.seg0; s < p.seg0 + p.nseg; ++s) ktot += (segs[s].K + KCmax - 1) / KCmax * KCmax;
    if (ktot == 0 && p.beta) continue;   // nothing to add
    const int tm = kTileShapes[shape].tm, tn = kTileShapes[shape].tn;
    for (int b = 0; b < p.batch; ++b)
      for (int n0 = 0; n0 < p.N; n0 += tn)
        for (int m0 = 0; m0 < p.M; m0 += tm) {
          T[shape].push_back(GemmTile{static_cast<int32_t>(pi), b, m0, n0});
          cost[shape].push_back(double(ktot) + 8.0);
        }
  }
  // Longest first (LPT) for the persistent round-robin, by cost class
  // (within 25 %), and inside a class the tiles that read the same B
  // columns (problems whose first segment has the same B operand, e.g. the
  // three MPO channels applied to one psi block) next to each other, M-tiles
  // innermost: consecutive tiles run at the same time on one XCD, so B is
  // fetched from HBM once and re-read from that XCD's L2.  A plan with row
  // groups orders by (group, batch, m0) first instead: the tiles that read
  // the same A rows run together (such plans have far more tiles than the
  // grid, so the cost order matters less than the shared fetch).
  const bool grouped = std::any_of(group.begin(), group.end(), [](int64_t g) { return g >= 0; });
  auto bkey = [&](const GemmTile& g) -> uint64_t {
    const GemmProb& p = probs[g.prob];
    if (!p.nseg) return 0;
    const GemmSeg& q = segs[p.seg0];
    return (static_cast<uint64_t>((q.flags >> 12) & 15) << 56) ^ reinterpret_cast<uint64_t>(q.B) ^
           (static_cast<uint64_t>(g.batch) << 40);
  };
  for (int t = 0; t < kNumTileShapes; ++t) {
    std::vector<size_t> ord(T[t].size());
    std::iota(ord.begin(), ord.end(), 0);
    std::vector<int> cls(T[t].size());
    std::vector<uint64_t> bk(T[t].size());
    for (size_t i = 0; i < ord.size(); ++i) {
      cls[i] = static_cast<int>(std::floor(std::log(cost[t][i]) / std::log(1.25)));
      bk[i] = bkey(T[t][i]);
    }
    std::stable_sort(ord.begin(), ord.end(), [&](size_t a, size_t b) {
      if (grouped) {
        const GemmTile &x = T[t][a], &y = T[t][b];
        const int64_t gx = group[x.prob], gy = group[y.prob];
        if (gx != gy) return gx < gy;
        if (x.batch != y.batch) return x.batch < y.batch;
        if (x.m0 != y.m0) return x.m0 < y.m0;
        if (x.prob != y.prob) return x.prob < y.prob;
        return x.n0 < y.n0;
      }
      if (cls[a] != cls[b]) return cls[a] > cls[b];
      if (bk[a] != bk[b]) return bk[a] < bk[b];
      if (T[t][a].n0 != T[t][b].n0) return T[t][a].n0 < T[t][b].n0;
      if (T[t][a].prob != T[t][b].prob) return T[t][a].prob < T[t][b].prob;
      return T[t][a].m0 < T[t][b].m0;
    });
    std::vector<GemmTile> sorted;
    sorted.reserve(ord.size());
    for (auto o : ord) sorted.push_back(T[t][o]);
    T[t].swap(sorted);
  }
  if (!rows_built) build_rows(row_probs);   // the same for every policy
  built[mode] = true;
  tiles_uploaded[mode] = false;
}

void GemmPlan::upload(hipStream_t s) {
  if (!uploaded) {
    // a new set of problems: nothing on the device holds any more (freeing
    // waits for launches that still read it)
    d_bufs.clear();
    rows_uploaded = direct_uploaded = false;
    for (int m = 0; m < kTileModes; ++m) tiles_uploaded[m] = false;
  }
  // (each byte of the staging copy is touched once: on the host a plan of many
  // small blocks costs mostly the first use of its pages)
  struct Placed {
    const void* from;
    size_t at, bytes;
    std::function<void(const char*)> set;
  };
  size_t total = 0;
  std::vector<Placed> placed;
  auto put = [&](const auto& v, auto& d) {
    d = nullptr;
    if (v.empty()) return;
    const size_t at = (total + 15) / 16 * 16;
    total = at + v.size() * sizeof(v[0]);
    placed.push_back(Placed{v.data(), at, v.size() * sizeof(v[0]), [&d, at](const char* base) {
                              d = reinterpret_cast<std::remove_reference_t<decltype(d)>>(base + at);
                            }});
  };
  if (!uploaded) {
    put(probs, d_probs);
    put(segs, d_segs);
  }
  if (!direct_uploaded) put(direct, d_direct);
  if (!rows_uploaded) {
    put(row_in, d_row_in);
    put(row_out, d_row_out);
    put(row_blk, d_row_blk);
    put(rows, d_rows);
  }
  for (int m = 0; m < kTileModes; ++m)
    if (built[m] && !tiles_uploaded[m])
      for (int t = 0; t < kNumTileShapes; ++t) put(tiles[m][t], d_tiles[m][t]);
  if (total) {
    DevBuf<char> buf(total);
    const std::unique_ptr<char[]> host(new char[total]);
    for (const Placed& p : placed) {
      std::memcpy(host.get() + p.at, p.from, p.bytes);
      p.set(buf.get());
    }
    buf.upload(host.get(), total, s);
    d_bufs.push_back(std::move(buf));
  }
  uploaded = direct_uploaded = rows_uploaded = true;
  for (int m = 0; m < kTileModes; ++m) tiles_uploaded[m] = built[m];
}

int GemmPlan::route(int precision) const {
  const LaunchCfg& c = cfg[precision];
  if (c.direct && !direct.empty()) return 4;
  int r = rows.empty() ? 0 : 2;
  for (const auto& t : tiles[c.tile_mode])
    if (!t.empty()) r |= 1;
  return r;
}

bool GemmPlan::on_device(int precision) const {
  const LaunchCfg& c = cfg[precision];
  if (c.direct && !direct.empty()) return uploaded && direct_uploaded;
  return uploaded && rows_uploaded && built[c.tile_mode] && tiles_uploaded[c.tile_mode];
}

void GemmPlan::clear() {
  probs.clear();
  segs.clear();
  group.clear();
  row_in.clear();
  row_out.clear();
  row_blk.clear();
  rows.clear();
  rows_built = rows_uploaded = false;
  direct.clear();
  direct_uploaded = false;
  for (int m = 0; m < kTileModes; ++m) {
    for (auto& t : tiles[m]) t.clear();
    built[m] = false;
    tiles_uploaded[m] = false;
  }
  flops = 0.0;
  uploaded = false;
  tuned[0] = tuned[1] = false;
}

uint64_t GemmPlan::signature(int precision) const {
  auto lg = [](int64_t v) { int b = 0; while ((int64_t(1) << b) < v) ++b; return b; };
  std::map<std::array<int, 4>, double> hist;
  double tot = 0.0;
  for (const GemmProb& p : probs) {
    int64_t k = 0;
    for (int s = p.seg0; s < p.seg0 + p.nseg; ++s) k += segs[s].K;
    const double f = double(p.M) * double(p.N) * double(k) * double(p.batch);
    hist[{lg(p.M), lg(p.N), lg(std::max<int64_t>(k, 1)), p.batch > 1 ? 1 : 0}] += f;
    tot += f;
  }
  uint64_t h = 1469598103934665603ull ^ static_cast<uint64_t>(precision);
  auto mix = [&h](uint64_t v) { h ^= v; h *= 1099511628211ull; };
  for (auto& kv : hist) {
    const int q = tot > 0 ? static_cast<int>(std::lround(20.0 * kv.second / tot)) : 0;
    if (!q) continue;
    for (int v : kv.first) mix(static_cast<uint64_t>(v));
    mix(static_cast<uint64_t>(q));
  }
  return h;
}

namespace {

std::mutex g_tune_mu;
std::unordered_map<uint64_t, LaunchCfg> g_tune_cache;

void apply_choice(GemmPlan& plan, int precision, const LaunchCfg& c, hipStream_t s) {
  plan.cfg[precision] = c;
  if (!plan.built[c.tile_mode]) plan.build_tiles_mode(c.tile_mode);
  plan.upload(s);
}

}  // namespace

bool autotune(GemmPlan& plan, int precision, hipStream_t s, const GemmBases* bases, double min_flops) {
  if (plan.tuned[precision]) return true;
  const char* e = std::getenv("CAM_AUTOTUNE");
  if ((e && *e == '0') || plan.flops < min_flops) return false;
  for (const GemmProb& p : plan.probs)
    CAM_REQUIRE(!p.beta, "autotune: a plan that accumulates into its output cannot be re-run");
  // (a plan with few outputs and a long K can be small and be tuned; what a
  // plan without the choice found does not decide it)
  const bool small = !plan.direct.empty();
  const uint64_t key = plan.signature(precision) ^ (small ? 0x9e3779b97f4a7c15ull : 0);
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tune_cache.find(key);
    if (it != g_tune_cache.end()) {
      apply_choice(plan, precision, it->second, s);
      plan.tuned[precision] = true;
      return true;
    }
  }
  hipEvent_t ev0, ev1;
  HIP_CHECK(hipEventCreate(&ev0));
  HIP_CHECK(hipEventCreate(&ev1));
  auto time_it = [&](const LaunchCfg& c) {
    apply_choice(plan, precision, c, s);
    launch_grouped_gemm(plan, precision, s, bases);   // warm
    float best = 1e30f;
    for (int r = 0; r < 2; ++r) {
      HIP_CHECK(hipEventRecord(ev0, s));
      launch_grouped_gemm(plan, precision, s, bases);
      HIP_CHECK(hipEventRecord(ev1, s));
      HIP_CHECK(hipEventSynchronize(ev1));
      float ms = 0.f;
      HIP_CHECK(hipEventElapsedTime(&ms, ev0, ev1));
      best = std::min(best, ms);
    }
    return best;
  };
  LaunchCfg cur = plan.cfg[precision];
  // a small plan: the one-launch kernel against the best tiles
  float tdirect = 1e30f;
  if (small) {
    cur.direct = true;
    tdirect = time_it(cur);
    cur.direct = false;
  }
  // coordinate descent: product form, then tile policy, then K chunk, then
  // grid size
  float tcur = time_it(cur);
  auto try_axis = [&](int LaunchCfg::*field, std::initializer_list<int> vals) {
    for (int v : vals) {
      if (cur.*field == v) continue;
      LaunchCfg c = cur;
      c.*field = v;
      const float t = time_it(c);
      if (t < tcur) { tcur = t; cur = c; }
    }
  };
  try_axis(&LaunchCfg::algo, {kAlgo3M, kAlgo4M});
  try_axis(&LaunchCfg::tile_mode, {1, 0, 2, 3});
  try_axis(&LaunchCfg::kc, {16, 8});
  try_axis(&LaunchCfg::wg_per_cu, {4, 2, 8});
  if (tdirect < tcur) cur.direct = true;
  apply_choice(plan, precision, cur, s);
  // leave the output of the chosen configuration (every candidate computes
  // the same values; this keeps the last write consistent with the choice)
  launch_grouped_gemm(plan, precision, s, bases);
  HIP_CHECK(hipEventDestroy(ev0));
  HIP_CHECK(hipEventDestroy(ev1));
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tune_cache[key] = cur;
  }
  plan.tuned[precision] = true;
  return true;
}

void launch_grouped_gemm(GemmPlan& plan, int precision, hipStream_t s, const GemmBases* bases,
                         int grid_limit) {
  const LaunchCfg& c = plan.cfg[precision];
  if (c.direct && !plan.direct.empty()) {
    if (!plan.on_device(precision)) plan.upload(s);
    GemmBases b{};
    if (bases) b = *bases;
    if (precision == 0) launch_direct<double>(plan, s, grid_limit, b);
    else launch_direct<float>(plan, s, grid_limit, b);
    return;
  }
  if (!plan.built[c.tile_mode]) plan.build_tiles_mode(c.tile_mode);
  if (!plan.on_device(precision)) plan.upload(s);
  GemmBases b{};
  if (bases) b = *bases;
  if (precision == 0) {
    launch_shape<double, 64, 64>(plan, c, 0, s, grid_limit, b);
    launch_shape<double, 32, 64>(plan, c, 1, s, grid_limit, b);
    launch_shape<double, 64, 32>(plan, c, 2, s, grid_limit, b);
    launch_shape<double, 128, 64>(plan, c, 3, s, grid_limit, b);
    launch_shape<double, 64, 128>(plan, c, 4, s, grid_limit, b);
    launch_shape<double, 128, 32>(plan, c, 5, s, grid_limit, b);
    launch_rows<double>(plan, s, grid_limit, b);
  } else {
    launch_shape<float, 64, 64>(plan, c, 0, s, grid_limit, b);
    launch_shape<float, 32, 64>(plan, c, 1, s, grid_limit, b);
    launch_shape<float, 64, 32>(plan, c, 2, s, grid_limit, b);
    launch_shape<float, 128, 64>(plan, c, 3, s, grid_limit, b);
    launch_shape<float, 64, 128>(plan, c, 4, s, grid_limit, b);
    launch_shape<float, 128, 32>(plan, c, 5, s, grid_limit, b);
    launch_rows<float>(plan, s, grid_limit, b);
  }
}

}  // namespace cam
