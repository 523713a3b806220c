// Device helpers shared by the transform kernels: how a line of 2^M elements
// is split into register rounds and where a round's elements and roots lie,
// and the conversions between the register format's residues and integers.
#pragma once
#include "kernels.h"

namespace annie {

// Word offset of the slot at list position pos (0 without a slot list).
__device__ __forceinline__ size_t slot_offset(const uint32_t* ids, size_t stride, uint32_t pos) {
  return ids ? size_t(ids[pos]) * stride : size_t(0);
}

// Roots of one register round (levels [d0, d0 + RR)) for each of the
// thread's 2^LR >> RR groups: the 2^RR - 1 roots of a group in heap order,
// level e of the round at entries 2^e - 1 .. 2^{e+1} - 2.  A round's roots are
// loaded one round ahead of their use, so their latency overlaps the previous
// round's butterflies and LDS exchange.
template <int LR, int RR>
struct RoundTw {
  static constexpr int G = (1 << LR) >> RR, W = (1 << RR) - 1;
  uint32_t w[G * W];
};

// Position inside the line of element jj of sub-group s held by thread slot tg
// in a round covering levels [d0, d0 + RR) of a line of 2^m elements.  A thread
// holds 2^LR elements (LR levels per full round): 2^LR >> RR groups of 2^RR
// elements, group g = tg + s * (2^m / 2^LR)
// (consecutive threads take consecutive groups, so round 0 reads and the
// last inverse round writes coalesced); group g spans
// node*2^{m-d0} + off + j*2^{m-d0-RR}.
template <int LR, int RR>
__device__ __forceinline__ uint32_t group_base(int m, int d0, uint32_t tg, int s, uint32_t& node) {
  const uint32_t g = tg + (uint32_t(s) << (m - LR));
  const int lst = m - d0 - RR;
  node = g >> lst;
  const uint32_t off = g & ((1u << lst) - 1u);
  return (node << (m - d0)) + off;
}

// Move the thread's 2^LR elements of round (d0, RR) between registers and a store.
template <int LR, int RR, class Ld>
__device__ __forceinline__ void round_load(uint32_t (&x)[1 << LR], int m, int d0, uint32_t tg, Ld&& ld) {
#pragma unroll
  for (int s = 0; s < ((1 << LR) >> RR); ++s) {
    uint32_t node;
    const uint32_t b = group_base<LR, RR>(m, d0, tg, s, node);
    const int lst = m - d0 - RR;
#pragma unroll
    for (int j = 0; j < (1 << RR); ++j) x[s * (1 << RR) + j] = ld(b + (uint32_t(j) << lst));
  }
}

template <int LR, int RR, class St>
__device__ __forceinline__ void round_store(const uint32_t (&x)[1 << LR], int m, int d0, uint32_t tg, St&& st) {
#pragma unroll
  for (int s = 0; s < ((1 << LR) >> RR); ++s) {
    uint32_t node;
    const uint32_t b = group_base<LR, RR>(m, d0, tg, s, node);
    const int lst = m - d0 - RR;
#pragma unroll
    for (int j = 0; j < (1 << RR); ++j) st(b + (uint32_t(j) << lst), x[s * (1 << RR) + j]);
  }
}

// Word i of a root table, line or operand (i < 2^30: tables and planes are at
// most 2^23 words), addressed by a 32-bit byte offset from the base, so the
// compiler can use the scalar-base + 32-bit vector-offset form instead of a
// 64-bit address per thread (fewer VGPRs: a row pass of 2^9 drops from 85 to
// 64 and runs eight waves per SIMD instead of five).
__device__ __forceinline__ uint32_t ld_w(const uint32_t* base, uint32_t i) {
  return *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(base) + (i << 2));
}

__device__ __forceinline__ void st_w(uint32_t* base, uint32_t i, uint32_t v) {
  *reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(base) + (i << 2)) = v;
}

// Load the roots of round (d0, RR) of the line whose root node is lineRoot
// (heap index at level 0 of this pass).
template <int LR, int RR>
__device__ __forceinline__ void round_tw(RoundTw<LR, RR>& T, int m, int d0, uint32_t tg, uint32_t lineRoot,
                                         const TwDev* tw) {
#pragma unroll
  for (int s = 0; s < RoundTw<LR, RR>::G; ++s) {
    uint32_t node;
    group_base<LR, RR>(m, d0, tg, s, node);
    const uint32_t H0 = (lineRoot << d0) + node;
#pragma unroll
    for (int e = 0; e < RR; ++e)
#pragma unroll
      for (int blk = 0; blk < (1 << e); ++blk) T.w[s * RoundTw<LR, RR>::W + (1 << e) - 1 + blk] = ld_w(tw, (H0 << e) + blk);
  }
}

// Round schedule of a line of 2^M elements: rounds of LR levels (2^LR
// elements per thread), the last one taking the remainder.  Everything is
// fixed at compile time, so each round reads and writes a statically known
// memory (global or LDS).
template <int M, int LR>
struct Sched {
  static constexpr int NR = (M + LR - 1) / LR;
  template <int I>
  static constexpr int rr() { return (M - LR * I) < LR ? (M - LR * I) : LR; }
};

template <int M, int LR, int I>
using SchedTw = RoundTw<LR, Sched<M, LR>::template rr<I>()>;

__device__ __forceinline__ uint32_t lpad(uint32_t i) { return i + (i >> 5); }

// Column group of a column-pass workgroup.  Workgroups are dispatched to the
// eight XCDs round-robin (XCD = workgroup id mod 8), and each XCD has its own
// L2; a group of C columns covers 4C bytes of a 128-byte line, so the G = 32 / C
// workgroups x, x + 8, ..., x + 8 (G - 1) (same XCD, dispatched together) take
// the G parts of one line: within each run of 8G ids, x -> G (x mod 8) +
// (x div 8 mod G), a permutation of the run.
__device__ __forceinline__ uint32_t col_group(uint32_t C) {
  const uint32_t x = blockIdx.x;
  const uint32_t G = 32u / C;
  if (G < 2u || gridDim.x % (8u * G) != 0u) return x;
  return (x & ~(8u * G - 1u)) | ((x & 7u) * G) | ((x >> 3) & (G - 1u));
}

// Signed value of one coefficient from its K residues (each in [0, p_k)):
// mixed-radix digits u_{K-1} = r_{K-1}, u_j = (...((r_j - u_{K-1}) / p_{K-1}) - ...) / p_{j+1}
// mod p_j, with u_0 taken in (-p_0/2, p_0/2], then Horner over the primes,
// the accumulator growing by one limb per step (after step j it holds a
// signed value below 2^{32 (j+1) - 1} in magnitude).  Result sign-extended
// to L >= K limbs.
template <int K, int L>
__device__ __forceinline__ void garner(const uint32_t (&r)[K], uint32_t (&acc)[L]) {
  uint32_t u[K];
#pragma unroll
  for (int j = K - 1; j >= 0; --j) {
    uint32_t v = r[j];
#pragma unroll
    for (int i = K - 1; i > j; --i) v = submul_c(v, u[i], PLIT.ginv[i][j], PLIT.ginvq[i][j], PRIMES[j]);
    u[j] = v;
  }
  const int32_t i0 = (u[0] > (PRIMES[0] >> 1)) ? int32_t(u[0] - PRIMES[0]) : int32_t(u[0]);
  acc[0] = uint32_t(i0);
  uint32_t sg = uint32_t(i0 >> 31);
#pragma unroll
  for (int j = 1; j < K; ++j) {
    const uint32_t pj = PRIMES[j];
    uint64_t c = u[j];
#pragma unroll
    for (int i = 0; i < j; ++i) {
      const uint64_t t = uint64_t(acc[i]) * pj + c;
      acc[i] = uint32_t(t);
      c = t >> 32;
    }
    acc[j] = sg * pj + uint32_t(c);
    sg = uint32_t(int32_t(acc[j]) >> 31);
  }
#pragma unroll
  for (int i = K; i < L; ++i) acc[i] = sg;
}

// Residue of a signed digit (|d| < 2^95) modulo p_k.
__device__ __forceinline__ uint32_t digit_residue_wide(const uint32_t (&d)[DIGIT_LIMBS], int k) {
  const uint32_t p = PRIMES[k];
  const bool neg = int32_t(d[2]) < 0;
  uint32_t a0 = d[0], a1 = d[1], a2 = d[2];
  if (neg) {  // |d| = ~d + 1
    a0 = ~a0;
    a1 = ~a1;
    a2 = ~a2;
    const uint64_t t0 = uint64_t(a0) + 1;
    a0 = uint32_t(t0);
    const uint64_t t1 = uint64_t(a1) + (t0 >> 32);
    a1 = uint32_t(t1);
    a2 += uint32_t(t1 >> 32);
  }
  uint32_t r = (a0 >= p) ? a0 - p : a0;
  r = addmod(r, mont_c(a1, PLIT.c32[k], PLIT.c32q[k], p), p);
  r = addmod(r, mont_c(a2, PLIT.c64[k], PLIT.c64q[k], p), p);
  return neg ? submod(0u, r, p) : r;
}

}  // namespace annie
