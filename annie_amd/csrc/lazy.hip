// gfx950 kernels of the short-prime path (lazy.h): transforms over 28-bit
// primes on signed, lazily reduced residues, and CRT + carry passes between
// residues and digit registers.
//
// Arithmetic.  A residue is any signed 32-bit word congruent to it.  The
// Montgomery product by a constant |w| <= p / 2, hi(b w) - hi(lo(b w p^-1) p), is
// at most p / 2 + |b| p / 2^33 <= 0.75 p in magnitude for every word b, so the
// forward butterfly (a, b) -> (a + t, a - t) takes six instructions and no
// correction while its values fit: they grow by 0.5-0.75 p per level.  Measured
// on a register-resident chain (2,048 workgroups of 256): 4.9 issue slots per
// butterfly against 9.4 with the corrections that primes above 2^31 need.
//
// Three sets of primes (lazy.h), W: 0 below 2^28.2 (a word holds +-6.9 p: eight
// levels between reductions), 1 below 2^29.3 (2^21, +-3.2 p) and 2 below 2^29.9
// (2^22, +-2.1 p), as few primes with roots of order 2^{LN + 1} are smaller at
// the longest lengths.  W = 0 reduces by a quotient (lz_red), a whole round at a
// time; W > 0 takes one p off by the sign (lz_cond), where a sum would not fit.
// The bounds are tracked at compile time in units of p / 256 (lz_walk,
// lz_round_inv).
#include "lazy.h"
#include "rounds.h"

namespace annie {

constexpr int lz_lim(int W) { return W == 0 ? 1766 : W == 1 ? 828 : 545; }   // floor(256 2^31 / p)
constexpr int lz_gain(int W) { return W == 0 ? 37 : W == 1 ? 80 : 121; }     // 1024 p / 2^33
constexpr int LZ_RED = 264;                                                   // lz_red: [0, 1.03 p)
constexpr int lz_in(int W) { return W == 0 ? 384 : 262; }                     // a digit's residue as loaded
constexpr int lz_out(int W) { return W == 0 ? 410 : W == 1 ? 270 : 256; }     // what an inverse round starts from
constexpr int lz_less(int s) { return s > 512 ? s - 256 : 256; }              // lz_cond of a value within s

// Forward bounds: lz_level is the bound after one level from bound s (the
// sums' first operand is reduced when `c`), lz_level_cond whether it has to be;
// lz_walk the bound at the start of round `upto` of a line of 2^M elements (or
// at its end), and lz_fwd_red whether round I reduces its elements first.
constexpr bool lz_level_cond(int W, int s) { return W > 0 && s + 129 + s * lz_gain(W) / 1024 > lz_lim(W); }
constexpr int lz_level(int W, int s) { return (lz_level_cond(W, s) ? lz_less(s) : s) + 129 + s * lz_gain(W) / 1024; }
constexpr int lz_levels(int W, int s, int rr) {
  for (int l = 0; l < rr; ++l) s = lz_level(W, s);
  return s;
}
constexpr int lz_walk(int W, int M, int LR, int s, int upto) {
  for (int i = 0, left = M; left > 0; ++i) {
    const int rr = left < LR ? left : LR;
    left -= rr;
    if (W == 0 && lz_levels(W, s, rr) > lz_lim(W)) s = LZ_RED;
    if (i == upto) return s;
    s = lz_levels(W, s, rr);
  }
  return s;
}
constexpr bool lz_fwd_red(int W, int M, int LR, int s, int I) {
  int at = s;
  for (int i = 0, left = M; i < I; ++i) {
    const int rr = left < LR ? left : LR;
    left -= rr;
    if (W == 0 && lz_levels(W, at, rr) > lz_lim(W)) at = LZ_RED;
    at = lz_levels(W, at, rr);
  }
  const int left = M - LR * I;
  return W == 0 && lz_levels(W, at, left < LR ? left : LR) > lz_lim(W);
}
constexpr bool lz_safe(int W, int M, int LR, int s) { return lz_walk(W, M, LR, s, -1) <= lz_lim(W); }
static_assert(lz_safe(0, 13, 3, lz_in(0)) && lz_safe(0, 13, 4, lz_in(0)) && lz_safe(0, 10, 5, lz_in(0)) &&
                  lz_safe(0, 10, 4, lz_lim(0)) && lz_safe(0, 10, 3, lz_lim(0)) && lz_safe(1, 10, 5, lz_in(1)) &&
                  lz_safe(1, 11, 4, lz_lim(1)) && lz_safe(2, 10, 5, lz_in(2)) && lz_safe(2, 12, 4, lz_lim(2)),
              "a forward line leaves its words");

struct LzP {
  uint32_t p, q, bar;
};

// round_load / round_store (rounds.h) with the position in two parts: the
// group's first element b, a thread's, and c = j 2^lst, a constant. They share
// no bit, so an accessor that permutes or pads bit by bit forms one address per
// group and leaves c to the instruction's offset or the uniform base. Before,
// each element's address was formed by itself: a squaring mod 2^21 coefficients
// took 88.3 us and takes 86.2, one of 2^12 22.0 and 21.6, 130 registers of 2^12
// 58.3 and 57.1.
template <int LR, int RR, class Ld>
__device__ __forceinline__ void lz_load(uint32_t (&x)[1 << LR], int m, int d0, uint32_t tg, Ld&& ld) {
#pragma unroll
  for (int s = 0; s < ((1 << LR) >> RR); ++s) {
    uint32_t node;
    const uint32_t b = group_base<LR, RR>(m, d0, tg, s, node);
#pragma unroll
    for (int j = 0; j < (1 << RR); ++j) x[s * (1 << RR) + j] = ld(b, uint32_t(j) << (m - d0 - RR));
  }
}
template <int LR, int RR, class St>
__device__ __forceinline__ void lz_store(const uint32_t (&x)[1 << LR], int m, int d0, uint32_t tg, St&& st) {
#pragma unroll
  for (int s = 0; s < ((1 << LR) >> RR); ++s) {
    uint32_t node;
    const uint32_t b = group_base<LR, RR>(m, d0, tg, s, node);
#pragma unroll
    for (int j = 0; j < (1 << RR); ++j) st(b, uint32_t(j) << (m - d0 - RR), x[s * (1 << RR) + j]);
  }
}

__device__ __forceinline__ int32_t lz_mulc(int32_t b, int32_t w, uint32_t wq, uint32_t p) {
  return __mulhi(b, w) - __mulhi(int32_t(uint32_t(b) * wq), int32_t(p));
}
__device__ __forceinline__ int32_t lz_mul(int32_t a, int32_t b, const LzP& P) {
  const uint32_t lo = uint32_t(a) * uint32_t(b);
  return __mulhi(a, b) - __mulhi(int32_t(lo * P.q), int32_t(P.p));
}
// x mod p in [0, 1.03 p): bar = floor(2^58 / p).
__device__ __forceinline__ int32_t lz_red(int32_t x, const LzP& P) {
  return x - int32_t(uint32_t(__mulhi(x, int32_t(P.bar)) >> 26) * P.p);
}

// Inverse bounds: before a sum and difference leave their words, one or both
// operands are reduced by lz_cond, once or twice, or by lz_red (codes 1, 2, 3;
// 0: not at all), whichever takes the fewest issue slots (2.3 and 3.6 each);
// after the last level of a round all elements are brought back within lz_out.
// Compared with one lz_cond for every sum: 55 instead of 74 slots per 32
// butterflies for W = 1.
template <int RR, int W>
struct LzPlan {
  uint8_t op[RR][1 << RR], end[1 << RR];
};
constexpr int lz_reduced(int W, int s, int op) {
  return op == 0 ? s : op == 3 ? (s < LZ_RED ? s : LZ_RED) : op == 1 ? lz_less(s) : lz_less(lz_less(s));
}
constexpr int lz_cost(int op) { return op == 0 ? 0 : op == 1 ? 23 : op == 2 ? 46 : 36; }
template <int RR, int W>
constexpr LzPlan<RR, W> lz_inv_plan() {
  LzPlan<RR, W> pl{};
  int bd[1 << RR] = {};
  for (int j = 0; j < (1 << RR); ++j) bd[j] = lz_out(W);
  const int first = W == 0 ? 3 : 1;  // W = 0: lz_red only
  for (int e = RR - 1; e >= 0; --e) {
    const int half = (1 << RR) >> (e + 1);
    for (int j = 0; j < (1 << RR); ++j) {
      if (j & half) continue;
      const int i = j + half;
      if (bd[j] + bd[i] > lz_lim(W)) {
        int best = 1 << 30;
        for (int a = 0; a < 4; ++a)
          for (int b = 0; b < 4; ++b) {
            if ((a > 0 && a < first) || (b > 0 && b < first)) continue;
            const int s = lz_reduced(W, bd[j], a) + lz_reduced(W, bd[i], b), cost = (lz_cost(a) + lz_cost(b)) * 4096 + s;
            if (s <= lz_lim(W) && cost < best) {
              best = cost;
              pl.op[e][j] = uint8_t(a);
              pl.op[e][i] = uint8_t(b);
            }
          }
        bd[j] = lz_reduced(W, bd[j], pl.op[e][j]);
        bd[i] = lz_reduced(W, bd[i], pl.op[e][i]);
      }
      const int s = bd[j] + bd[i];
      bd[j] = s;
      bd[i] = 130 + s * lz_gain(W) / 1024;
    }
  }
  for (int j = 0; j < (1 << RR); ++j)
    if (bd[j] > lz_out(W))
      for (int a : {1, 3, 2})
        if (a >= first && lz_reduced(W, bd[j], a) <= lz_out(W) && pl.end[j] == 0) pl.end[j] = uint8_t(a);
  return pl;
}

// x - p or x + p by the sign: within max(p, |x| - p).
__device__ __forceinline__ uint32_t lz_cond(uint32_t x, const LzP& P) {
  return x + (int32_t(x) < 0 ? P.p : 0u - P.p);
}

// The levels of one round from elements within s.
template <int LR, int RR, int W>
__device__ __forceinline__ void lz_round_fwd(uint32_t (&x)[1 << LR], const RoundTw<LR, RR>& T, const LzP& P, int s0) {
#pragma unroll
  for (int s = 0; s < RoundTw<LR, RR>::G; ++s) {
    int bound = s0;
#pragma unroll
    for (int e = 0; e < RR; ++e) {
      const bool cond = lz_level_cond(W, bound);
      bound = lz_level(W, bound);
      const int half = (1 << RR) >> (e + 1);
#pragma unroll
      for (int blk = 0; blk < (1 << e); ++blk) {
        const uint32_t r = T.w[s * RoundTw<LR, RR>::W + (1 << e) - 1 + blk], rq = r * P.q;
#pragma unroll
        for (int jj = 0; jj < half; ++jj) {
          uint32_t& a = x[s * (1 << RR) + blk * 2 * half + jj];
          uint32_t& b = x[s * (1 << RR) + blk * 2 * half + jj + half];
          const uint32_t t = uint32_t(lz_mulc(int32_t(b), int32_t(r), rq, P.p));
          if (cond) a = lz_cond(a, P);
          b = a - t;
          a = a + t;
        }
      }
    }
  }
}

// Inverse levels of a round; the elements start within lz_out, and end there
// too unless LAST (then within their words).
__device__ __forceinline__ void lz_apply(uint32_t& x, int op, const LzP& P) {
  if (op == 3) x = uint32_t(lz_red(int32_t(x), P));
  if (op == 1 || op == 2) x = lz_cond(x, P);
  if (op == 2) x = lz_cond(x, P);
}

template <int LR, int RR, int W, bool LAST>
__device__ __forceinline__ void lz_round_inv(uint32_t (&x)[1 << LR], const RoundTw<LR, RR>& T, const LzP& P) {
  constexpr LzPlan<RR, W> PL = lz_inv_plan<RR, W>();
#pragma unroll
  for (int s = 0; s < RoundTw<LR, RR>::G; ++s) {
    uint32_t* v = &x[s * (1 << RR)];
#pragma unroll
    for (int e = RR - 1; e >= 0; --e) {
      const int half = (1 << RR) >> (e + 1);
#pragma unroll
      for (int blk = 0; blk < (1 << e); ++blk) {
        const uint32_t r = T.w[s * RoundTw<LR, RR>::W + (1 << e) - 1 + blk], rq = r * P.q;
#pragma unroll
        for (int jj = 0; jj < half; ++jj) {
          const int j = blk * 2 * half + jj, i = j + half;
          lz_apply(v[j], PL.op[e][j], P);
          lz_apply(v[i], PL.op[e][i], P);
          const uint32_t d = v[j] - v[i];
          v[j] = v[j] + v[i];
          v[i] = uint32_t(lz_mulc(int32_t(d), int32_t(r), rq, P.p));
        }
      }
    }
    if constexpr (!LAST) {
#pragma unroll
      for (int j = 0; j < (1 << RR); ++j) lz_apply(v[j], PL.end[j], P);
    }
  }
}

// The roots of all rounds of a line, loaded before its first element arrives
// (lines of eight elements per thread: at most 32 words each way).
template <int M, int LR, int I>
struct LzRoots {
  SchedTw<M, LR, I> t;
  LzRoots<M, LR, I + 1> next;
  __device__ __forceinline__ void load(uint32_t tg, uint32_t lineRoot, const uint32_t* tw) {
    round_tw(t, M, LR * I, tg, lineRoot, tw);
    if constexpr (I + 1 < Sched<M, LR>::NR) next.load(tg, lineRoot, tw);
  }
  template <int J>
  __device__ __forceinline__ const SchedTw<M, LR, J>& get() const {
    if constexpr (J == I) return t;
    else return next.template get<J>();
  }
};
template <int M, int LR>
struct LzRoots<M, LR, (M + LR - 1) / LR> {};

// Forward rounds I.. .  ROOTS: 0 each round loads its own roots (from LDS), 1
// one round ahead (`cur` holds round I's), 2 all loaded (`all`).
template <int W, int M, int LR, int I, int ROOTS, int S0, class GLd, class LLd, class LSt, class Hook>
__device__ __forceinline__ void lz_fwd(uint32_t (&x)[1 << LR], uint32_t tg, uint32_t lineRoot, const uint32_t* tw,
                                       const LzP& P, GLd& gld, LLd& lld, LSt& lst, const SchedTw<M, LR, I>& cur,
                                       const LzRoots<M, LR, 0>& all, Hook&& at_last) {
  constexpr int RR = Sched<M, LR>::template rr<I>();
  constexpr bool END = I + 1 == Sched<M, LR>::NR;
  SchedTw<M, LR, I> own;
  if constexpr (ROOTS == 0) round_tw(own, M, LR * I, tg, lineRoot, tw);
  SchedTw<M, LR, END ? I : I + 1> nxt;
  if constexpr (ROOTS == 1 && !END) round_tw(nxt, M, LR * (I + 1), tg, lineRoot, tw);
  if constexpr (END) at_last();
  if constexpr (I > 0) lz_load<LR, RR>(x, M, LR * I, tg, lld);
  if constexpr (lz_fwd_red(W, M, LR, S0, I)) {
#pragma unroll
    for (int i = 0; i < (1 << LR); ++i) x[i] = uint32_t(lz_red(int32_t(x[i]), P));
  }
  constexpr int S = lz_walk(W, M, LR, S0, I);
  if constexpr (ROOTS == 0) lz_round_fwd<LR, RR, W>(x, own, P, S);
  else if constexpr (ROOTS == 1) lz_round_fwd<LR, RR, W>(x, cur, P, S);
  else lz_round_fwd<LR, RR, W>(x, all.template get<I>(), P, S);
  if constexpr (!END) {
    lz_store<LR, RR>(x, M, LR * I, tg, lst);
    __syncthreads();
    lz_fwd<W, M, LR, I + 1, ROOTS, S0>(x, tg, lineRoot, tw, P, gld, lld, lst, nxt, all, at_last);
  }
}

// Inverse rounds I down to 0, from the elements of round NR - 1 in x.  FINAL:
// the values go to a carry, which takes any word.
template <int W, int M, int LR, int I, int ROOTS, bool FINAL, class GSt, class LLd, class LSt>
__device__ __forceinline__ void lz_inv(uint32_t (&x)[1 << LR], uint32_t tg, uint32_t lineRoot, const uint32_t* tw,
                                       const LzP& P, GSt& gst, LLd& lld, LSt& lst, const SchedTw<M, LR, I>& cur,
                                       const LzRoots<M, LR, 0>& all) {
  constexpr int RR = Sched<M, LR>::template rr<I>();
  SchedTw<M, LR, I> own;
  if constexpr (ROOTS == 0) round_tw(own, M, LR * I, tg, lineRoot, tw);
  SchedTw<M, LR, I == 0 ? 0 : I - 1> nxt;
  if constexpr (ROOTS == 1 && I > 0) round_tw(nxt, M, LR * (I - 1), tg, lineRoot, tw);
  if constexpr (I + 1 < Sched<M, LR>::NR) lz_load<LR, RR>(x, M, LR * I, tg, lld);
  constexpr bool LAST = I == 0 && FINAL;
  if constexpr (ROOTS == 0) lz_round_inv<LR, RR, W, LAST>(x, own, P);
  else if constexpr (ROOTS == 1) lz_round_inv<LR, RR, W, LAST>(x, cur, P);
  else lz_round_inv<LR, RR, W, LAST>(x, all.template get<I>(), P);
  if constexpr (I > 0) {
    lz_store<LR, RR>(x, M, LR * I, tg, lst);
    __syncthreads();
    lz_inv<W, M, LR, I - 1, ROOTS, FINAL>(x, tg, lineRoot, tw, P, gst, lld, lst, nxt, all);
  } else {
    lz_store<LR, RR>(x, M, 0, tg, gst);
  }
}

// Residue of a digit (low limbs d, for DL = 3 the top limb h) times b =
// 2^{-32 (DL - 1)}: one Montgomery reduction per limb below the top one.  A digit
// has at most 59 (DL = 2) or 76 bits, so the result is within 1.5 p.
template <int DL>
__device__ __forceinline__ int32_t lz_residue(const uint2 d, uint32_t h, const LzP& P) {
  const uint32_t g = __umulhi(d.x * P.q, P.p);
  if constexpr (DL == 2) return int32_t(d.y - g);
  uint32_t lo;
  const bool br = __builtin_sub_overflow(d.y, g, &lo);
  return int32_t(h - (br ? 1u : 0u) - __umulhi(lo * P.q, P.p));
}
template <int DL>
__device__ __forceinline__ int32_t lz_digit(const uint32_t* x, size_t n, uint32_t i, const LzP& P) {
  return lz_residue<DL>(reinterpret_cast<const uint2*>(x)[i], DL == 3 ? x[2 * n + i] : 0u, P);
}
// Digit u + i with u uniform: a scalar base and a 32-bit offset, for the column
// passes, whose elements lie n2 apart.
template <int DL>
__device__ __forceinline__ int32_t lz_digit_at(const uint32_t* x, size_t n, uint32_t u, uint32_t i, const LzP& P) {
  const char* lo = reinterpret_cast<const char*>(x + 2 * size_t(u));
  return lz_residue<DL>(*reinterpret_cast<const uint2*>(lo + (i << 3)), DL == 3 ? ld_w(x + 2 * n + u, i) : 0u, P);
}

__device__ __forceinline__ uint32_t lz_slot(const uint32_t* ids, uint32_t pos) {
  return ids ? uint32_t(__builtin_amdgcn_readfirstlane(int(ids[pos]))) : 0u;
}

// Kernel arguments that a kernel needs in any case, read together at its
// start: left to itself the compiler loads each one where a branch first
// needs it, and the round trips follow one another (a dozen in the carry, a
// quarter of its time at the shortest lengths).
template <class T>
__device__ __forceinline__ void lz_pin1(const T v) {
  asm volatile("" : : "s"(v));
}
template <class... T>
__device__ __forceinline__ void lz_pin(const T... v) {
  (lz_pin1(v), ...);
}

__device__ __forceinline__ uint32_t lz_multiplier(const LzMult& m, uint32_t pos, uint32_t slot) {
  if (m.a_slot != nullptr) return m.a_slot[pos] & ~SLOT_SNAP;
  if (m.bits_mode == 1) return ((m.bits[pos >> 5] >> (pos & 31u)) & 1u) ? m.slot_base[slot] : 1u;
  return m.a;
}

// A transform of length 2^LN split over 2^SP workgroups (SP = LN - M > 0, the
// single-pass kernels of short launches): workgroup `row` computes the node of
// level SP it owns straight from the digits, position i of it from the 2^SP
// digits i + t 2^M, so that no column pass and no exchange come before it; the
// carry undoes those levels as it loads (LzJoin).  Position i from digits x_t:
// level 0 pairs t and t + 2^{SP - 1} with root r(0, 0), and so on; the sign of
// each level's root is the branch that leads to `row`.  Within 1.5 p + 0.8 p SP.
constexpr int lz_split_in(int SP) { return lz_in(0) + 205 * SP; }
struct LzBranch {
  int32_t r[2];
  uint32_t rq[2];
};
template <int SP>
__device__ __forceinline__ LzBranch lz_branch(const uint32_t* twf, uint32_t row, const LzP& P) {
  LzBranch b{};
#pragma unroll
  for (int l = 0; l < SP; ++l) {
    const uint32_t node = row >> (SP - l);
    const int32_t r = int32_t(twf[(1u << l) + node]);
    b.r[l] = ((row >> (SP - 1 - l)) & 1u) ? -r : r;
    b.rq[l] = uint32_t(b.r[l]) * P.q;
  }
  return b;
}

// Lines of fewer than 64 threads run several to a block, up to 1,024 threads.
constexpr int lz_row_threads(int M, int LR) { return (1 << M >> LR) > 512 || (1 << M >> LR) < 64 ? 1024 : 512; }

// Row pass (the whole transform of lengths up to 2^13, SRC = limbs of a digit;
// the levels from m1 on of longer ones, SRC = 0: planes in place).  What stays
// between transforms (y^, n^, N^, t^) is kept in the order in which the
// threads hold it, element e of thread tg at e T + tg, so that its loads and
// stores are consecutive.
// Grid: (rows / lines, slots, planes), so that the cyclic planes, which go
// forward and back, start before the negacyclic ones, which only go forward
// here; block: lines of 2^M / 2^LR threads.
template <int M, int LR, int MODE, int SRC, int W, int SP>
__global__ void __launch_bounds__(lz_row_threads(M, LR)) k_lz_row(const LzNtt A) {
  extern __shared__ uint32_t lds[];
  constexpr uint32_t S = 1u << M, T = S >> LR;
  constexpr int NR = Sched<M, LR>::NR, RL = Sched<M, LR>::template rr<NR - 1>();
  constexpr int ROOTS = LR <= 3 ? 2 : 1;
  lz_pin(A.slot_ids, A.slot_stride, A.LN, A.KR, A.pl0, A.x, A.wr, A.wq, A.fwdR, A.invR, A.fwdQ, A.invQ, A.nir, A.nq, A.tq, A.neg);
  constexpr int S0 = SRC == 0 ? lz_lim(W) : SP > 0 ? lz_split_in(SP) : lz_in(W);
  static_assert(lz_safe(W, M, LR, S0), "a forward line leaves its words");
  const uint32_t slot = lz_slot(A.slot_ids, blockIdx.y);
  const size_t so = size_t(slot) * A.slot_stride, n = size_t(1) << A.LN;
  const int pl = A.pl0 + int(blockIdx.z);
  const bool cyc = MODE != LZ_MULN && pl < A.KR;
  const int k = cyc ? pl : pl - A.KR;
  const LzP P{A.c.p[k], A.c.q[k], A.c.bar[k]};
  constexpr bool ONE = T >= 64;
  const uint32_t line = ONE ? 0u : threadIdx.x / T, tg = ONE ? threadIdx.x : threadIdx.x % T;
  const uint32_t row = (SRC && SP == 0) ? 0u : (ONE || SRC) ? blockIdx.x : blockIdx.x * uint32_t(A.cols) + line;
  const uint32_t lineRoot = SRC ? (1u << SP) + row : (1u << A.m1) + row;
  const size_t base = so + size_t(k) * n + size_t(row) * S;
  uint32_t* X = lds + line * (S + (S >> 5));
  uint32_t* w = (cyc ? A.wr : A.wq) + base;
  const uint32_t* twf = (cyc ? A.fwdR : A.fwdQ) + size_t(k) * n;
  const uint32_t* twi = (cyc ? A.invR : A.invQ) + size_t(k) * n;

  const LzBranch br = lz_branch<SP>(twf, row, P);
  auto gld = [&](uint32_t b, uint32_t c) {
    if constexpr (SRC == 0) {
      return ld_w(w + c, b);
    } else if constexpr (SP == 0) {
      return uint32_t(lz_digit<SRC>(A.x + so, n, b + c, P));
    } else {
      int32_t d[1 << SP];
#pragma unroll
      for (int t = 0; t < (1 << SP); ++t) d[t] = lz_digit<SRC>(A.x + so, n, b + c + uint32_t(t) * S, P);
#pragma unroll
      for (int l = 0; l < SP; ++l)
#pragma unroll
        for (int t = 0; t < (1 << SP >> (l + 1)); ++t)
          d[t] += lz_mulc(d[t + (1 << SP >> (l + 1))], br.r[l], br.rq[l], P.p);
      return uint32_t(d[0]);
    }
  };
  auto gst = [&](uint32_t b, uint32_t c, uint32_t v) { st_w(w + c, b, v); };
  // lpad(i) = i + i/32, and b and c share no bit: lpad(b + c) = lpad(b) + lpad(c).
  auto lld = [&](uint32_t b, uint32_t c) { return X[lpad(b) + lpad(c)]; };
  auto lst = [&](uint32_t b, uint32_t c, uint32_t v) { X[lpad(b) + lpad(c)] = v; };

  uint32_t x[1 << LR], op[1 << LR], oy[1 << LR];
  LzRoots<M, LR, 0> rf, ri;
  SchedTw<M, LR, 0> t0;
  SchedTw<M, LR, NR - 1> ti;
  const bool back = MODE == LZ_MULN || (cyc && (MODE == LZ_SQR || A.op != LZ_FWD));
  if constexpr (ROOTS == 2) rf.load(tg, lineRoot, twf);
  else round_tw(t0, M, 0, tg, lineRoot, twf);
  lz_load<LR, Sched<M, LR>::template rr<0>()>(x, M, 0, tg, gld);
  if constexpr (MODE == LZ_MULN && SRC != 0) {
    // m' + 2, or m' + R + 2 = m' for a negative m': R N = -2 N mod Q.
    if (tg == 0u && A.neg != nullptr && A.neg[so] == 0u)
      x[0] = uint32_t(lz_red(int32_t(x[0] + 2u * uint32_t(A.c.one[k])), P));
  }
  if constexpr (ROOTS == 2) {
    if (back) ri.load(tg, lineRoot, twi);
  }
  auto prefetch = [&] {
    if constexpr (ROOTS == 1) {
      if (back) round_tw(ti, M, LR * (NR - 1), tg, lineRoot, twi);
    }
    if (back) {
      const uint32_t* o = (MODE == LZ_MULN ? A.nq : A.nir) + base;
#pragma unroll
      for (int e = 0; e < (1 << LR); ++e) op[e] = ld_w(o, uint32_t(e) * T + tg);
    }
    if constexpr (MODE == LZ_MULN) {
      const uint32_t* o = A.tq + base;
#pragma unroll
      for (int e = 0; e < (1 << LR); ++e) oy[e] = ld_w(o, uint32_t(e) * T + tg);
    }
  };
  lz_fwd<W, M, LR, 0, ROOTS, S0>(x, tg, lineRoot, twf, P, gld, lld, lst, t0, rf, prefetch);

  if constexpr (MODE == LZ_GEN) {
    if (A.op == LZ_MULY) {
      const uint32_t* o = (cyc ? A.yr : A.yq) + base;
#pragma unroll
      for (int e = 0; e < (1 << LR); ++e) oy[e] = ld_w(o, uint32_t(e) * T + tg);
    } else {
#pragma unroll
      for (int e = 0; e < (1 << LR); ++e) oy[e] = uint32_t(A.c.one[k]);
    }
  }
  if (back) {
#pragma unroll
    for (int e = 0; e < (1 << LR); ++e) {
      if constexpr (MODE == LZ_MULN) {
        // Within 0.88 p + 0.72 p.
        x[e] = uint32_t(lz_mul(int32_t(x[e]), int32_t(op[e]), P)) - oy[e];
        if constexpr (W > 0) x[e] = lz_cond(x[e], P);
      } else {
        const int32_t y = MODE == LZ_SQR ? int32_t(x[e]) : int32_t(oy[e]);
        x[e] = uint32_t(lz_mul(lz_mul(int32_t(x[e]), y, P), int32_t(op[e]), P));
      }
    }
    // Single-pass values go to the carry; a column pass or LzJoin follows
    // otherwise.
    lz_inv<W, M, LR, NR - 1, ROOTS, SRC != 0 && SP == 0>(x, tg, lineRoot, twi, P, gst, lld, lst, ti, ri);
  } else {
    int32_t c = A.scale[k];
    if (MODE == LZ_SQR || A.op != LZ_FWD) {
      const uint32_t a = lz_multiplier(A.mul, blockIdx.y, slot);
      c = lz_mulc(int32_t(a), A.c.cq[k], uint32_t(A.c.cq[k]) * P.q, P.p);
    }
    const uint32_t cp = uint32_t(c) * P.q;
#pragma unroll
    for (int e = 0; e < (1 << LR); ++e) {
      int32_t v = int32_t(x[e]);
      if constexpr (MODE == LZ_SQR) {
        v = lz_mulc(lz_mul(v, v, P), c, cp, P.p);
      } else {
        if (A.op != LZ_FWD) v = lz_mul(v, int32_t(oy[e]), P);
        if (c != 0) v = lz_mulc(v, c, cp, P.p);
      }
      st_w(w, uint32_t(e) * T + tg, uint32_t(v));
    }
    (void)RL;
  }
}

// Column passes of lengths from 2^14 on: the first M = m1 levels on columns of
// stride n2 = n / 2^M, A.cols (16 for M = 10) consecutive columns per block,
// interleaved and XOR-swizzled in LDS as the passes over the long primes.
// Grid: (column groups, slots, planes); at 2^10 (column groups x planes, slots):
// a unit of two column groups covers whole 128-byte lines and goes to one XCD
// (id mod 8) with all its planes in turn, so that the digits are read from
// memory once for all planes (25 MB instead of 15 times that at 2^21).
// Sixteen columns of 2^10 take 64 KiB of LDS, two workgroups a CU; eight read
// and wrote 1.4 times the data (half-used lines left L2 before the neighbouring
// group came; nine planes of 2^21 back 60 -> 43 us, fifteen forward 77 -> 66).
template <int M, int LR>
struct LzCol {
  static constexpr bool LDS_ROOTS = M < 10;
  static constexpr int C = 16;  // columns per block at M = 10
  static constexpr int THREADS = (M >= 10) ? (C << (M - LR)) : 1024;
  static constexpr int WAVES = 4;
};

struct LzTile {
  int pl;
  uint32_t col0;
};
template <int M>
__device__ __forceinline__ LzTile lz_tile(const LzNtt& A, uint32_t C) {
  if constexpr (M < 10) {
    return {A.pl0 + int(blockIdx.z), col_group(C) * C};
  } else {
    constexpr uint32_t G = 32u / LzCol<M, 5>::C;  // column groups of a 128-byte line
    const uint32_t per = G * uint32_t(A.planes), t = blockIdx.x >> 3;
    const uint32_t unit = (t / per) * 8u + (blockIdx.x & 7u), r = t % per;
    // Divided in vector registers, but uniform: without the return to scalar ones
    // every address derived from them is formed per lane.  With the digits'
    // scalar bases (lz_digit_at) 1,527 instead of 1,756 vector instructions in the
    // forward pass at 2^21: 349.3 -> 346.8 us per squaring, 604.8 -> 598.5 at 2^22.
    return {A.pl0 + __builtin_amdgcn_readfirstlane(int(r / G)),
            uint32_t(__builtin_amdgcn_readfirstlane(int((unit * G + r % G) * C)))};
  }
}

template <int M, int LR, int DL, int W>
__global__ void __launch_bounds__((LzCol<M, LR>::THREADS), (LzCol<M, LR>::WAVES)) k_lz_colf(const LzNtt A) {
  extern __shared__ uint32_t lds[];
  lz_pin(A.slot_ids, A.slot_stride, A.LN, A.KR, A.pl0, A.planes, A.cols, A.x, A.wr, A.wq, A.fwdR, A.invR, A.fwdQ, A.invQ, A.neg);
  constexpr uint32_t S = 1u << M;
  constexpr int NR = Sched<M, LR>::NR, DLV = LR * (NR - 1), RL = Sched<M, LR>::template rr<NR - 1>();
  const uint32_t slot = lz_slot(A.slot_ids, blockIdx.y);
  const size_t so = size_t(slot) * A.slot_stride, n = size_t(1) << A.LN;
  const uint32_t C = (M >= 10) ? uint32_t(LzCol<M, LR>::C) : uint32_t(A.cols);
  const LzTile tile = lz_tile<M>(A, C);
  const int pl = tile.pl;
  const bool cyc = pl < A.KR;
  const int k = cyc ? pl : pl - A.KR;
  const LzP P{A.c.p[k], A.c.q[k], A.c.bar[k]};
  const uint32_t line = threadIdx.x % C, tg = threadIdx.x / C;
  const uint32_t n2 = uint32_t(n >> M), col0 = tile.col0;
  uint32_t* dst = (cyc ? A.wr : A.wq) + so + size_t(k) * n + col0;
  const uint32_t* twf = (cyc ? A.fwdR : A.fwdQ) + size_t(k) * n;
  const uint32_t* xd = A.x + so;

  auto gld = [&](uint32_t b, uint32_t c) { return uint32_t(lz_digit_at<DL>(xd, n, col0 + c * n2, line + b * n2, P)); };
  auto gst = [&](uint32_t b, uint32_t c, uint32_t v) { st_w(dst + c * n2, line + b * n2, v); };
  auto lld = [&](uint32_t b, uint32_t c) { return lds[b * C + c * C + (line ^ ((b >> LR) & (C - 1u)) ^ ((c >> LR) & (C - 1u)))]; };
  auto lst = [&](uint32_t b, uint32_t c, uint32_t v) { lds[b * C + c * C + (line ^ ((b >> LR) & (C - 1u)) ^ ((c >> LR) & (C - 1u)))] = v; };

  constexpr int ROOTS = LzCol<M, LR>::LDS_ROOTS ? 0 : 1;  // 2^10: one round ahead, from the table
  uint32_t x[1 << LR];
  LzRoots<M, LR, 0> none;
  SchedTw<M, LR, 0> t0;
  if constexpr (ROOTS == 1) round_tw(t0, M, 0, tg, 1u, twf);
  lz_load<LR, Sched<M, LR>::template rr<0>()>(x, M, 0, tg, gld);
  if (A.neg != nullptr && threadIdx.x == 0u && col0 == 0u && A.neg[so] == 0u)
    x[0] = uint32_t(lz_red(int32_t(x[0] + 2u * uint32_t(A.c.one[k])), P));  // m' + 2, as in k_lz_row
  if constexpr (LzCol<M, LR>::LDS_ROOTS) {
    uint32_t* roots = lds + C * S;
    for (uint32_t i = threadIdx.x; i < S; i += blockDim.x) roots[i] = twf[i];
    __syncthreads();
    lz_fwd<W, M, LR, 0, 0, lz_in(W)>(x, tg, 1u, roots, P, gld, lld, lst, t0, none, [] {});
  } else {
    lz_fwd<W, M, LR, 0, ROOTS, lz_in(W)>(x, tg, 1u, twf, P, gld, lld, lst, t0, none, [] {});
  }
  lz_store<LR, RL>(x, M, DLV, tg, gst);
}

template <int M, int LR, int W>
__global__ void __launch_bounds__((LzCol<M, LR>::THREADS), (LzCol<M, LR>::WAVES)) k_lz_coli(const LzNtt A) {
  extern __shared__ uint32_t lds[];
  lz_pin(A.slot_ids, A.slot_stride, A.LN, A.KR, A.pl0, A.planes, A.cols, A.x, A.wr, A.wq, A.fwdR, A.invR, A.fwdQ, A.invQ, A.neg);
  constexpr uint32_t S = 1u << M;
  constexpr int NR = Sched<M, LR>::NR, DLV = LR * (NR - 1), RL = Sched<M, LR>::template rr<NR - 1>();
  const size_t so = size_t(lz_slot(A.slot_ids, blockIdx.y)) * A.slot_stride, n = size_t(1) << A.LN;
  const uint32_t C = (M >= 10) ? uint32_t(LzCol<M, LR>::C) : uint32_t(A.cols);
  const LzTile tile = lz_tile<M>(A, C);
  const int pl = tile.pl;
  const bool cyc = pl < A.KR;
  const int k = cyc ? pl : pl - A.KR;
  const LzP P{A.c.p[k], A.c.q[k], A.c.bar[k]};
  const uint32_t line = threadIdx.x % C, tg = threadIdx.x / C;
  const uint32_t n2 = uint32_t(n >> M);
  uint32_t* w = (cyc ? A.wr : A.wq) + so + size_t(k) * n + tile.col0;
  const uint32_t* twi = (cyc ? A.invR : A.invQ) + size_t(k) * n;

  auto gld = [&](uint32_t b, uint32_t c) { return ld_w(w + c * n2, line + b * n2); };
  auto gst = [&](uint32_t b, uint32_t c, uint32_t v) { st_w(w + c * n2, line + b * n2, v); };
  auto lld = [&](uint32_t b, uint32_t c) { return lds[b * C + c * C + (line ^ ((b >> LR) & (C - 1u)) ^ ((c >> LR) & (C - 1u)))]; };
  auto lst = [&](uint32_t b, uint32_t c, uint32_t v) { lds[b * C + c * C + (line ^ ((b >> LR) & (C - 1u)) ^ ((c >> LR) & (C - 1u)))] = v; };

  constexpr int ROOTS = LzCol<M, LR>::LDS_ROOTS ? 0 : 1;  // 2^10: one round ahead, from the table
  uint32_t x[1 << LR];
  LzRoots<M, LR, 0> none;
  SchedTw<M, LR, NR - 1> ti;
  lz_load<LR, RL>(x, M, DLV, tg, gld);
  if constexpr (LzCol<M, LR>::LDS_ROOTS) {
    uint32_t* roots = lds + C * S;
    for (uint32_t i = threadIdx.x; i < S; i += blockDim.x) roots[i] = twi[i];
    __syncthreads();
    lz_inv<W, M, LR, NR - 1, 0, true>(x, tg, 1u, roots, P, gst, lld, lst, ti, none);
  } else {
    if constexpr (ROOTS == 1) round_tw(ti, M, DLV, tg, 1u, twi);
    lz_inv<W, M, LR, NR - 1, ROOTS, true>(x, tg, 1u, twi, P, gst, lld, lst, ti, none);
  }
}

// ---------------------------------------------------------------------------
// CRT + carry, one coefficient per thread.
//
// A wave takes 64 consecutive coefficients and finishes the last 64 - ND; the
// first ND are the previous wave's, computed again for what they carry over,
// so no wave waits for another and neighbours exchange by lane shifts.  A
// coefficient V is cut into ND base-B digits d_0 .. d_{ND-1} (the last one
// signed); the sum s_i = d_0 + B-aligned digits of the ND - 1 coefficients
// below it is formed by ND - 1 shift-and-add steps; s_i = q B + r with r in
// [-B/2, B/2), and the digit is r + q of the coefficient below.  Values are
// kept exactly: what leaves lane i is what lane i + 1 adds, and what crosses
// the top of the number enters digit 0, negated modulo B^n + 1.  Digits lie in
// [-B/2 - 16, B/2 + 16).
// ---------------------------------------------------------------------------

template <int DL>
struct LzDig;
template <>
struct LzDig<2> {
  int64_t v;
};
template <>
struct LzDig<3> {
  uint64_t v;
  int32_t h;
};

// The value of the lane below (lane 0: 0).
__device__ __forceinline__ uint32_t lz_shr1(uint32_t v) {
  return uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x138, 0xf, 0xf, false));  // wave_shr:1
}
__device__ __forceinline__ LzDig<2> lz_below(const LzDig<2>& d) {
  const uint64_t u = uint64_t(d.v);
  return {int64_t(uint64_t(lz_shr1(uint32_t(u))) | (uint64_t(lz_shr1(uint32_t(u >> 32))) << 32))};
}
__device__ __forceinline__ LzDig<3> lz_below(const LzDig<3>& d) {
  return {uint64_t(lz_shr1(uint32_t(d.v))) | (uint64_t(lz_shr1(uint32_t(d.v >> 32))) << 32),
          int32_t(lz_shr1(uint32_t(d.h)))};
}
__device__ __forceinline__ LzDig<2> lz_add(const LzDig<2>& a, const LzDig<2>& b) { return {a.v + b.v}; }
__device__ __forceinline__ LzDig<3> lz_add(const LzDig<3>& a, const LzDig<3>& b) {
  const uint64_t v = a.v + b.v;
  return {v, a.h + b.h + (v < a.v ? 1 : 0)};
}
__device__ __forceinline__ LzDig<2> lz_neg(const LzDig<2>& a) { return {-a.v}; }
__device__ __forceinline__ LzDig<3> lz_neg(const LzDig<3>& a) { return {0ull - a.v, ~a.h + (a.v == 0 ? 1 : 0)}; }
__device__ __forceinline__ LzDig<2> lz_small(LzDig<2>, int32_t v) { return {int64_t(v)}; }
__device__ __forceinline__ LzDig<3> lz_small(LzDig<3>, int32_t v) { return {uint64_t(int64_t(v)), v >> 31}; }
__device__ __forceinline__ bool lz_zero(const LzDig<2>& a) { return a.v == 0; }
__device__ __forceinline__ bool lz_zero(const LzDig<3>& a) { return a.v == 0 && a.h == 0; }
__device__ __forceinline__ bool lz_minus(const LzDig<2>& a) { return a.v < 0; }
__device__ __forceinline__ bool lz_minus(const LzDig<3>& a) { return a.h < 0; }

// s = q B + r, r in [-B/2, B/2): returns q, leaves r in s.  sh = cbits mod 32
// (DL = 2: B = 2^(32 + sh), sh > 0; DL = 3: B = 2^(64 + sh)).
__device__ __forceinline__ int32_t lz_split(LzDig<2>& s, uint32_t sh) {
  const int64_t q = (s.v + (int64_t(1) << (31 + sh))) >> (32 + sh);
  s.v -= q << (32 + sh);
  return int32_t(q);
}
__device__ __forceinline__ int32_t lz_split(LzDig<3>& s, uint32_t sh) {
  // Adding B/2 = 2^(63 + sh) carries from bit 63 when sh = 0.
  const int32_t top = sh == 0u ? s.h + int32_t(s.v >> 63) : s.h + (int32_t(1) << (sh - 1u));
  const int32_t q = top >> sh;
  s.h -= int32_t(uint32_t(q) << sh);
  return q;
}

template <int DL>
__device__ __forceinline__ LzDig<DL> lz_load_digit(const uint32_t* x, size_t n, uint32_t i) {
  const uint2 d = reinterpret_cast<const uint2*>(x)[i];
  LzDig<DL> r;
  r.v = uint64_t(d.x) | (uint64_t(d.y) << 32);
  if constexpr (DL == 3) r.h = int32_t(x[2 * n + i]);
  return r;
}
template <int DL>
__device__ __forceinline__ void lz_store_digit(uint32_t* x, size_t n, uint32_t i, const LzDig<DL>& d) {
  const uint64_t u = uint64_t(d.v);
  reinterpret_cast<uint2*>(x)[i] = make_uint2(uint32_t(u), uint32_t(u >> 32));
  if constexpr (DL == 3) x[2 * n + i] = uint32_t(d.h);
}

// The lowest digit of the two's complement limbs v, which move down by B
// (their count L drops by DL - 1); the top digit is what is left.
template <int DL, int L>
__device__ __forceinline__ LzDig<DL> lz_take(uint32_t (&v)[LZ_MAXL], uint32_t sh) {
  const uint32_t mask = (1u << sh) - 1u;
  LzDig<DL> d;
  if constexpr (DL == 2) {
    d.v = int64_t(uint64_t(v[0]) | (uint64_t(v[1] & mask) << 32));
  } else {
    d.v = uint64_t(v[0]) | (uint64_t(v[1]) << 32);
    d.h = int32_t(v[2] & mask);
  }
#pragma unroll
  for (int j = 0; j + DL < L; ++j) v[j] = __builtin_amdgcn_alignbit(v[j + DL], v[j + DL - 1], sh);
  v[L - DL] = uint32_t(int32_t(v[L - 1]) >> sh);
  return d;
}
template <int DL, int L>
__device__ __forceinline__ LzDig<DL> lz_top(const uint32_t (&v)[LZ_MAXL]) {
  LzDig<DL> d;
  const uint32_t s1 = uint32_t(int32_t(v[L - 1]) >> 31);
  d.v = uint64_t(v[0]) | (uint64_t(L > 1 ? v[1] : s1) << 32);
  if constexpr (DL == 3) d.h = int32_t(L > 2 ? v[2] : s1);
  return d;
}

// d_J .. d_{ND-1} of v, then s = d_J + (what the lane below has from d_{J+1} on).
template <int DL, int L, int ND, bool NEGA, int J>
__device__ __forceinline__ LzDig<DL> lz_horner(uint32_t (&v)[LZ_MAXL], uint32_t sh, bool wrap) {
  if constexpr (J == ND - 1) {
    return lz_top<DL, L>(v);
  } else {
    const LzDig<DL> d = lz_take<DL, L>(v, sh);
    LzDig<DL> up = lz_below(lz_horner<DL, L - (DL - 1), ND, NEGA, J + 1>(v, sh, wrap));
    if (NEGA && wrap) up = lz_neg(up);
    return lz_add(d, up);
  }
}

template <int DL, int L, int ND, bool NEGA>
__device__ __forceinline__ LzDig<DL> lz_finish(uint32_t (&v)[LZ_MAXL], uint32_t sh, bool wrap) {
  LzDig<DL> s = lz_horner<DL, L, ND, NEGA, 0>(v, sh, wrap);
  const int32_t q = lz_split(s, sh);
  int32_t c = int32_t(lz_shr1(uint32_t(q)));
  if (NEGA && wrap) c = -c;
  return lz_add(s, lz_small(s, c));
}

// The lane's digit brought into [-B/2, B/2): three carry steps (a longer run of
// carries would need three digits at the edge of their range in a row, and
// keeps the value all the same).  The LZ_BALANCE lowest lanes are not final.
constexpr int LZ_BALANCE = 3;
template <int DL>
__device__ __forceinline__ LzDig<DL> lz_balance(LzDig<DL> s, uint32_t sh, bool flip) {
#pragma unroll
  for (int step = 0; step < LZ_BALANCE; ++step) {
    const int32_t q = lz_split(s, sh);
    int32_t c = int32_t(lz_shr1(uint32_t(q)));
    if (flip) c = -c;
    s = lz_add(s, lz_small(s, c));
  }
  return s;
}

// A digit as residues of the plan's first K primes.
template <int K, int DL>
__device__ __forceinline__ void lz_store_residues(uint32_t* dst, size_t n, uint32_t i, const LzDig<DL>& s) {
  uint32_t d[DIGIT_LIMBS];
  const uint64_t u = uint64_t(s.v);
  d[0] = uint32_t(u);
  d[1] = uint32_t(u >> 32);
  if constexpr (DL == 3) d[2] = uint32_t(s.h);
  else d[2] = uint32_t(int32_t(d[1]) >> 31);
#pragma unroll
  for (int k = 0; k < K; ++k) st_w(dst + size_t(k) * n, i, digit_residue_wide(d, k));
}

// The coefficient as two's complement limbs.  Column l sums KP products below p
// 2^32: 9 2^(28.2 + 32) < 2^63.4 for the shortest primes; with the wider ones
// (WIDE) the sums are kept in two halves of at most five products, below
// 2^64.
template <int SET, int KP, int L>
__device__ __forceinline__ void lz_crt(const int32_t (&r)[KP], uint32_t (&v)[LZ_MAXL]) {
  constexpr LzCrt<KP, L> C = lz_make_crt<SET, KP, L>();
  constexpr bool WIDE = lz_width(SET) > 0;
  constexpr int H = WIDE ? 4 : KP;  // products of the first half: 4 2^(29.9 + 32) < 2^64
  uint64_t col[L], cob[WIDE ? L : 1];
#pragma unroll
  for (int l = 0; l < L; ++l) col[l] = 0;
  if constexpr (WIDE) {
#pragma unroll
    for (int l = 0; l < L; ++l) cob[l] = 0;
  }
  float f = 0.5f;
#pragma unroll
  for (int k = 0; k < KP; ++k) {
    int32_t y = lz_mulc(r[k], C.c[k], C.cq[k], C.p[k]);
    y += (y >> 31) & int32_t(C.p[k]);
    f += float(y) * C.inv[k];
#pragma unroll
    for (int l = 0; l < L; ++l) {
      if (k < H) col[l] += uint64_t(uint32_t(y)) * C.M[k][l];
      else cob[WIDE ? l : 0] += uint64_t(uint32_t(y)) * C.M[k][l];
    }
  }
  const uint32_t q = uint32_t(f);
  uint64_t t = 0;
#pragma unroll
  for (int l = 0; l < L; ++l) {
    if constexpr (WIDE) {
      const uint64_t lo = (col[l] & 0xffffffffull) + (cob[l] & 0xffffffffull) + (t & 0xffffffffull) + uint64_t(q) * C.NP[l];
      v[l] = uint32_t(lo);
      t = (col[l] >> 32) + (cob[l] >> 32) + (t >> 32) + (lo >> 32);
    } else {
      // col + carry < 2^63.5 and q NP < 2^36: no overflow.
      t += col[l];
      t += uint64_t(q) * C.NP[l];
      v[l] = uint32_t(t);
      t >>= 32;
    }
  }
}

// Residue of a plane at coefficient i: the word itself, or, after a transform
// split over 2^SP workgroups, its last SP inverse levels: coefficient t 2^M + j
// from the values y_b of position j (each within 1.6 p).  The signs of a level
// hang on bits of t alone and its roots multiply out, so two sums times two
// constants of (plane, t) and one reduction do: join holds them, a pair per t
// (one for SP = 1), filled by k_lz_roots.  |sum| <= 2 3.2 p p / 2 and the result
// is within 0.8 p.  Level by level, with a reduced product for each of three
// butterflies, the two carries of 2^13 coefficients split four ways took 5.4 and
// 4.2 us, now 4.0 and 3.4; a squaring of 2^14 coefficients 30.7 us, now 27.2.
template <int SP>
struct LzJoin {
  uint32_t y[1 << SP];
  uint2 c;
  __device__ __forceinline__ void load(const uint32_t* src, uint32_t i, int LN, const uint32_t* join) {
    const int M = LN - SP;
    const uint32_t j = SP == 0 ? i : i & ((1u << M) - 1u);
#pragma unroll
    for (int b = 0; b < (1 << SP); ++b) y[b] = ld_w(src + (size_t(b) << M), j);
    if constexpr (SP == 1) c.x = ld_w(join, 2u * (i >> M));
    if constexpr (SP == 2) c = *reinterpret_cast<const uint2*>(join + 2u * (i >> M));
  }
  // neg: minus the lowest bit of t, the sign of the first level.
  __device__ __forceinline__ int32_t value(uint32_t neg, uint32_t q, uint32_t p) const {
    if constexpr (SP == 0) {
      return int32_t(y[0]);
    } else {
      int64_t v = int64_t(int32_t(y[0] + (y[1] ^ neg) - neg)) * int32_t(c.x);
      if constexpr (SP == 2) v += int64_t(int32_t(y[2] + (y[3] ^ neg) - neg)) * int32_t(c.y);
      return int32_t(v >> 32) - __mulhi(int32_t(uint32_t(v) * q), int32_t(p));
    }
  }
};

// Grid: (ceil(waves / 4), slots); block 256.
// EX > 0: the result leaves in the external format, EX residue planes at dst (one
// slot), by waves with the three more halo lanes that the balancing takes.  One
// launch and a pass over the digits less than k_lz_export behind it: a call on
// 2^10 coefficients 32.5 -> 30.4 us with its synchronisation, on 2^16 55.0 ->
// 53.9.
template <int SET, int KP, int L, int ND, int DL, bool NEGA, int EX, int SP>
__global__ void __launch_bounds__(256) k_lz_carry(const LzCarry A) {
  constexpr int H = EX > 0 ? ND + LZ_BALANCE : ND, W = 64 - H;
  lz_pin(A.src, A.dst, A.dst2, A.neg, A.slot_ids, A.slot_stride, A.LN, A.cbits, A.cbits_slot, A.snap, A.mul.a, A.mul.a_slot,
         A.mul.bits_mode, A.mul.slot_base, A.mul.bits[blockIdx.y >> 5 & (INLINE_SLOTS / 32 - 1)]);
  const size_t n = size_t(1) << A.LN;
  const uint32_t slot = lz_slot(A.slot_ids, blockIdx.y);
  const size_t so = size_t(slot) * A.slot_stride;
  const int lane = int(threadIdx.x & 63u);
  const int wave = __builtin_amdgcn_readfirstlane(int(blockIdx.x * 4u + (threadIdx.x >> 6)));
  const int top = int((n - 1) / W);
  if (wave > top) return;
  for (int w = wave;; --w) {
    const int i = w * W + lane - H;
    const uint32_t idx = i < 0 ? uint32_t(i + int(n)) : (uint32_t(i) < n ? uint32_t(i) : uint32_t(n - 1));
    // Everything that comes from memory is asked for before the first wait.
    LzJoin<SP> in[KP];
#pragma unroll
    for (int k = 0; k < KP; ++k) in[k].load(A.src + so + size_t(k) * n, idx, A.LN, A.join + 8 * k);
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t cbits = A.cbits_slot ? A.cbits_slot[slot] : uint32_t(A.cbits);
    const uint32_t sh = cbits & 31u;
    const uint32_t a = lz_multiplier(A.mul, blockIdx.y, slot);
    bool snap = false;
    if (A.dst2 != nullptr) {
      snap = A.snap != nullptr ? (A.snap[blockIdx.y] & SLOT_SNAP) != 0u
                               : (A.mul.bits_mode == 2 && ((A.mul.bits[blockIdx.y >> 5] >> (blockIdx.y & 31u)) & 1u));
    }
    int32_t r[KP];
    const uint32_t neg = SP == 0 ? 0u : 0u - ((idx >> (A.LN - SP)) & 1u);
#pragma unroll
    for (int k = 0; k < KP; ++k) r[k] = in[k].value(neg, cx_inv32(lz_prime(SET, k)), lz_prime(SET, k));
    uint32_t v[LZ_MAXL];
    lz_crt<SET, KP, L>(r, v);
    if (a != 1u) {
      uint64_t t = 0;
#pragma unroll
      for (int l = 0; l < L; ++l) {
        t += uint64_t(v[l]) * a;
        v[l] = uint32_t(t);
        t >>= 32;
      }
    }
    const LzDig<DL> d = lz_finish<DL, L, ND, NEGA>(v, sh, i == 0);
    const bool own = lane >= H && uint32_t(i) < n;
    if constexpr (EX > 0) {
      const LzDig<DL> b = lz_balance<DL>(d, sh, NEGA && i == 0);
      if (own) lz_store_residues<EX, DL>(A.dst, n, uint32_t(i), b);
      return;
    }
    if (w == wave && own) {
      lz_store_digit<DL>(A.dst + so, n, uint32_t(i), d);
      if (snap) lz_store_digit<DL>(A.dst2 + so, n, uint32_t(i), d);
    }
    if (A.neg == nullptr || wave != top) return;
    // The sign of the number is that of its highest nonzero digit: nearly
    // always the top one; the last wave goes on downwards if its digits are
    // all zero.
    const uint64_t nz = __ballot(own && !lz_zero(d));
    const uint64_t mi = __ballot(own && lz_minus(d));
    if (nz != 0ull || w == 0) {
      if (lane == 0) A.neg[so] = nz != 0ull ? uint32_t((mi >> (63 - __clzll((long long)(nz)))) & 1ull) : 0u;
      return;
    }
  }
}

// Residues of the plan's K primes -> digits (mod B^n + 1, which keeps every
// register): the CRT value of each coefficient, carried as above.
template <int K, int DL>
__global__ void __launch_bounds__(256) k_lz_import(const LzConv A) {
  constexpr int ND = 3, W = 64 - ND, L = K + 1;
  const size_t n = size_t(1) << A.LN;
  const int lane = int(threadIdx.x & 63u), w = int(blockIdx.x * 4u + (threadIdx.x >> 6));
  const int i = w * W + lane - ND;
  if (w * W >= int(n)) return;
  const uint32_t idx = i < 0 ? uint32_t(i + int(n)) : (uint32_t(i) < n ? uint32_t(i) : uint32_t(n - 1));
  uint32_t r[K], acc[L], v[LZ_MAXL];
#pragma unroll
  for (int k = 0; k < K; ++k) r[k] = ld_w(A.src + size_t(k) * n, idx);
  garner<K, L>(r, acc);
#pragma unroll
  for (int l = 0; l < L; ++l) v[l] = acc[l];
  const LzDig<DL> d = lz_finish<DL, L, ND, true>(v, uint32_t(A.cbits) & 31u, i == 0);
  if (lane >= ND && uint32_t(i) < n) lz_store_digit<DL>(A.dst, n, uint32_t(i), d);
}

// Digits -> residues of the plan's K primes, of the balanced digits.  neg: the register is m' (mod B^n - 1) of that sign, exported as the
// squaring defines it: m' + 2, plus R = B^n - 1 when negative.
template <int K, int DL>
__global__ void __launch_bounds__(256) k_lz_export(const LzConv A) {
  constexpr int H = LZ_BALANCE, W = 64 - H;
  const size_t n = size_t(1) << A.LN;
  const int lane = int(threadIdx.x & 63u), w = int(blockIdx.x * 4u + (threadIdx.x >> 6));
  const int i = w * W + lane - H;
  if (w * W >= int(n)) return;
  const uint32_t idx = i < 0 ? uint32_t(i + int(n)) : (uint32_t(i) < n ? uint32_t(i) : uint32_t(n - 1));
  const uint32_t sh = uint32_t(A.cbits) & 31u;
  LzDig<DL> s = lz_load_digit<DL>(A.src, n, idx);
  s = lz_balance<DL>(s, sh, A.neg == nullptr && i == 0);
  if (lane < H || uint32_t(i) >= n) return;
  if (A.neg != nullptr) {
    const bool neg = A.neg[0] != 0u;
    if (i == 0) s = lz_add(s, lz_small(s, neg ? 1 : 2));
    if (neg && uint32_t(i) == n - 1) {
      if constexpr (DL == 2) s.v += int64_t(1) << (32 + sh);
      else s.h += int32_t(1) << sh;
    }
  }
  lz_store_residues<K, DL>(A.dst, n, uint32_t(i), s);
}

// A register that holds a non-negative number below B^n / 2, as binary words: 2
// cbits words per wave of 64 digits, list position after list position.  Digit
// i borrows from digit i + 1 when the highest nonzero digit at or below it is
// negative: a ballot finds it in the wave, and the digits before the wave are
// searched 64 at a time (one step unless they are all zero).
// Grid: (ceil(n / 256), positions); block 256; digits from `count` on are zero.
template <int DL>
__global__ void __launch_bounds__(256) k_lz_pack(const LzPack A) {
  __shared__ uint32_t u[4][64 * DL + 1];
  const size_t n = size_t(1) << A.LN;
  const uint32_t slot = lz_slot(A.slot_ids, blockIdx.y);
  const uint32_t* x = A.src + size_t(slot) * A.slot_stride;
  const uint32_t cb = A.cbits_slot ? A.cbits_slot[slot] : uint32_t(A.cbits), sh = cb & 31u;
  const int lane = int(threadIdx.x & 63u), wv = int(threadIdx.x >> 6);
  const uint32_t w0 = blockIdx.x * 256u + uint32_t(wv) * 64u;
  LzDig<DL> d = lz_load_digit<DL>(x, n, w0 + uint32_t(lane));
  const uint64_t nz = __ballot(!lz_zero(d)), mi = __ballot(lz_minus(d));
  uint32_t below = 0;  // whether the digits before the wave are a negative number
  for (uint32_t b = w0; b != 0u; b -= 64u) {
    const LzDig<DL> e = lz_load_digit<DL>(x, n, b - 64u + uint32_t(lane));
    const uint64_t ez = __ballot(!lz_zero(e)), em = __ballot(lz_minus(e));
    if (ez != 0ull) {
      below = uint32_t((em >> (63 - __clzll((long long)ez))) & 1ull);
      break;
    }
  }
  const uint64_t under = nz & ((1ull << lane) - 1ull);
  const uint32_t borrow = under != 0ull ? uint32_t((mi >> (63 - __clzll((long long)under))) & 1ull) : below;
  d = lz_add(d, lz_small(d, -int32_t(borrow)));
  if (lz_minus(d)) {
    if constexpr (DL == 2) d.v += int64_t(1) << (32 + sh);
    else d.h += int32_t(1) << sh;
  }
  u[wv][lane * DL] = uint32_t(uint64_t(d.v));
  u[wv][lane * DL + 1] = uint32_t(uint64_t(d.v) >> 32);
  if constexpr (DL == 3) u[wv][lane * DL + 2] = uint32_t(d.h);
  if (lane == 0) u[wv][64 * DL] = 0u;
  __syncthreads();
  uint32_t* out = A.dst + size_t(blockIdx.y) * A.out_stride + size_t(w0 / 32u) * cb;
  for (uint32_t w = uint32_t(lane); w < 2u * cb; w += 64u) {
    // Bits [32 w, 32 w + 32) of the wave's digits: at most two digits (cb >= 32).
    const uint32_t i = (32u * w) / cb, off = 32u * w - i * cb, k = off >> 5, r = off & 31u;
    const uint32_t* p = &u[wv][i * DL];
    uint32_t v = p[k] >> r;
    if (r != 0u && int(k) + 1 < DL) v |= p[k + 1] << (32u - r);
    const uint32_t have = cb - off;  // bits of digit i from off on
    if (have < 32u) v = (v & ((1u << have) - 1u)) | (i < 63u ? p[DL] << have : 0u);
    out[w] = v;
  }
}

// Root tables (heap-indexed as make_tables in plan.h) in signed Montgomery form,
// |w| <= p / 2: entry 2^l + b is psi^e with e = 2 h brv_l(b) (cyclic) or h (2
// brv_l(b) + 1) (negacyclic), h = n / 2^{l+1}, or its inverse psi^{2n - e}.  pw
// holds psi^i for i < 2^s, then psi^{i 2^s}, per prime (s = ceil(LN / 2)).  Behind
// the tables, for a transform split over 2^SP workgroups, eight words per plane
// (KR cyclic, KQ negacyclic) for LzJoin.
__global__ void __launch_bounds__(256)
k_lz_roots(uint32_t* tw, const uint32_t* pw, int LN, int SP, int KR, int KQ, const LzPrimes C) {
  const uint32_t n = 1u << LN, idx = blockIdx.x * 256u + threadIdx.x;
  const int k = int(blockIdx.y);
  if (idx >= n) return;
  const LzP P{C.p[k], C.q[k], C.bar[k]};
  const int s = (LN + 1) / 2;
  const uint32_t* w = pw + size_t(k) * ((1u << s) + (1u << (LN + 1 - s)));
  const int l = idx == 0u ? 0 : 31 - __clz(int(idx));
  const uint32_t b = idx == 0u ? 0u : idx - (1u << l);
  const uint32_t br = l == 0 ? 0u : __brev(b) >> (32 - l), h = n >> (l + 1), mask = 2u * n - 1u;
  auto root = [&](uint32_t e) {
    const int32_t lo = int32_t(w[e & ((1u << s) - 1u)]), hi = int32_t(w[(1u << s) + (e >> s)]);
    uint32_t v = uint32_t(lz_red(lz_mul(lo, hi, P), P));
    if (v >= P.p) v -= P.p;
    return v > P.p / 2 ? v - P.p : v;
  };
  const uint32_t eR = idx == 0u ? 0u : (2u * h * br) & mask, eQ = idx == 0u ? 0u : (h * (2u * br + 1u)) & mask;
  tw[size_t(k) * n + idx] = root(eR);
  tw[(size_t(KR) + k) * n + idx] = root((2u * n - eR) & mask);
  if (k < KQ) {
    tw[(2 * size_t(KR) + k) * n + idx] = root(eQ);
    tw[(2 * size_t(KR) + KQ + k) * n + idx] = root((2u * n - eQ) & mask);
  }
  if (SP > 0 && idx < (2u << SP)) {
    // Of coefficient block t: the factor of y_0 (idx even) or y_2, inverse roots
    // of entries 1 (the last level) and 2 or 3, and -1 = psi^n where the last
    // level subtracts.
    const uint32_t t = idx >> 1, j = idx & 1u, last = t >> (SP - 1), first = SP == 2 ? t & 1u : 0u;
    uint32_t* join = tw + (2 * size_t(KR) + 2 * size_t(KQ)) * n;
    const uint32_t sign = last != 0u && j != 0u ? n : 0u;
    const uint32_t cyc = first * j * (n / 2u), nega = last * (n / 2u) + first * (n / 4u) * (1u + 2u * j);
    join[8 * k + idx] = root((2u * n - cyc + sign) & mask);
    if (k < KQ) join[8 * (KR + k) + idx] = root((2u * n - nega + sign) & mask);
  }
}

// Instantiations, looked up by the host engine (lz_geometry chooses among
// them): whole transforms, split ones, row passes, column passes.
#define LZ_ROW(M, LR, SRC, W, SP)                                             \
  template __global__ void k_lz_row<M, LR, LZ_SQR, SRC, W, SP>(const LzNtt);  \
  template __global__ void k_lz_row<M, LR, LZ_MULN, SRC, W, SP>(const LzNtt); \
  template __global__ void k_lz_row<M, LR, LZ_GEN, SRC, W, SP>(const LzNtt);
#define LZ_ROW1(M, LR, SP) LZ_ROW(M, LR, 2, 0, SP) LZ_ROW(M, LR, 3, 0, SP)
LZ_ROW1(8, 3, 0)
LZ_ROW1(9, 3, 0)
LZ_ROW1(10, 3, 0)
LZ_ROW1(11, 3, 0)
LZ_ROW1(12, 3, 0)
LZ_ROW1(10, 4, 0)
LZ_ROW1(11, 4, 0)
LZ_ROW1(12, 4, 0)
LZ_ROW1(13, 4, 0)
LZ_ROW1(11, 3, 1)
LZ_ROW1(12, 3, 1)
LZ_ROW1(11, 3, 2)
LZ_ROW1(12, 3, 2)
LZ_ROW(7, 3, 0, 0, 0)
LZ_ROW(8, 3, 0, 0, 0)
LZ_ROW(9, 3, 0, 0, 0)
LZ_ROW(10, 4, 0, 0, 0)
LZ_ROW(11, 3, 0, 0, 0)
LZ_ROW(12, 4, 0, 0, 0)
LZ_ROW(11, 4, 0, 1, 0)
LZ_ROW(12, 4, 0, 2, 0)
#define LZ_COL(M, LR, W)                                        \
  template __global__ void k_lz_colf<M, LR, 2, W>(const LzNtt); \
  template __global__ void k_lz_colf<M, LR, 3, W>(const LzNtt); \
  template __global__ void k_lz_coli<M, LR, W>(const LzNtt);
LZ_COL(7, 4, 0)
LZ_COL(8, 4, 0)
LZ_COL(10, 5, 1)
LZ_COL(10, 5, 2)
#define LZ_CARRY(SET, SP)                                                            \
  template __global__ void k_lz_carry<SET, 6, 6, 5, 2, false, 0, SP>(const LzCarry);\
  template __global__ void k_lz_carry<SET, 4, 4, 3, 2, true, 0, SP>(const LzCarry); \
  template __global__ void k_lz_carry<SET, 4, 4, 3, 2, true, 3, SP>(const LzCarry); \
  template __global__ void k_lz_carry<SET, 7, 7, 4, 2, false, 0, SP>(const LzCarry);\
  template __global__ void k_lz_carry<SET, 5, 5, 3, 2, true, 0, SP>(const LzCarry); \
  template __global__ void k_lz_carry<SET, 5, 5, 3, 2, true, 4, SP>(const LzCarry); \
  template __global__ void k_lz_carry<SET, 9, 8, 4, 3, false, 0, SP>(const LzCarry);\
  template __global__ void k_lz_carry<SET, 6, 6, 3, 3, true, 0, SP>(const LzCarry); \
  template __global__ void k_lz_carry<SET, 6, 6, 3, 3, true, 5, SP>(const LzCarry);
LZ_CARRY(0, 0)
LZ_CARRY(0, 1)
LZ_CARRY(0, 2)
LZ_CARRY(1, 0)
LZ_CARRY(2, 0)
LZ_CARRY(3, 0)
template __global__ void k_lz_pack<2>(const LzPack);
template __global__ void k_lz_pack<3>(const LzPack);
#define LZ_CONV(K, DL)                                        \
  template __global__ void k_lz_import<K, DL>(const LzConv);  \
  template __global__ void k_lz_export<K, DL>(const LzConv);
LZ_CONV(3, 2)
LZ_CONV(4, 2)
LZ_CONV(5, 3)

}  // namespace annie
