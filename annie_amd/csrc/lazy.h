// The short-prime path: MMGW squarings on digit registers with 28-bit primes.
//
// A register is kept as its signed base-B digits (B = 2^cbits).  One product
// x y of two registers takes two carries and, in each RNS prime plane, two
// rounds of transforms:
//
//   cyclic planes      x^ y^ n^   -> m' = a x y N^-1 mod R   (one triple product)
//   negacyclic planes  m'^ N^ - a x^ y^ -> r' = m' N - a x y mod Q
//
// The triple product needs planes for n^2 (B/2)^3 instead of n (B/2)^2, but
// takes the carry of T_R and one forward and one inverse transform out of the
// chain, and the difference is taken between transforms, which takes the
// inverse transform and the carry of T_Q out (src/transformGPU.h:523-568 does
// each product on its own).
//
// The primes are below 2^28.2 (2^29.9 at 2^22), so that a signed 32-bit word
// holds +-6.9 p (2.1 p) and a butterfly needs no correction: see lazy.hip.  More
// planes (7 + 5 instead of 4 per transform at K = 4) and fewer transforms come to
// 29 plane transforms a squaring instead of 32, each at half the instructions, in
// four launches (lengths up to 2^13) or eight instead of six or twelve.
//
// Measured against the passes over the long primes, us per squaring: 2^10 (K = 4)
// 43.9 -> 14.0, 2^13 61.9 -> 19.7, 2^14 (K = 5) 77.4 -> 27.1, 2^16 78.6 -> 35.6,
// 2^19 154 -> 85.5, 2^21 (K = 5) 473 -> 347, 2^22 810 -> 599; one tick of a batch
// with its read-back: 130 slots of 2^12 138 -> 60, 300 slots of 2^9 (K = 5) 124 ->
// 33.5, nine of 2^13 71 -> 28.  2^23 has too few such primes and stays on the long
// ones.
#pragma once
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <vector>

#include "kernels.h"
#include "plan.h"

namespace annie {

constexpr int LZ_MAXP = 9;     // prime planes of a transform
constexpr int LZ_MAXL = 8;     // 32-bit limbs of a CRT value
constexpr uint32_t LZ_MAX_A = 4095;  // largest multiplier that the carries have room for
constexpr int LZ_MAX_LN = 22;

// The primes, k 2^e + 1: set 0 (e = 20, below 2^28.2) serves lengths up to 2^19,
// sets 1 - 3 (e = 21, 22, 23, below 2^28.2, 2^29.3, 2^29.9) 2^20 - 2^22: the
// negacyclic transform needs 2^{LN + 1}-th roots of unity, and these are the
// largest such primes below the fewest bits that leave enough of them.  Fixed
// sets make the CRT's constants instruction literals.
constexpr int LZ_SETS = 4;
constexpr uint32_t LZ_K[LZ_SETS][LZ_MAXP] = {{291, 277, 262, 258, 246, 238, 235, 220, 211},
                                             {131, 129, 123, 119, 110, 101, 95, 89, 81},
                                             {154, 142, 112, 99, 90, 55, 40, 39, 37},
                                             {119, 107, 105, 90, 77, 71, 56, 45, 20}};
constexpr int lz_set(int LN) { return LN <= 19 ? 0 : LN - 19; }
constexpr int lz_width(int set) { return set <= 1 ? 0 : set - 1; }  // W in lazy.hip
constexpr uint32_t lz_prime(int set, int k) { return (LZ_K[set][k] << (20 + set)) + 1u; }

// Planes and limbs of RNS size K of the plan (K = 3, 4, 5).
struct LzShape {
  int KR, KQ;  // cyclic planes (m'), negacyclic planes (r')
  int DL;      // 32-bit limbs of a digit
};
static inline LzShape lz_shape(int K) {
  if (K == 3) return {6, 4, 2};
  if (K == 4) return {7, 5, 2};
  return {9, 6, 3};
}

// Constants of one transform prime and of the register format.
struct LzPrimes {
  uint32_t p[LZ_MAXP], q[LZ_MAXP];  // prime, p^-1 mod 2^32
  uint32_t bar[LZ_MAXP];            // floor(2^58 / p): quotients by p
  int32_t cq[LZ_MAXP];              // 2^32 times the scale of x^ y^, n^-1 b^-2 2^64, b = 2^{-32 (DL - 1)}
  int32_t one[LZ_MAXP];             // transform of the register 1: b mod p
};

// Where the multiplier and the snapshot flag of each list position come from
// (see CarryArgs): one multiplier for all, an array, or bits.
struct LzMult {
  uint32_t a;
  const uint32_t* a_slot;
  int bits_mode;  // 1: slot_base[slot] where the position's bit is set, else 1
  const uint32_t* slot_base;
  uint32_t bits[INLINE_SLOTS / 32];
};

enum LzMode : int {
  LZ_SQR = 0,   // cyclic planes: (x^)^2 n^ and back; negacyclic: a (x^)^2
  LZ_MULN = 1,  // negacyclic planes: m'^ N^ - t^ and back
  LZ_GEN = 2,   // one of the operations below, chosen at run time
};
enum LzOp : int {
  LZ_FWD = 0,    // forward, times `scale` where it is given
  LZ_MULY = 1,   // as LZ_SQR with x^ y^
  LZ_MUL1 = 2,   // as LZ_SQR with x^ 1^
};

// One NTT pass over planes [pl0, pl0 + gridDim.z): plane k < KR is the cyclic
// transform of prime k, plane KR + k the negacyclic one.  Pointers address
// slot 0; slot s lies at + s * slot_stride words.
struct LzNtt {
  LzPrimes c;
  const uint32_t *fwdR, *invR, *fwdQ, *invQ;  // roots, prime k at + k n
  const uint32_t* x;                          // digits (first pass)
  uint32_t *wr, *wq;                          // cyclic / negacyclic planes
  const uint32_t *tq;                         // LZ_MULN: t^ planes
  const uint32_t *yr, *yq;                    // LZ_MULY: y^ planes
  const uint32_t *nir, *nq;                   // transformed N^-1 mod R and N
  const uint32_t* neg;                        // first pass over m': its sign (null: x is no m')
  const uint32_t* slot_ids;
  size_t slot_stride;
  int LN, m1, KR, pl0, planes, cols, op;
  int32_t scale[LZ_MAXP];                     // LZ_FWD: scale of each prime's planes (0: none)
  LzMult mul;
};

// CRT of the planes and carry.
struct LzCarry {
  const uint32_t* src;                        // planes
  const uint32_t* join;                       // constants of a split transform (LzJoin), prime k at + 8 k
  uint32_t* dst;                              // digits
  uint32_t* dst2;                             // snapshot of flagged positions, or null
  uint32_t* neg;                              // receives the sign of the number, or null
  const uint32_t* slot_ids;
  size_t slot_stride;
  int LN, cbits;
  const uint32_t* cbits_slot;
  const uint32_t* snap;                       // per-position flags (SLOT_SNAP), or null; bits_mode 2: mul.bits
  LzMult mul;                                 // multiplier of every coefficient
};

// Digits <-> residues of the plan's K primes (the external register format).
struct LzConv {
  const uint32_t* src;
  uint32_t* dst;
  const uint32_t* neg;  // export of m': + 2 (and + R - 2 + ... when negative), or null
  int LN, cbits;
};

// Digits -> binary words.
struct LzPack {
  const uint32_t* src;
  uint32_t* dst;  // out_stride words per list position
  const uint32_t* slot_ids;
  size_t slot_stride, out_stride;
  int LN, cbits;
  const uint32_t* cbits_slot;
};

static inline std::vector<uint32_t> lz_primes(int LN, int count) {
  std::vector<uint32_t> out;
  for (int k = 0; k < count && LN <= LZ_MAX_LN; ++k) out.push_back(lz_prime(lz_set(LN), k));
  return out;
}

// CRT constants of the first KP primes of a set, on L limbs (modulo 2^{32 L}):
// V = sum y_i M_i - round(sum y_i / p_i) P with y_i = r_i M_i^-1 mod p_i, M_i = P /
// p_i; c: M_i^-1 in signed Montgomery form, cq = c p^-1 mod 2^32, NP = -P.
template <int KP, int L>
struct LzCrt {
  uint32_t p[KP], cq[KP], M[KP][L], NP[L];
  int32_t c[KP];
  float inv[KP];
};

template <int SET, int KP, int L>
constexpr LzCrt<KP, L> lz_make_crt() {
  LzCrt<KP, L> t{};
  auto times = [](uint32_t (&v)[L], uint32_t m) {
    uint64_t c = 0;
    for (int l = 0; l < L; ++l) {
      c += uint64_t(v[l]) * m;
      v[l] = uint32_t(c);
      c >>= 32;
    }
  };
  uint32_t P[L] = {1};
  for (int k = 0; k < KP; ++k) times(P, lz_prime(SET, k));
  uint64_t borrow = 0;
  for (int l = 0; l < L; ++l) {
    const uint64_t v = 0 - uint64_t(P[l]) - borrow;
    t.NP[l] = uint32_t(v);
    borrow = (v >> 32) ? 1 : 0;
  }
  for (int k = 0; k < KP; ++k) {
    const uint32_t p = lz_prime(SET, k);
    uint32_t M[L] = {1};
    uint64_t r = 1;
    for (int j = 0; j < KP; ++j)
      if (j != k) {
        times(M, lz_prime(SET, j));
        r = r * lz_prime(SET, j) % p;
      }
    for (int l = 0; l < L; ++l) t.M[k][l] = M[l];
    const uint32_t c = uint32_t((uint64_t(cx_powmod(uint32_t(r), uint64_t(p) - 2, p)) << 32) % p);
    t.p[k] = p;
    t.c[k] = c > p / 2 ? int32_t(c) - int32_t(p) : int32_t(c);
    t.cq[k] = uint32_t(t.c[k]) * cx_inv32(p);
    t.inv[k] = float(1.0 / double(p));
  }
  return t;
}

// A generator of the 2-part: g with g^((p-1)/2) = -1 (any quadratic
// non-residue), so that g^((p-1) / 2^j) has order exactly 2^j.
static inline uint32_t lz_nonresidue(uint32_t p) {
  uint32_t g = 2;
  while (powmod_plain(g, (uint64_t(p) - 1) / 2, p) != p - 1) ++g;
  return g;
}

// Whether a plan with digit width cbits runs on the short-prime path: digits
// of the shapes that the carries are built for, and CRT ranges wide enough
// for every coefficient.  Digits lie in [-B/2 - 16, B/2 + 16), so the cyclic
// coefficients are below n^2 (B/2)^3 and the negacyclic ones below
// (1 + a) n (B/2)^2 (both by a factor 1 + 2^-20); with 0.4 bits to spare the
// quotient sum y_i / p_i, exact to 2^-19 in single precision, rounds right.
static inline bool lz_fits(const Plan& pl, int cbits, uint32_t a, const std::vector<uint32_t>& primes) {
  if (pl.K < 3 || pl.K > 5 || pl.LN < 8 || pl.LN > LZ_MAX_LN || a > LZ_MAX_A) return false;
  const LzShape sh = lz_shape(pl.K);
  if (pl.K == 5 ? (cbits < 64 || cbits > 76) : (cbits < 34 || cbits > 59)) return false;
  if (int(primes.size()) < sh.KR) return false;
  double lr = 0, lq = 0;
  for (int k = 0; k < sh.KR; ++k) lr += std::log2(double(primes[k]));
  for (int k = 0; k < sh.KQ; ++k) lq += std::log2(double(primes[k]));
  const double needR = 2.0 * pl.LN + 3.0 * cbits - 2.0, needQ = pl.LN + 2.0 * cbits - 1.0 + std::log2(1.0 + a);
  // The carries keep 4 (K = 3: 5) and 3 digits of a value times a.
  const int nd = pl.K == 3 ? 5 : 4;
  return needR + 0.4 < lr && needQ + 0.4 < lq && needR + std::log2(double(a)) < nd * cbits + 2.0 &&
         needQ < 3.0 * cbits + 3.0;
}

}  // namespace annie
