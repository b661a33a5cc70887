// gl_field.h -- Goldilocks field arithmetic for gfx950 (p = 2^64 - 2^32 + 1).
//
// Written from the field's special form, not from the reference's carry-chain code:
//   2^64 = 2^32 - 1 (mod p),   2^96 = -1 (mod p),   2^192 = 1 (mod p).
// Every function here takes canonical operands (< p) unless it says otherwise and returns a
// canonical result, so stored results compare bit-exactly with the CPU oracle.  The device
// arithmetic is built from single-instruction asm statements (namespace isa below).
// Semantics replaced: crates/boojum-cuda/native/goldilocks.cuh:90-183 (add/sub/mul/reduce).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gl {

typedef uint64_t u64;
typedef uint32_t u32;

constexpr u64 P = 0xFFFFFFFF00000001ull;
constexpr u64 EPS = 0xFFFFFFFFull;  // 2^64 mod p

__host__ __device__ __forceinline__ u64 canon(u64 x) { return x >= P ? x - P : x; }

// Device memory read and written through the global address space.  Through a generic pointer
// (one loaded from memory, or derived from one) the compiler emits flat_* instructions, which
// count against lgkmcnt as well as vmcnt: every wait for an LDS access then also waits for the
// flat loads and stores still in flight, serialising a tile's stores behind its LDS reads.
// global_* instructions count against vmcnt only.
template <typename T>
__device__ __forceinline__ T gload(const T *p) {
  return *(const __attribute__((address_space(1))) T *)p;
}
template <typename T>
__device__ __forceinline__ void gstore(T *p, T v) {
  *(__attribute__((address_space(1))) T *)p = v;
}

// Single gfx950 instructions, one asm statement each, with carries and lane masks in SGPR pairs:
// the compiler schedules them like any other instruction (interleaving independent work) and
// inserts the wait states a VALU-written SGPR needs before a VALU or SALU instruction reads it.
// What they cost (measured on MI355X, waves of 64 at 8 per SIMD): every instruction here issues
// at the full-width VALU rate (4.2-4.9 cycles per wave instruction per SIMD: carry-writing adds,
// v_mad_u64_u32, 64-bit compares and shifts alike); so the arithmetic below is written for the
// fewest VALU instructions, and among those for the fewest scalar mask operations (plain C on the
// 64-bit lane masks) between them, each of which costs the chain wait states (see add_eps).
namespace isa {

__device__ __forceinline__ u32 lo(u64 x) { return (u32)x; }
__device__ __forceinline__ u32 hi(u64 x) { return (u32)(x >> 32); }
__device__ __forceinline__ u64 pack(u32 l, u32 h) { return ((u64)h << 32) | l; }

// a + b, carry out
__device__ __forceinline__ u32 add_co(u32 a, u32 b, u64 &co) {
  u32 r;
  asm("v_add_co_u32 %0, %1, %2, %3" : "=v"(r), "=s"(co) : "v"(a), "v"(b));
  return r;
}
// a + b + ci, carry out
__device__ __forceinline__ u32 addc(u32 a, u32 b, u64 ci, u64 &co) {
  u32 r;
  asm("v_addc_co_u32 %0, %1, %2, %3, %4" : "=v"(r), "=s"(co) : "v"(a), "v"(b), "s"(ci));
  return r;
}
// a + ci, carry out
__device__ __forceinline__ u32 addc0(u32 a, u64 ci, u64 &co) {
  u32 r;
  asm("v_addc_co_u32 %0, %1, %2, 0, %3" : "=v"(r), "=s"(co) : "v"(a), "s"(ci));
  return r;
}
__device__ __forceinline__ u32 addc0(u32 a, u64 ci) {
  u64 co;
  return addc0(a, ci, co);
}
// a - b, borrow out
__device__ __forceinline__ u32 sub_co(u32 a, u32 b, u64 &bo) {
  u32 r;
  asm("v_sub_co_u32 %0, %1, %2, %3" : "=v"(r), "=s"(bo) : "v"(a), "v"(b));
  return r;
}
// a - b - bi, borrow out
__device__ __forceinline__ u32 subb(u32 a, u32 b, u64 bi, u64 &bo) {
  u32 r;
  asm("v_subb_co_u32 %0, %1, %2, %3, %4" : "=v"(r), "=s"(bo) : "v"(a), "v"(b), "s"(bi));
  return r;
}
// a - bi, borrow out
__device__ __forceinline__ u32 subb0(u32 a, u64 bi, u64 &bo) {
  u32 r;
  asm("v_subb_co_u32 %0, %1, %2, 0, %3" : "=v"(r), "=s"(bo) : "v"(a), "s"(bi));
  return r;
}
__device__ __forceinline__ u32 subb0(u32 a, u64 bi) {
  u64 bo;
  return subb0(a, bi, bo);
}
// a b + c (64-bit c), carry out
__device__ __forceinline__ u64 mad(u32 a, u32 b, u64 c, u64 &co) {
  u64 r;
  asm("v_mad_u64_u32 %0, %1, %2, %3, %4" : "=v"(r), "=s"(co) : "v"(a), "v"(b), "v"(c));
  return r;
}
// a b (full 64-bit product)
__device__ __forceinline__ u64 mul32(u32 a, u32 b) {
  u64 r, co;
  asm("v_mad_u64_u32 %0, %1, %2, %3, 0" : "=v"(r), "=s"(co) : "v"(a), "v"(b));
  return r;
}
// h (2^32 - 1) + l, carry out (the multiplier is the inline constant -1)
__device__ __forceinline__ u64 mad_eps(u32 h, u64 l, u64 &co) {
  u64 r;
  asm("v_mad_u64_u32 %0, %1, %2, -1, %3" : "=v"(r), "=s"(co) : "v"(h), "v"(l));
  return r;
}
// lane mask of x >= p
__device__ __forceinline__ u64 ge_p(u64 x) {
  u64 m;
  asm("v_cmp_ge_u64_e64 %0, %1, %2" : "=s"(m) : "v"(x), "s"(P));
  return m;
}
// 1 in the lanes of m, else 0
__device__ __forceinline__ u32 one_if(u64 m) {
  u32 r;
  asm("v_cndmask_b32_e64 %0, 0, 1, %1" : "=v"(r) : "s"(m));
  return r;
}

// x + EPS in the lanes of m, wrapping mod 2^64.  2 VALU and no mask logic: a form with a borrowing
// subtract and a carrying add is as many VALU instructions, but puts a scalar mask operation and
// three wait states into the chain (12-bit contiguous NTT pass 5 % slower).
__device__ __forceinline__ u64 add_eps(u64 x, u64 m) { return (u64)one_if(m) * (u32)EPS + x; }
// x - EPS in the lanes of m (low word + 1, high word - 1 unless the low word carried)
__device__ __forceinline__ u64 minus_eps(u32 x0, u32 x1, u64 m) {
  u64 k;
  const u32 r0 = addc0(x0, m, k);
  return pack(r0, subb0(x1, m & ~k));
}

}  // namespace isa

// a, b < p: canonical a + b.  s = a + b with carry c; when c, s + EPS (= a + b - p < p); when
// not, s >= p selects s + EPS (wrapping to s - p).  5 VALU.
__device__ __forceinline__ u64 add(u64 a, u64 b) {
  using namespace isa;
  u64 c, c2;
  const u32 s0 = add_co(lo(a), lo(b), c);
  const u32 s1 = addc(hi(a), hi(b), c, c2);
  return add_eps(pack(s0, s1), c2 | ge_p(pack(s0, s1)));
}

// a < p, b < p: canonical a - b.  d = a - b with borrow; a borrow selects d - EPS (= a - b + p,
// in (0, p)).  With a any u64 and b < p the result is a lazy residue in [0, 2^64): d - EPS
// cannot wrap since then d >= 2^64 - b > EPS.  4 VALU.
__device__ __forceinline__ u64 sub(u64 a, u64 b) {
  using namespace isa;
  u64 c, bw;
  const u32 d0 = sub_co(lo(a), lo(b), c);
  const u32 d1 = subb(hi(a), hi(b), c, bw);
  return minus_eps(d0, d1, bw);
}

// Canonical form of any u64: x >= p selects x + EPS (wrapping to x - p).  3 VALU.
__device__ __forceinline__ u64 reduce1(u64 x) {
  using namespace isa;
  return add_eps(x, ge_p(x));
}

__device__ __forceinline__ u64 neg(u64 a) { return a ? P - a : 0; }

// Canonical residue of lo + hl (2^32 - 1) - hh - bi (lo < 2^64; hl, hh < 2^32, hh + bi < 2^32; bi a
// 0/1 lane mask), i.e. of lo + (hl + (hh + bi) 2^32) 2^64 by 2^64 = 2^32 - 1 and 2^96 = -1.
//   t = lo - hh - bi; a borrow selects t - EPS (t > 2^64 - 2^32 then, no wrap);
//   R = hl EPS + t with carry c (one v_mad_u64_u32); a carry selects R + EPS, canonical since
//   R < hl EPS <= (2^32 - 1)^2; without one, R >= p selects R + EPS (wrapping to R - p).
// 8 VALU, 2 scalar mask operations.
__device__ __forceinline__ u64 reduce3b(u64 lo_, u32 hl, u32 hh, u64 bi) {
  using namespace isa;
  u64 c, b1, b;
  const u32 t0 = subb(lo(lo_), hh, bi, b1);
  const u32 t1 = subb0(hi(lo_), b1, b);
  const u64 R = mad_eps(hl, minus_eps(t0, t1, b), c);
  return add_eps(R, c | ge_p(R));
}
__device__ __forceinline__ u64 reduce3(u64 lo_, u32 hl, u32 hh) {
  using namespace isa;
  u64 c, b1, b;
  const u32 t0 = sub_co(lo(lo_), hh, b1);
  const u32 t1 = subb0(hi(lo_), b1, b);
  const u64 R = mad_eps(hl, minus_eps(t0, t1, b), c);
  return add_eps(R, c | ge_p(R));
}

// Canonical residue of lo + hl (2^32 - 1) (lo < 2^64, hl < 2^32): R = hl EPS + lo with carry c;
// when c, R + EPS is canonical (R < hl EPS); otherwise R >= p selects R + EPS (= R - p).  4 VALU.
__device__ __forceinline__ u64 reduce2(u64 lo_, u32 hl) {
  using namespace isa;
  u64 c;
  const u64 R = mad_eps(hl, lo_, c);
  return add_eps(R, c | ge_p(R));
}

// Reduces lo + hi * 2^64 (any 128-bit value) to a canonical residue.
__device__ __forceinline__ u64 reduce128(u64 lo_, u64 hi_) { return reduce3(lo_, (u32)hi_, (u32)(hi_ >> 32)); }

// a, b any u64; result canonical.  The 128-bit product is a0 b0 + (a0 b1 + a1 b0) 2^32 +
// a1 b1 2^64 from four v_mad_u64_u32 (the middle sum's carry cy weighs 2^96 = -1 mod p); its
// words r0..r3 reduce as [r0, r1] + r2 EPS - r3 - cy.  15 VALU, no register moves.
__device__ __forceinline__ u64 mul(u64 a, u64 b) {
  using namespace isa;
  u64 cy, k1, k2, dead;
  const u64 z = mul32(lo(a), lo(b));
  const u64 x = mul32(hi(a), lo(b));
  const u64 y = mad(lo(a), hi(b), x, cy);
  const u64 w = mul32(hi(a), hi(b));
  const u32 r1 = add_co(hi(z), lo(y), k1);
  const u32 r2 = addc(lo(w), hi(y), k1, k2);
  const u32 r3 = addc0(hi(w), k2, dead);
  return reduce3b(pack(lo(z), r1), r2, r3, cy);
}

// a, b any u64; result a lazy residue (any u64).  The words r0..r3 and cy as in mul:
//   t = [r0, r1] - r3 - cy; a borrow selects t - EPS (t > 2^64 - 2^32, no wrap);
//   R = r2 EPS + t; a carry selects R + EPS (R < r2 EPS <= (2^32 - 1)^2, no wrap).
// 14 VALU, and two scalar mask operations where mul has six.
__device__ __forceinline__ u64 mul_lazy(u64 a, u64 b) {
  using namespace isa;
  u64 cy, k1, k2, b1, bw, c, dead;
  const u64 z = (u64)lo(a) * lo(b);
  const u64 x = (u64)hi(a) * lo(b);
  const u64 y = mad(lo(a), hi(b), x, cy);
  const u64 w = (u64)hi(a) * hi(b);
  const u32 r1 = add_co(hi(z), lo(y), k1);
  const u32 r2 = addc(lo(w), hi(y), k1, k2);
  const u32 r3 = addc0(hi(w), k2, dead);
  const u32 t0 = subb(lo(z), r3, cy, b1);
  const u32 t1 = subb0(r1, b1, bw);
  const u64 R = mad_eps(r2, minus_eps(t0, t1, bw), c);
  return (u64)one_if(c) * (u32)EPS + R;
}

// a any u64, b < p; lazy a + b: a carry selects s + EPS (s < p - 1 then, no wrap).  4 VALU.
__device__ __forceinline__ u64 add_lazy(u64 a, u64 b) {
  using namespace isa;
  u64 c, c2, dead;
  const u32 s0 = add_co(lo(a), lo(b), c);
  const u32 s1 = addc(hi(a), hi(b), c, c2);
  return mad_eps(one_if(c2), pack(s0, s1), dead);
}

__device__ __forceinline__ u64 sqr(u64 a) { return mul(a, a); }

// x * 2^E for 0 < E < 64, x any u64: x << E is (lo, hi) with hi < 2^E.
template <int E>
__device__ __forceinline__ u64 shl(u64 x) {
  static_assert(E > 0 && E < 64, "shift out of range");
  const u64 lo_ = x << E, hi_ = x >> (64 - E);
  if constexpr (E <= 32)
    return reduce2(lo_, (u32)hi_);
  else
    return reduce3(lo_, (u32)hi_, (u32)(hi_ >> 32));
}

// x * 2^-M for 0 < M <= 32, x any u64: with x = q 2^M + r,
// x 2^-M = q + r 2^(192-M) = q - (r 2^(32-M)) 2^64 = q - (r 2^(32-M)) (2^32 - 1),
// where q < 2^(64-M) < p and the subtrahend <= (2^32 - 1)^2 < p.
template <int M>
__device__ __forceinline__ u64 shr(u64 x) {
  static_assert(M > 0 && M <= 32, "shift out of range");
  const u64 q = x >> M;
  const u32 r = M == 32 ? (u32)x : (u32)x << (32 - M);
  u64 dead;
  return sub(q, isa::mad_eps(r, 0, dead));
}

// x * 2^E for a compile-time E in [0, 192); x any u64, result canonical.  Uses 2^96 = -1 and, for
// 64 <= E < 96, 2^E = -2^-(96-E).  `negate` reports a sign the caller must apply.
template <int E>
__device__ __forceinline__ u64 mul_pow2_signed(u64 x, bool &negate) {
  static_assert(E >= 0 && E < 192, "shift exponent out of range");
  constexpr int F = E % 96;
  constexpr bool s1 = E >= 96;
  if constexpr (F == 0) {
    negate = s1;
    return x;
  } else if constexpr (F < 64) {
    negate = s1;
    return shl<F>(x);
  } else {
    negate = !s1;
    return shr<96 - F>(x);
  }
}

template <int E>
__device__ __forceinline__ u64 mul_pow2(u64 x) {
  bool negate;
  const u64 y = mul_pow2_signed<E>(x, negate);
  return negate ? neg(y) : y;
}

// Generic runtime a^e, for tests and set-up code.
__device__ __forceinline__ u64 pow_u64(u64 a, u64 e) {
  u64 r = 1;
  while (e) {
    if (e & 1) r = mul(r, a);
    a = sqr(a);
    e >>= 1;
  }
  return r;
}

// a^(2^K), lazy
template <int K>
__device__ __forceinline__ u64 sqr_times(u64 a) {
#pragma unroll 1
  for (int i = 0; i < K; i++) a = mul_lazy(a, a);
  return a;
}

// a^-1 = a^(p-2) (0 maps to 0), a any u64; result canonical.  With e_k = a^(2^k - 1):
// p - 2 = (2^31 - 1) 2^33 + 2^32 - 1, so the inverse is e_31^(2^33) e_32: 64 squarings and 9
// products (126 by binary exponentiation).
__device__ __forceinline__ u64 inv(u64 a) {
  const u64 e2 = mul_lazy(mul_lazy(a, a), a), e3 = mul_lazy(mul_lazy(e2, e2), a);
  const u64 e6 = mul_lazy(sqr_times<3>(e3), e3), e12 = mul_lazy(sqr_times<6>(e6), e6);
  const u64 e24 = mul_lazy(sqr_times<12>(e12), e12), e30 = mul_lazy(sqr_times<6>(e24), e6);
  const u64 e31 = mul_lazy(mul_lazy(e30, e30), a), e32 = mul_lazy(mul_lazy(e31, e31), a);
  return mul(sqr_times<33>(e31), e32);
}

// l + h 2^32 as a lazy residue, for l, h < 2^62: with h = h0 + h1 2^32 the value is
// l + h0 2^32 + h1 EPS < 2^64 + 2^63, so it overflows at most once, and adding EPS for that
// overflow does not wrap.  4 VALU.
__device__ __forceinline__ u64 fold_words(u64 l, u64 h) {
  using namespace isa;
  u64 c1, c2, dead;
  const u32 s = add_co(hi(l), lo(h), c1);
  const u64 r = mad_eps(hi(h), pack(lo(l), s), c2);
  return mad_eps(one_if(c1 | c2), r, dead);
}

}  // namespace gl
