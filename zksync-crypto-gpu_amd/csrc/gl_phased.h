// gl_phased.h -- the NTT passes' field arithmetic in phases, for interleaving independent
// operations.
//
// A product, a DIT butterfly and a DIF butterfly are each split into a fixed sequence of
// phases (one to three single-instruction steps each, from gl_field.h's isa namespace).  A
// batch of independent operations runs phase 0 of every member, then phase 1 of every member,
// and so on, so the instructions of different operations alternate: the wait states a
// VALU-written carry needs before it is read, and the latency of each dependent step, are
// filled with other operations' work instead of idle issue slots.  The arithmetic, and so every
// result, is exactly gl::mul / gl::add / gl::sub / gl::mul_pow2_signed's.
#pragma once

#include <utility>

#include "gl_field.h"

namespace gl {
namespace ph {

// Operations interleaved at once (the rest of a batch follows in further groups): enough to
// fill the carry wait states, few enough that their temporaries fit the registers.
#ifndef BA_ILP
#define BA_ILP 4
#endif
constexpr int ILP = BA_ILP;

template <typename F, int... I>
__device__ __forceinline__ void sfor_impl(F &&f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void sfor(F &&f) {
  sfor_impl(f, std::make_integer_sequence<int, N>{});
}

// ---------------------------------------------------------------- product (canonical result)
struct Mul {
  u64 a, b, r;
  u64 z, y, w, R, cy, k1, k2, c, b1, bw, m, k;
  u32 r1, r2, r3, t0, t1, one;
};
constexpr int MUL_PHASES = 12;

// phase P of gl::mul(s.a, s.b) -> s.r (LAZY: gl::mul_lazy)
template <int P, bool LAZY = false>
__device__ __forceinline__ void mul_phase(Mul &s) {
  using namespace isa;
  if constexpr (P == 0) {
    s.z = mul32(lo(s.a), lo(s.b));
    s.y = mul32(hi(s.a), lo(s.b));
  } else if constexpr (P == 1) {
    s.y = mad(lo(s.a), hi(s.b), s.y, s.cy);
    s.w = mul32(hi(s.a), hi(s.b));
  } else if constexpr (P == 2) {
    s.r1 = add_co(hi(s.z), lo(s.y), s.k1);
  } else if constexpr (P == 3) {
    s.r2 = addc(lo(s.w), hi(s.y), s.k1, s.k2);
  } else if constexpr (P == 4) {
    s.r3 = addc0(hi(s.w), s.k2);
  } else if constexpr (P == 5) {
    s.t0 = subb(lo(s.z), s.r3, s.cy, s.b1);
  } else if constexpr (P == 6) {
    s.t1 = subb0(s.r1, s.b1, s.bw);
  } else if constexpr (P == 7) {
    s.t0 = addc0(s.t0, s.bw, s.k);
  } else if constexpr (P == 8) {
    s.t1 = subb0(s.t1, s.bw & ~s.k);
  } else if constexpr (P == 9) {
    s.R = mad_eps(s.r2, pack(s.t0, s.t1), s.c);
  } else if constexpr (P == 10) {
    s.one = one_if(LAZY ? s.c : s.c | ge_p(s.R));
  } else if constexpr (P == 11) {
    s.r = (u64)s.one * (u32)EPS + s.R;
  }
}

// For i < N (compile-time): x(i) *= y(i), where x(ic) returns a reference to the operand and
// y(ic) its multiplier (ic: std::integral_constant<int, i>), interleaved ILP at a time; the first
// LAZY products are lazy.
template <int N, int LAZY = 0, typename X, typename Y>
__device__ __forceinline__ void mul_batch(X &&x, Y &&y) {
  constexpr int GROUPS = (N + ILP - 1) / ILP;
  sfor<GROUPS>([&](auto g_) {
    constexpr int g = decltype(g_)::value;
    constexpr int M = (g + 1) * ILP <= N ? ILP : N - g * ILP;
    Mul st[M];
    sfor<M>([&](auto j_) {
      constexpr int j = decltype(j_)::value;
      st[j].a = x(std::integral_constant<int, g * ILP + j>{});
      st[j].b = y(std::integral_constant<int, g * ILP + j>{});
    });
    sfor<MUL_PHASES>([&](auto p_) {
      sfor<M>([&](auto j_) {
        constexpr int j = decltype(j_)::value;
        mul_phase<decltype(p_)::value, (g * ILP + j < LAZY)>(st[j]);
      });
    });
    sfor<M>([&](auto j_) {
      constexpr int j = decltype(j_)::value;
      x(std::integral_constant<int, g * ILP + j>{}) = st[j].r;
    });
  });
}

// ---------------------------------------------------------------- shift by 2^F, canonical result
// The three forms of gl::shl / gl::shr (x any u64):
//   F in (0, 32]:  x << F = lo + hl 2^64 -> reduce2                          4 phases
//   F in (32, 64): x << F = lo + (hl + hh 2^32) 2^64 -> reduce3              8 phases
//   F in [64, 96): 2^F = -2^-(96-F): x 2^-M = q - r 2^(32-M) EPS, M = 96 - F  6 phases
constexpr int shift_phases(int F) { return F == 0 ? 0 : F <= 32 ? 4 : F < 64 ? 8 : 6; }

struct Shift {
  u64 x, t;  // in, out
  u64 lo, R, c, b1, bw, k, q, u;
  u32 hl, hh, d0, d1, t0, r, one;
};

template <int F, int P>
__device__ __forceinline__ void shift_phase(Shift &s) {
  using namespace isa;
  if constexpr (F == 0) {
    if constexpr (P == 0) s.t = s.x;  // (a zero-length form: never called with P >= 0 in a batch)
  } else if constexpr (F <= 32) {
    if constexpr (P == 0) {
      s.lo = s.x << F;
      s.hl = (u32)(s.x >> (64 - F));
    } else if constexpr (P == 1) {
      s.R = mad_eps(s.hl, s.lo, s.c);
    } else if constexpr (P == 2) {
      s.one = one_if(s.c | ge_p(s.R));
    } else if constexpr (P == 3) {
      s.t = (u64)s.one * (u32)EPS + s.R;
    }
  } else if constexpr (F < 64) {
    if constexpr (P == 0) {
      s.lo = s.x << F;
      const u64 h = s.x >> (64 - F);
      s.hl = (u32)h;
      s.hh = (u32)(h >> 32);
    } else if constexpr (P == 1) {
      s.d0 = sub_co(isa::lo(s.lo), s.hh, s.b1);
    } else if constexpr (P == 2) {
      s.d1 = subb0(isa::hi(s.lo), s.b1, s.bw);
    } else if constexpr (P == 3) {
      s.d0 = addc0(s.d0, s.bw, s.k);
    } else if constexpr (P == 4) {
      s.d1 = subb0(s.d1, s.bw & ~s.k);
    } else if constexpr (P == 5) {
      s.R = mad_eps(s.hl, pack(s.d0, s.d1), s.c);
    } else if constexpr (P == 6) {
      s.one = one_if(s.c | ge_p(s.R));
    } else if constexpr (P == 7) {
      s.t = (u64)s.one * (u32)EPS + s.R;
    }
  } else {
    constexpr int M = 96 - F;
    if constexpr (P == 0) {
      s.q = s.x >> M;
      s.r = M == 32 ? (u32)s.x : (u32)s.x << (32 - M);
    } else if constexpr (P == 1) {
      s.u = mad_eps(s.r, 0, s.k);
    } else if constexpr (P == 2) {
      s.d0 = sub_co(lo(s.q), lo(s.u), s.c);
    } else if constexpr (P == 3) {
      s.d1 = subb(hi(s.q), hi(s.u), s.c, s.bw);
    } else if constexpr (P == 4) {
      s.t0 = addc0(s.d0, s.bw, s.k);
    } else if constexpr (P == 5) {
      s.t = pack(s.t0, subb0(s.d1, s.bw & ~s.k));
    }
  }
}

// ---------------------------------------------------------------- add and subtract
// (s, d) = (a + b, a - b), canonical, from canonical a, b: 4 phases.  LAZY: a any u64, b canonical,
// s and d lazy residues (gl::add_lazy, gl::sub).
struct AddSub {
  u64 a, b, s, d;
  u64 cs, c2, cd, bw, kd;
  u32 s0, s1, d0, d1, one;
};
constexpr int ADDSUB_PHASES = 4;

template <int P, bool LAZY = false>
__device__ __forceinline__ void addsub_phase(AddSub &s) {
  using namespace isa;
  if constexpr (P == 0) {
    s.s0 = add_co(lo(s.a), lo(s.b), s.cs);
    s.d0 = sub_co(lo(s.a), lo(s.b), s.cd);
  } else if constexpr (P == 1) {
    s.s1 = addc(hi(s.a), hi(s.b), s.cs, s.c2);
    s.d1 = subb(hi(s.a), hi(s.b), s.cd, s.bw);
  } else if constexpr (P == 2) {
    s.one = one_if(LAZY ? s.c2 : s.c2 | ge_p(pack(s.s0, s.s1)));
    s.d0 = addc0(s.d0, s.bw, s.kd);
  } else if constexpr (P == 3) {
    s.s = (u64)s.one * (u32)EPS + pack(s.s0, s.s1);
    s.d = pack(s.d0, subb0(s.d1, s.bw & ~s.kd));
  }
}

// ---------------------------------------------------------------- butterflies
// DIT: (a, b) <- (a + 2^E b, a - 2^E b): the shift, then add/sub; a negative factor (2^96 = -1,
// 2^F = -2^-(96-F) for 64 <= F < 96) swaps the sum and the difference.
// DIF: (a, b) <- (a + b, 2^E (a - b)), the sign folded into the order of the subtraction.
template <int E>
struct PowForm {
  static constexpr int F = E % 96;
  static constexpr bool NEG = F == 0 ? E >= 96 : (F < 64 ? E >= 96 : E < 96);
  static constexpr int SP = shift_phases(F);
};

// a, b: the butterfly's operands in, its results out
struct Bfly {
  u64 a, b;
  Shift sh;
  AddSub as;
};

// LAZY: a any u64, results lazy; b canonical, or any u64 where a shift or REDUCE (E = 0: gl::reduce1, 2
// phases) makes it canonical first.
constexpr int dit_pre_phases(int E, bool reduce) { return shift_phases(E % 96) + (reduce ? 2 : 0); }

template <int E, int P, bool LAZY, bool REDUCE>
__device__ __forceinline__ void dit_phase(Bfly &s) {
  using Fm = PowForm<E>;
  static_assert(!REDUCE || Fm::SP == 0, "a shift makes its result canonical");
  constexpr int SP = dit_pre_phases(E, REDUCE);
  if constexpr (P == 0) s.sh.x = s.b, s.as.a = s.a;
  if constexpr (REDUCE && P == 0) s.sh.one = isa::one_if(isa::ge_p(s.sh.x));
  if constexpr (REDUCE && P == 1) s.sh.x = (u64)s.sh.one * (u32)EPS + s.sh.x;
  if constexpr (!REDUCE && P < SP) shift_phase<Fm::F, P>(s.sh);
  if constexpr (P == SP) s.as.b = Fm::SP ? s.sh.t : s.sh.x;
  if constexpr (P >= SP && P < SP + ADDSUB_PHASES) addsub_phase<P - SP, LAZY>(s.as);
  if constexpr (P == SP + ADDSUB_PHASES - 1) {
    s.a = Fm::NEG ? s.as.d : s.as.s;
    s.b = Fm::NEG ? s.as.s : s.as.d;
  }
}

template <int E, int P>
__device__ __forceinline__ void dif_phase(Bfly &s) {
  using Fm = PowForm<E>;
  if constexpr (P == 0) {
    // 2^E (a - b) = +-2^F' (a - b): the sign the shift form carries is folded into the order
    s.as.a = Fm::NEG ? s.b : s.a;
    s.as.b = Fm::NEG ? s.a : s.b;
  }
  if constexpr (P < ADDSUB_PHASES) addsub_phase<P>(s.as);
  if constexpr (P == ADDSUB_PHASES - 1) {
    s.a = s.as.s;  // a + b either way
    s.sh.x = s.as.d;
    if constexpr (Fm::SP == 0) s.b = s.as.d;
  }
  if constexpr (P >= ADDSUB_PHASES && P < ADDSUB_PHASES + Fm::SP) shift_phase<Fm::F, P - ADDSUB_PHASES>(s.sh);
  if constexpr (Fm::SP > 0 && P == ADDSUB_PHASES + Fm::SP - 1) s.b = s.sh.t;
}
template <int E>
constexpr int dif_phases() {
  return ADDSUB_PHASES + PowForm<E>::SP;
}

}  // namespace ph
}  // namespace gl
