// poseidon2.hip -- Poseidon2 over Goldilocks, width 12 (rate 8, capacity 4): the Merkle leaf
// and node hashes that consume LDE cosets.
//
// Entry points mirror boojum_cuda::poseidon2::GpuTreeHasher for the Goldilocks hasher
// (crates/boojum-cuda/src/poseidon2.rs:165-316: compute_leaf_hashes, compute_node_hashes,
// build_merkle_tree_leaves, build_merkle_tree_nodes, build_merkle_tree) with the same slice
// lengths, layouts and preconditions (violations return BA_ERROR_INVALID_VALUE instead of
// panicking).  The permutation is the Poseidon2 paper's (eprint 2023/323, Fig. 1 and Appendix B)
// for the instance the reference runs (crates/boojum-cuda/native/poseidon2/gl/poseidon2_gl_st.cu:9-22,
// poseidon2_gl_constants.cuh.template): external matrix M_E = circ(2 M4, M4, M4) first; 4 full
// rounds; 22 partial rounds with M_I = J + diag(2^mu); 4 full rounds; S-box x^7.  Its 30 x 12
// round constants come from boojum (poseidon_goldilocks_params), which the reference tree does
// not hold: a caller installs them once per context with ba_poseidon2_gl_set_round_constants.
//
// What bounds it: VALU issue, ~9.9 k instructions per permutation against 64 bytes of input, the
// digests being independent.  The state stays lazy (any u64 residue) between layers, see below:
// 2^20 leaves of 64 values take 2.23 ms (3.8 G permutations/s), where canonical lanes at 16.2 k
// instructions took 3.0 ms.  Three kernels share the arithmetic: one thread per digest with all 12
// lanes in registers (throughput), a quad of threads per digest (latency, few digests), and 16 threads
// per digest (latency, fewest), chosen by the digest count (QUAD_MAX, ROW_MAX below).
#include <utility>
#include <vector>

#include "api_internal.h"
#include "gl_field.h"

namespace {

using gl::u32;
using gl::u64;

constexpr int WIDTH = 12, RATE = 8, CAPACITY = 4;
constexpr int HALF_FULL_ROUNDS = 4, PARTIAL_ROUNDS = 22, ROUNDS = 2 * HALF_FULL_ROUNDS + PARTIAL_ROUNDS;
constexpr int THREADS = 256;
constexpr int QUADS = THREADS / 4;
// Digest count up to which a launch takes the quad kernels.  A thread's chain alone takes ~39 us
// per permutation whatever the count, until 2^17 digests give every SIMD two waves; a quad's takes
// 18 us and does 1.7 times the work.  Node hashes, thread / quad, us: 2^10 39 / 18, 2^15 39 / 24,
// 2^16 40 / 40, 2^16.6 47 / 61, 2^18 87 / 128.
constexpr u32 QUAD_MAX = 65536;
// Below that, up to which count 16 threads take a digest: a row's chain is 11.5 us, which two waves per
// SIMD (2^13 digests) still nearly hide.  Node hashes, quad / row, us: 2^4 18.1 / 11.4, 2^10 18.6 /
// 11.6, 2^12 18.9 / 12.2, 2^13 19.3 / 16.0, 2^14 20.0 / 25.8, 2^16 40 / 84.
constexpr u32 ROW_MAX = 8192;

// Lazy arithmetic: state lanes are any u64 (a residue mod p, not reduced below it).  gl::mul_lazy
// takes and returns such values; the linear layers take a value's two words into two 64-bit
// accumulators ("planes": value = l + h 2^32), where adding a word times a small factor is one
// v_mad_u64_u32 without carries, and fold each output back once.  Digests are reduced below p when
// they are stored.
struct Planes {
  u64 l, h;
};

// word * f + acc (no carry out: the planes stay below 2^62)
__device__ __forceinline__ u64 mac(u32 word, u32 f, u64 acc) {
  u64 dead;
  return gl::isa::mad(word, f, acc, dead);
}
template <int F>
__device__ __forceinline__ u64 mac_const(u32 word, u64 acc) {
  u64 r, dead;
  if constexpr (F <= 64)
    asm("v_mad_u64_u32 %0, %1, %2, %3, %4" : "=v"(r), "=s"(dead) : "v"(word), "n"(F), "v"(acc));
  else
    asm("v_mad_u64_u32 %0, %1, %2, %3, %4" : "=v"(r), "=s"(dead) : "v"(word), "s"(F), "v"(acc));
  return r;
}
// the word itself as a plane
__device__ __forceinline__ u64 plane(u32 word) {
  u64 r, dead;
  asm("v_mad_u64_u32 %0, %1, %2, 1, 0" : "=v"(r), "=s"(dead) : "v"(word));
  return r;
}
// word in a scalar register + acc
__device__ __forceinline__ u64 plus_scalar(u32 word, u64 acc) {
  u64 r, dead;
  asm("v_mad_u64_u32 %0, %1, %2, 1, %3" : "=v"(r), "=s"(dead) : "s"(word), "v"(acc));
  return r;
}
// a 2^K + b, K <= 4
template <int K>
__device__ __forceinline__ u64 shl_add(u64 a, u64 b) {
  u64 r;
  asm("v_lshl_add_u64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "n"(K), "v"(b));
  return r;
}
__device__ __forceinline__ Planes operator+(const Planes &a, const Planes &b) {
  return {shl_add<0>(a.l, b.l), shl_add<0>(a.h, b.h)};
}
__device__ __forceinline__ u64 folded(const Planes &v) { return gl::fold_words(v.l, v.h); }

// M4 of Appendix B, [[5,7,1,3],[4,6,1,1],[1,3,5,7],[1,1,4,6]], as an addition chain on one plane
__device__ __forceinline__ void m4(u64 (&x)[4]) {
  const u64 a = shl_add<0>(x[0], x[1]), b = shl_add<0>(x[2], x[3]);
  const u64 c = shl_add<1>(x[1], b);  // 2 x1 + x2 + x3
  const u64 d = shl_add<1>(x[3], a);  // x0 + x1 + 2 x3
  x[3] = shl_add<2>(b, d);            // x0 + x1 + 4 x2 + 6 x3
  x[1] = shl_add<2>(a, c);            // 4 x0 + 6 x1 + x2 + x3
  x[0] = shl_add<0>(d, x[1]);
  x[2] = shl_add<0>(c, x[3]);
}

// M_E = circ(2 M4, M4, M4): every lane plus the sum of its position over the tiles, then M4 on each
// tile; plus the next round's constants rc[0..12).  Planes stay below 65 * 2^32.  LAST: the layer
// after the last round, which adds nothing and whose lanes 4..7 nobody reads (a digest is lanes
// 0..3, the next chunk keeps lanes 8..11).
template <bool LAST>
__device__ __forceinline__ void external_layer(u64 (&s)[WIDTH], const u64 *__restrict__ rc) {
  using namespace gl::isa;
  u64 sl[4], sh[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    sl[j] = mac_const<1>(lo(s[8 + j]), mac_const<1>(lo(s[4 + j]), plane(lo(s[j]))));
    sh[j] = mac_const<1>(hi(s[8 + j]), mac_const<1>(hi(s[4 + j]), plane(hi(s[j]))));
  }
#pragma unroll
  for (int t = 0; t < 3; t++) {
    if (LAST && t == 1) continue;
    u64 l[4], h[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      l[j] = mac_const<1>(lo(s[4 * t + j]), sl[j]);
      h[j] = mac_const<1>(hi(s[4 * t + j]), sh[j]);
    }
    m4(l);
    m4(h);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      if (!LAST) {
        const u64 k = rc[4 * t + j];
        l[j] = plus_scalar(lo(k), l[j]);
        h[j] = plus_scalar(hi(k), h[j]);
      }
      s[4 * t + j] = folded({l[j], h[j]});
    }
  }
}

// M_I = J + diag(2^mu)
constexpr int MU[WIDTH] = {4, 14, 11, 8, 0, 5, 2, 9, 13, 6, 3, 12};

// f(i) for i = 1..11 as constants
template <int I = 1, typename F>
__device__ __forceinline__ void for_lanes(F &&f) {
  f(std::integral_constant<int, I>{});
  if constexpr (I + 1 < WIDTH) for_lanes<I + 1>(f);
}

__device__ __forceinline__ u64 sbox(u64 x) {
  const u64 x2 = gl::mul_lazy(x, x), x3 = gl::mul_lazy(x, x2), x4 = gl::mul_lazy(x2, x2);
  return gl::mul_lazy(x3, x4);
}

// Two partial rounds.  Lanes 1..11 are linear in both, so they are folded once for the pair: with
// x, y the two S-box outputs, S = x + sum_i s_i the first round's sum and d_i = 2^mu_i,
//   lane i after two rounds = d_i^2 s_i + d_i S + (y + 11 S + sum_i d_i s_i),   i = 1..11.
// Planes stay below 2^60 + 2^47.  270 VALU, against 308 for two rounds one after the other.
// rc: the constants on lane 0 after each of the two.
__device__ __forceinline__ void partial_pair(u64 (&s)[WIDTH], u64 rc_first, u64 rc_second) {
  using namespace gl::isa;
  const u64 x = sbox(s[0]);
  Planes sum{plane(lo(x)), plane(hi(x))}, weighted{0, 0};
  for_lanes([&](auto i_) {
    constexpr int i = decltype(i_)::value;
    sum = {mac_const<1>(lo(s[i]), sum.l), mac_const<1>(hi(s[i]), sum.h)};
    weighted = {mac_const<1 << MU[i]>(lo(s[i]), weighted.l), mac_const<1 << MU[i]>(hi(s[i]), weighted.h)};
  });
  const u64 S = folded(sum);
  const u64 y = sbox(folded({plus_scalar(lo(rc_first), mac_const<1 << MU[0]>(lo(x), sum.l)),
                             plus_scalar(hi(rc_first), mac_const<1 << MU[0]>(hi(x), sum.h))}));
  const Planes second{mac_const<1>(lo(y), mac_const<WIDTH - 1>(lo(S), weighted.l)),
                      mac_const<1>(hi(y), mac_const<WIDTH - 1>(hi(S), weighted.h))};
  for_lanes([&](auto i_) {
    constexpr int i = decltype(i_)::value, D = 1 << MU[i];
    s[i] = folded({mac_const<D * D>(lo(s[i]), mac_const<D>(lo(S), second.l)),
                   mac_const<D * D>(hi(s[i]), mac_const<D>(hi(S), second.h))});
  });
  s[0] = folded({plus_scalar(lo(rc_second), mac_const<1 << MU[0]>(lo(y), second.l)),
                 plus_scalar(hi(rc_second), mac_const<1 << MU[0]>(hi(y), second.h))});
}

// rc: the device table of round constants (30 + 1 rows, see ba_poseidon2_gl_set_round_constants).
// Each layer adds the constants of the round after it.  The loops keep the code at three round
// bodies (20 KB, inside the instruction cache, where 30 unrolled rounds are 130 KB).
__device__ __forceinline__ void permute(u64 (&s)[WIDTH], const u64 *__restrict__ rc) {
  auto sboxes = [&]() {
#pragma unroll
    for (int i = 0; i < WIDTH; i++) s[i] = sbox(s[i]);
  };
  const u64 *row = rc;
  external_layer<false>(s, row);
#pragma unroll 1
  for (int r = 0; r < ROUNDS - PARTIAL_ROUNDS - 1; r++) {
    row += WIDTH;
    sboxes();
    external_layer<false>(s, row);
    if (r + 1 == HALF_FULL_ROUNDS) {
#pragma unroll 1
      for (int k = 0; k < PARTIAL_ROUNDS / 2; k++) {
        partial_pair(s, row[WIDTH], row[2 * WIDTH]);
        row += 2 * WIDTH;
      }
      // the first full round's other constants
#pragma unroll
      for (int i = 1; i < WIDTH; i++) s[i] = gl::add_lazy(s[i], row[i]);
    }
  }
  sboxes();
  external_layer<true>(s, row);
}

// ---------------------------------------------------------------- one quad of threads per digest
// Thread j of a quad holds lanes j, 4 + j and 8 + j (position j of each tile): the sums over tiles
// are its own, M4 and the sum over all lanes are quad permutations.  A permutation is then a chain
// of ~4.2 k instructions instead of ~9.9 k, for 1.7 times the work in all.
struct Quad {
  u32 j;       // position in the quad
  u32 m4[4];   // M4[j][(j + k) mod 4]
  u32 mu[3];   // 2^mu of lanes j, 4 + j, 8 + j
};

template <int CTRL>
__device__ __forceinline__ u32 quad_perm(u32 x) {
  return (u32)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xF, 0xF, true);
}
constexpr int NEXT1 = 0x39, NEXT2 = 0x4E, NEXT3 = 0x93, SWAP1 = 0xB1;  // thread j reads j + 1, + 2, + 3, j ^ 1

__device__ __forceinline__ Quad quad_of(u32 j) {
  // rows of M4 rotated to start at the diagonal, 4 bits per entry; mu, 4 bits per tile
  const u32 rows = j == 0 ? 0x3175u : j == 1 ? 0x4116u : j == 2 ? 0x3175u : 0x4116u;
  const u32 mus = j == 0 ? 0xD04u : j == 1 ? 0x65Eu : j == 2 ? 0x32Bu : 0xC98u;
  Quad q;
  q.j = j;
#pragma unroll
  for (int k = 0; k < 4; k++) q.m4[k] = (rows >> (4 * k)) & 15u;
#pragma unroll
  for (int t = 0; t < 3; t++) q.mu[t] = 1u << ((mus >> (4 * t)) & 15u);
  return q;
}

// rc: this thread's three constants
__device__ __forceinline__ void quad_external(u64 (&s)[3], const Quad &q, const u64 (&rc)[3]) {
  using namespace gl::isa;
  Planes m[3];
#pragma unroll
  for (int t = 0; t < 3; t++) {
    const u32 l = lo(s[t]), h = hi(s[t]);
    m[t] = {mul32(l, q.m4[0]), mul32(h, q.m4[0])};
    m[t] = {mac(quad_perm<NEXT1>(l), q.m4[1], m[t].l), mac(quad_perm<NEXT1>(h), q.m4[1], m[t].h)};
    m[t] = {mac(quad_perm<NEXT2>(l), q.m4[2], m[t].l), mac(quad_perm<NEXT2>(h), q.m4[2], m[t].h)};
    m[t] = {mac(quad_perm<NEXT3>(l), q.m4[3], m[t].l), mac(quad_perm<NEXT3>(h), q.m4[3], m[t].h)};
  }
  const Planes sum = m[0] + m[1] + m[2];
#pragma unroll
  for (int t = 0; t < 3; t++) {
    const Planes v = m[t] + sum;
    s[t] = folded({mac_const<1>(lo(rc[t]), v.l), mac_const<1>(hi(rc[t]), v.h)});
  }
}

// rc0: the next round's lane-0 constant in thread 0, 0 in the others
__device__ __forceinline__ void quad_internal(u64 (&s)[3], const Quad &q, u64 rc0) {
  using namespace gl::isa;
  Planes sum{plane(lo(s[0])), plane(hi(s[0]))};
#pragma unroll
  for (int t = 1; t < 3; t++) sum = {mac_const<1>(lo(s[t]), sum.l), mac_const<1>(hi(s[t]), sum.h)};
  auto across = [](u64 x, auto perm) { return shl_add<0>(x, pack(perm(lo(x)), perm(hi(x)))); };
  auto one = [](u32 w) { return quad_perm<SWAP1>(w); };
  auto two = [](u32 w) { return quad_perm<NEXT2>(w); };
  sum = {across(across(sum.l, one), two), across(across(sum.h, one), two)};
  const Planes first{mac_const<1>(lo(rc0), sum.l), mac_const<1>(hi(rc0), sum.h)};
#pragma unroll
  for (int t = 0; t < 3; t++) {
    const Planes &base = t == 0 ? first : sum;
    s[t] = folded({mac(lo(s[t]), q.mu[t], base.l), mac(hi(s[t]), q.mu[t], base.h)});
  }
}

__device__ __forceinline__ void quad_permute(u64 (&s)[3], const Quad &q, const u64 *__restrict__ rc) {
  // each round's constants are loaded one round ahead
  const u64 *row = rc + q.j;
  u64 k[3] = {row[0], row[4], row[8]};
  auto step = [&]() {
    row += WIDTH;
    k[0] = row[0], k[1] = row[4], k[2] = row[8];
  };
  {
    const u64 k0[3] = {k[0], k[1], k[2]};
    step();
    quad_external(s, q, k0);
  }
#pragma unroll 1
  for (int half = 0; half < 2; half++) {
#pragma unroll 1
    for (int r = 0; r < HALF_FULL_ROUNDS; r++) {
      const u64 kr[3] = {k[0], k[1], k[2]};
      if (!(half && r + 1 == HALF_FULL_ROUNDS)) step();
#pragma unroll
      for (int t = 0; t < 3; t++) s[t] = sbox(s[t]);
      quad_external(s, q, kr);
    }
    if (half) break;
#pragma unroll 1
    for (int r = 0; r < PARTIAL_ROUNDS; r++) {
      const u64 kr[3] = {k[0], k[1], k[2]};
      step();
      const u64 x = sbox(s[0]);
      if (q.j == 0) s[0] = x;
      quad_internal(s, q, r + 1 == PARTIAL_ROUNDS && q.j ? 0 : kr[0]);
      if (r + 1 == PARTIAL_ROUNDS) {  // the first full round's other constants
        if (q.j) s[0] = gl::add_lazy(s[0], kr[0]);
        s[1] = gl::add_lazy(s[1], kr[1]);
        s[2] = gl::add_lazy(s[2], kr[2]);
      }
    }
  }
}

// ---------------------------------------------------------------- 16 threads per digest
// Thread i < 12 of a row of 16 holds lane i; the last four only keep the row sums whole.  Sums over
// tiles and over all lanes are DPP row rotations.  A permutation is a chain of ~2.7 k instructions, for
// 2.6 times the quad's work in all.
struct Row {
  u32 lane;
  u32 m4[4];  // M4[j][(j + k) mod 4], j the position in the tile; 0 in idle threads
  u32 mu;     // 2^mu of the lane; 0 in idle threads
  u32 mask;   // the lane's low 21 bits, nothing in idle threads
  u32 width;  // 22, 0 in idle threads
};

template <int N>
__device__ __forceinline__ u32 row_ror(u32 x) {
  return (u32)__builtin_amdgcn_update_dpp(0, (int)x, 0x120 + N, 0xF, 0xF, true);
}

__device__ __forceinline__ Row row_of(u32 lane) {
  const bool live = lane < WIDTH;
  const u32 rows = !live ? 0 : lane & 1 ? 0x4116u : 0x3175u;
  constexpr u64 MUS = 0xC36D'9250'8BE4ull;  // mu, 4 bits per lane
  Row q;
  q.lane = lane;
#pragma unroll
  for (int k = 0; k < 4; k++) q.m4[k] = (rows >> (4 * k)) & 15u;
  q.mu = live ? 1u << ((u32)(MUS >> (4 * lane)) & 15u) : 0;
  q.mask = live ? 0x1FFFFFu : 0;
  q.width = live ? 22 : 0;
  return q;
}

__device__ __forceinline__ u64 row_external(u64 s, const Row &q, u64 rc) {
  using namespace gl::isa;
  const u32 l = lo(s), h = hi(s);
  Planes m{mul32(l, q.m4[0]), mul32(h, q.m4[0])};
  m = {mac(quad_perm<NEXT1>(l), q.m4[1], m.l), mac(quad_perm<NEXT1>(h), q.m4[1], m.h)};
  m = {mac(quad_perm<NEXT2>(l), q.m4[2], m.l), mac(quad_perm<NEXT2>(h), q.m4[2], m.h)};
  m = {mac(quad_perm<NEXT3>(l), q.m4[3], m.l), mac(quad_perm<NEXT3>(h), q.m4[3], m.h)};
  auto across = [](u64 x, auto ror) { return shl_add<0>(x, pack(ror(lo(x)), ror(hi(x)))); };
  auto eight = [](u32 w) { return row_ror<8>(w); };
  auto four = [](u32 w) { return row_ror<4>(w); };
  const Planes sum{across(across(m.l, eight), four), across(across(m.h, eight), four)};
  const Planes v = m + sum;
  return folded({mac_const<1>(lo(rc), v.l), mac_const<1>(hi(rc), v.h)});
}

// The sum over the row runs on three 21/22-bit limbs, whose 16 values stay inside a word: a step is
// three 32-bit additions instead of two 64-bit ones with two moves each.  rc: 0 outside lane 0, but
// after the last partial round
__device__ __forceinline__ u64 row_internal(u64 s, const Row &q, u64 rc) {
  using namespace gl::isa;
  u32 a = lo(s) & q.mask;
  u32 b = __builtin_amdgcn_alignbit(hi(s), lo(s), 21) & q.mask;
  u32 c = __builtin_amdgcn_ubfe(hi(s), 10, q.width);
  a += row_ror<8>(a), b += row_ror<8>(b), c += row_ror<8>(c);
  a += row_ror<4>(a), b += row_ror<4>(b), c += row_ror<4>(c);
  a += row_ror<2>(a), b += row_ror<2>(b), c += row_ror<2>(c);
  a += row_ror<1>(a), b += row_ror<1>(b), c += row_ror<1>(c);
  // a + 2^21 b + 2^42 c: planes below 2^47 and 2^36
  const Planes sum{mac_const<1 << 21>(b, mac_const<1>(a, lo(rc))), mac_const<1 << 10>(c, hi(rc))};
  return folded({mac(lo(s), q.mu, sum.l), mac(hi(s), q.mu, sum.h)});
}

__device__ __forceinline__ u64 row_permute(u64 s, const Row &q, const u64 *__restrict__ rc) {
  // each round's constants are loaded one round ahead
  const u64 *row = rc + (q.lane < WIDTH ? q.lane : WIDTH - 1);
  u64 k = row[0], kr = k;
  auto step = [&]() {
    kr = k;
    row += WIDTH;
    k = row[0];
  };
  step();
  s = row_external(s, q, kr);
#pragma unroll 1
  for (int half = 0; half < 2; half++) {
#pragma unroll 1
    for (int r = 0; r < HALF_FULL_ROUNDS; r++) {
      kr = k;
      if (!(half && r + 1 == HALF_FULL_ROUNDS)) step();
      s = row_external(sbox(s), q, kr);
    }
    if (half) break;
#pragma unroll 1
    for (int r = 0; r < PARTIAL_ROUNDS; r++) {
      step();
      const u64 x = sbox(s);
      s = row_internal(q.lane == 0 ? x : s, q, kr);
    }
  }
  return s;
}

// Leaf gid absorbs values[gid * rows + r + c * rows * count] (c < cols, r < rows, column by
// column) RATE at a time into lanes 0..7 (overwrite mode, zero-filled past the last value) and
// permutes after each chunk; digest word k goes to results[gid + k * count].
__global__ __launch_bounds__(THREADS) void leaves_kernel(const u64 *__restrict__ values, u64 *__restrict__ results,
                                                         u32 rows, u32 cols, u32 count, int load_intermediate,
                                                         int store_intermediate, const u64 *__restrict__ rc) {
  const u32 gid = blockIdx.x * THREADS + threadIdx.x;
  if (gid >= count) return;
  u64 s[WIDTH];
#pragma unroll
  for (int i = 0; i < WIDTH; i++) s[i] = 0;
  if (load_intermediate) {
#pragma unroll
    for (int k = 0; k < CAPACITY; k++) s[RATE + k] = results[gid + (u64)k * count];
  }
  const u64 *leaf = values + (u64)gid * rows;
  const u64 col_stride = (u64)rows * count;
  const u64 total = (u64)rows * cols;
  u32 r = 0;  // (row, column) of the next value, the same for every lane
  u64 c = 0;
  for (u64 off = 0; off < total; off += RATE) {
#pragma unroll
    for (int i = 0; i < RATE; i++) {
      s[i] = c < cols ? leaf[r + c * col_stride] : 0;
      if (++r == rows) r = 0, c++;
    }
    permute(s, rc);
  }
  const int from = store_intermediate ? RATE : 0;
#pragma unroll
  for (int k = 0; k < CAPACITY; k++) results[gid + (u64)k * count] = gl::reduce1(s[from + k]);
}

// Node gid hashes its children's digests: word k of the left child at values[2 (gid + k count)],
// of the right child at values[2 (gid + k count) + 1] (the layer below, read as word pairs).
__global__ __launch_bounds__(THREADS) void nodes_kernel(const u64 *__restrict__ values, u64 *__restrict__ results,
                                                        u32 count, const u64 *__restrict__ rc) {
  const u32 gid = blockIdx.x * THREADS + threadIdx.x;
  if (gid >= count) return;
  u64 s[WIDTH];
#pragma unroll
  for (int k = 0; k < CAPACITY; k++) {
    const u64 at = 2 * (gid + (u64)k * count);
    s[k] = values[at];
    s[CAPACITY + k] = values[at + 1];
  }
#pragma unroll
  for (int i = 2 * CAPACITY; i < WIDTH; i++) s[i] = 0;
  permute(s, rc);
#pragma unroll
  for (int k = 0; k < CAPACITY; k++) results[gid + (u64)k * count] = gl::reduce1(s[k]);
}

// The same two hashes by quads: thread j absorbs values j and 4 + j of each chunk, and holds word j
// of the digests.
__global__ __launch_bounds__(THREADS) void leaves_quad_kernel(const u64 *__restrict__ values,
                                                              u64 *__restrict__ results, u32 rows, u32 cols,
                                                              u32 count, int load_intermediate,
                                                              int store_intermediate, const u64 *__restrict__ rc) {
  const u32 gid = blockIdx.x * QUADS + (threadIdx.x >> 2);
  if (gid >= count) return;
  const Quad q = quad_of(threadIdx.x & 3);
  const u64 at = gid + (u64)q.j * count;
  u64 s[3] = {0, 0, load_intermediate ? results[at] : 0};
  const u64 *leaf = values + (u64)gid * rows;
  const u64 col_stride = (u64)rows * count;
  const u64 total = (u64)rows * cols;
  const u32 log_rows = 31 - __builtin_clz(rows);
  for (u64 off = 0; off < total; off += RATE) {
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const u64 v = off + 4 * t + q.j;
      s[t] = v < total ? leaf[(v & (rows - 1)) + (v >> log_rows) * col_stride] : 0;
    }
    quad_permute(s, q, rc);
  }
  results[at] = gl::reduce1(store_intermediate ? s[2] : s[0]);
}

__global__ __launch_bounds__(THREADS) void nodes_quad_kernel(const u64 *__restrict__ values,
                                                             u64 *__restrict__ results, u32 count,
                                                             const u64 *__restrict__ rc) {
  const u32 gid = blockIdx.x * QUADS + (threadIdx.x >> 2);
  if (gid >= count) return;
  const Quad q = quad_of(threadIdx.x & 3);
  const u64 at = gid + (u64)q.j * count;
  u64 s[3] = {values[2 * at], values[2 * at + 1], 0};
  quad_permute(s, q, rc);
  results[at] = gl::reduce1(s[0]);
}

// The same two hashes by rows: thread i < 8 absorbs value i of each chunk, thread i < 4 holds word i of
// a digest.
constexpr int DIGEST_ROWS = THREADS / 16;
__global__ __launch_bounds__(THREADS) void leaves_row_kernel(const u64 *__restrict__ values,
                                                             u64 *__restrict__ results, u32 rows, u32 cols,
                                                             u32 count, int load_intermediate,
                                                             int store_intermediate, const u64 *__restrict__ rc) {
  const u32 gid = blockIdx.x * DIGEST_ROWS + (threadIdx.x >> 4);
  if (gid >= count) return;
  const Row q = row_of(threadIdx.x & 15);
  u64 s = load_intermediate && q.lane >= RATE && q.lane < WIDTH ? results[gid + (u64)(q.lane - RATE) * count] : 0;
  const u64 *leaf = values + (u64)gid * rows;
  const u64 col_stride = (u64)rows * count;
  const u64 total = (u64)rows * cols;
  const u32 log_rows = 31 - __builtin_clz(rows);
  for (u64 off = 0; off < total; off += RATE) {
    const u64 v = off + q.lane;
    if (q.lane < RATE) s = v < total ? leaf[(v & (rows - 1)) + (v >> log_rows) * col_stride] : 0;
    s = row_permute(s, q, rc);
  }
  const u32 word = q.lane - (store_intermediate ? RATE : 0);
  if (word < CAPACITY) results[gid + (u64)word * count] = gl::reduce1(s);
}

__global__ __launch_bounds__(THREADS) void nodes_row_kernel(const u64 *__restrict__ values,
                                                            u64 *__restrict__ results, u32 count,
                                                            const u64 *__restrict__ rc) {
  const u32 gid = blockIdx.x * DIGEST_ROWS + (threadIdx.x >> 4);
  if (gid >= count) return;
  const Row q = row_of(threadIdx.x & 15);
  // word k of the left child in lane k, of the right child in lane 4 + k
  u64 s = q.lane < RATE ? values[2 * (gid + (u64)(q.lane & 3) * count) + (q.lane >> 2)] : 0;
  s = row_permute(s, q, rc);
  if (q.lane < CAPACITY) results[gid + (u64)q.lane * count] = gl::reduce1(s);
}

// The current device's context with installed round constants, or an error code.
int hasher_context(ba_context *&ctx) {
  ctx = ba_context_for_current_device();
  if (!ctx || !ctx->p2_round_constants) return BA_ERROR_NOT_INITIALIZED;
  return BA_SUCCESS;
}

u32 blocks_for(u64 count, u32 per_block) { return (u32)((count + per_block - 1) / per_block); }

int launch_nodes(const ba_context *ctx, const u64 *values, u64 *results, u32 count, hipStream_t stream) {
  if (count == 0) return BA_SUCCESS;
  if (count <= ROW_MAX)
    nodes_row_kernel<<<blocks_for(count, DIGEST_ROWS), THREADS, 0, stream>>>(values, results, count,
                                                                            ctx->p2_round_constants);
  else if (count <= QUAD_MAX)
    nodes_quad_kernel<<<blocks_for(count, QUADS), THREADS, 0, stream>>>(values, results, count,
                                                                        ctx->p2_round_constants);
  else
    nodes_kernel<<<blocks_for(count, THREADS), THREADS, 0, stream>>>(values, results, count, ctx->p2_round_constants);
  return (int)hipGetLastError();
}

// compute_node_hashes' preconditions (poseidon2.rs:231-239)
bool nodes_shape_ok(size_t values_len, size_t results_len) {
  return values_len % RATE == 0 && results_len % CAPACITY == 0 && values_len == 2 * results_len &&
         results_len / CAPACITY <= 0xFFFFFFFFull;
}

// build_merkle_tree_nodes' preconditions for every layer it will hash (poseidon2.rs:276-295)
bool node_layers_ok(size_t values_len, size_t results_len, uint32_t layers_count) {
  for (; layers_count; layers_count--) {
    if (values_len % RATE != 0 || values_len != results_len) return false;
    const size_t units = values_len / RATE;
    if (units == 0 || (units & (units - 1)) != 0) return false;  // values_len = RATE << layer
    if (!nodes_shape_ok(values_len, results_len >> 1)) return false;
    values_len = results_len >> 1;
    results_len -= results_len >> 1;
  }
  return true;
}

int run_node_layers(const ba_context *ctx, const u64 *values, size_t values_len, u64 *results, size_t results_len,
                    uint32_t layers_count, hipStream_t stream) {
  for (; layers_count; layers_count--) {
    const size_t half = results_len >> 1;
    const int rc = launch_nodes(ctx, values, results, (u32)(half / CAPACITY), stream);
    if (rc) return rc;
    values = results;
    values_len = half;
    results += half;
    results_len -= half;
  }
  (void)values_len;
  return BA_SUCCESS;
}

}  // namespace

extern "C" int ba_poseidon2_gl_set_round_constants(ba_context_t ctx, const uint64_t *round_constants) {
  return ba_guarded([&]() -> int {
    if (!ctx) return BA_ERROR_NOT_INITIALIZED;
    if (!round_constants) return BA_ERROR_INVALID_VALUE;
    int device = -1;
    if (hipGetDevice(&device) != hipSuccess || device != ctx->device) return BA_ERROR_INVALID_VALUE;
    // row r: the constants added before round r's S-boxes, lane 0 only in the partial rounds; a last
    // row of zeros is what the layer after the last round adds
    std::vector<u64> host(round_constants, round_constants + ROUNDS * WIDTH);
    host.resize((ROUNDS + 1) * WIDTH, 0);
    for (int i = 0; i < ROUNDS * WIDTH; i++) {
      const int r = i / WIDTH;
      const bool partial = r >= HALF_FULL_ROUNDS && r < HALF_FULL_ROUNDS + PARTIAL_ROUNDS;
      host[i] = partial && i % WIDTH ? 0 : gl::canon(host[i]);
    }
    if (!ctx->p2_round_constants) {
      void *p = nullptr;
      const hipError_t err = hipMalloc(&p, host.size() * sizeof(u64));
      if (err != hipSuccess) return err == hipErrorOutOfMemory ? BA_ERROR_OUT_OF_MEMORY : (int)err;
      ctx->p2_round_constants = (u64 *)p;
    }
    return (int)hipMemcpy(ctx->p2_round_constants, host.data(), host.size() * sizeof(u64), hipMemcpyHostToDevice);
  });
}

extern "C" int ba_poseidon2_gl_compute_leaf_hashes(const uint64_t *values, size_t values_len, uint64_t *results,
                                                   size_t results_len, uint32_t log_rows_per_hash,
                                                   int load_intermediate, int store_intermediate, ba_stream_t stream) {
  return ba_guarded([&]() -> int {
    ba_context *ctx = nullptr;
    if (const int rc = hasher_context(ctx)) return rc;
    // poseidon2.rs:186-207
    if (results_len % CAPACITY != 0 || log_rows_per_hash >= 32) return BA_ERROR_INVALID_VALUE;
    const size_t count = results_len / CAPACITY;
    if (count == 0) return BA_ERROR_INVALID_VALUE;
    const size_t rows = (size_t)1 << log_rows_per_hash;
    if (values_len % (count * rows) != 0) return BA_ERROR_INVALID_VALUE;
    const size_t cols = values_len / (count * rows);
    if (store_intermediate && (rows * cols) % RATE != 0) return BA_ERROR_INVALID_VALUE;
    if (cols > 0xFFFFFFFFull || count > 0xFFFFFFFFull || (values_len && !values) || !results)
      return BA_ERROR_INVALID_VALUE;
    const bool row = count <= ROW_MAX, quad = count <= QUAD_MAX;
    const auto kernel = row ? leaves_row_kernel : quad ? leaves_quad_kernel : leaves_kernel;
    const u32 per_block = row ? DIGEST_ROWS : quad ? QUADS : THREADS;
    kernel<<<blocks_for(count, per_block), THREADS, 0, (hipStream_t)stream>>>(
        values, results, (u32)rows, (u32)cols, (u32)count, load_intermediate, store_intermediate,
        ctx->p2_round_constants);
    return (int)hipGetLastError();
  });
}

extern "C" int ba_poseidon2_gl_compute_node_hashes(const uint64_t *values, size_t values_len, uint64_t *results,
                                                   size_t results_len, ba_stream_t stream) {
  return ba_guarded([&]() -> int {
    ba_context *ctx = nullptr;
    if (const int rc = hasher_context(ctx)) return rc;
    if (!nodes_shape_ok(values_len, results_len) || (results_len && (!values || !results)))
      return BA_ERROR_INVALID_VALUE;
    return launch_nodes(ctx, values, results, (u32)(results_len / CAPACITY), (hipStream_t)stream);
  });
}

extern "C" int ba_poseidon2_gl_build_merkle_tree_leaves(const uint64_t *values, size_t values_len, uint64_t *results,
                                                        size_t results_len, uint32_t log_rows_per_hash,
                                                        int load_intermediate, int store_intermediate,
                                                        ba_stream_t stream) {
  return ba_guarded([&]() -> int {
    // poseidon2.rs:253-274: the leaves count divides the values
    if (results_len % CAPACITY != 0 || results_len == 0 || values_len % (results_len / CAPACITY) != 0)
      return BA_ERROR_INVALID_VALUE;
    return ba_poseidon2_gl_compute_leaf_hashes(values, values_len, results, results_len, log_rows_per_hash,
                                               load_intermediate, store_intermediate, stream);
  });
}

extern "C" int ba_poseidon2_gl_build_merkle_tree_nodes(const uint64_t *values, size_t values_len, uint64_t *results,
                                                       size_t results_len, uint32_t layers_count, ba_stream_t stream) {
  return ba_guarded([&]() -> int {
    ba_context *ctx = nullptr;
    if (const int rc = hasher_context(ctx)) return rc;
    if (layers_count == 0) return BA_SUCCESS;
    if (!node_layers_ok(values_len, results_len, layers_count) || !values || !results) return BA_ERROR_INVALID_VALUE;
    return run_node_layers(ctx, values, values_len, results, results_len, layers_count, (hipStream_t)stream);
  });
}

extern "C" int ba_poseidon2_gl_build_merkle_tree(const uint64_t *values, size_t values_len, uint64_t *results,
                                                 size_t results_len, uint32_t log_rows_per_hash, uint32_t layers_count,
                                                 ba_stream_t stream) {
  return ba_guarded([&]() -> int {
    ba_context *ctx = nullptr;
    if (const int rc = hasher_context(ctx)) return rc;
    // poseidon2.rs:297-316
    if (layers_count == 0 || layers_count > 40 || results_len % (2 * CAPACITY) != 0) return BA_ERROR_INVALID_VALUE;
    const size_t leaves_count = results_len / (2 * CAPACITY);
    if (leaves_count == 0 || ((size_t)1 << (layers_count - 1)) > leaves_count || values_len % leaves_count != 0)
      return BA_ERROR_INVALID_VALUE;
    const size_t half = results_len >> 1;
    // every node layer is checked before the leaves launch, so a bad shape launches nothing
    if (!node_layers_ok(half, results_len - half, layers_count - 1)) return BA_ERROR_INVALID_VALUE;
    const int rc = ba_poseidon2_gl_compute_leaf_hashes(values, values_len, results, half, log_rows_per_hash, 0, 0, stream);
    if (rc) return rc;
    return run_node_layers(ctx, results, half, results + half, results_len - half, layers_count - 1, (hipStream_t)stream);
  });
}
