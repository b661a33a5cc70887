// barycentric.hip -- evaluation of polynomials given by their values on a coset domain at one
// point X, without interpolating: boojum_cuda::barycentric (crates/boojum-cuda/src/barycentric.rs:83-300).
//
// For the domain {c w^i : i < N} (w = omega_N, c the coset shift) and evaluations y_i,
//   f(X) = sum_i L_i y_i,   L_i = common / (X w^-i - c),   common = c (X^N - c^N) / (N c^N),
// the same factorisation the reference uses (native/barycentric.cu:11-93).  X is a base-field
// or extension-field element (F_p[u]/(u^2 - 7)); evaluations are base- or extension-field
// columns.  Layouts follow the reference's vectorized extension type: an extension vector of
// count elements is two planes (c0[count], c1[count]); an extension matrix column k starts at
// 2 k count; extension results are interleaved (c0, c1) per polynomial.
//
// Kernels:
//  * coefficients: each lane takes up to 8 elements, forms the denominators from the inverse power
//    table and inverts their 8 base-field norms at once (one field inversion and 3 multiplies per
//    element, Montgomery's trick), writing natural or bit-reversed order directly;
//  * batch evaluation: a grid over (row chunks of 4096, column groups), each lane 8 rows of a column
//    with their coefficients in registers across the columns of its group, exact sums of products
//    reduced once per column, one partial sum per (chunk, column); a second kernel, one wave per
//    column, sums the chunks.
#include <algorithm>
#include <mutex>
#include <vector>

#include "api_internal.h"
#include "gl_host.h"

namespace {

using gl::u32;
using gl::u64;

constexpr u32 kThreads = 256;
constexpr u32 kLogInvBatch = 3;

// Coefficients L_i = common / (X w^-i - c), common = (X^N - c^N) scale with scale = c / (N c^N) from
// the host; lane t of 2^log_t takes the 2^log_k elements at positions t + m 2^log_t.  The lane's
// natural indices are an arithmetic progression in both orders (bit-reversed: the low log_k bits of
// the index are the reversed m), so one table read and a constant step give all its powers of w.
// At an extension point X = a + b u the norm of X w^-i - c = (a w - c) + b w u (w short for w^-i) is
// w (w (a^2 - 7 b^2) - 2 a c) + c^2, in the base field: only norms are inverted, and
//   L_i = (w A - B + (w C - D) u) / norm,  A = e a - 7 f b, B = e c, C = f a - e b, D = f c,  common = e + f u.
// (A zero norm needs X on the domain, and then common = 0.)
// What bounds it: VALU issue, per lane ~170 instructions per extension element, ~1.0 k for the
// inversion and ~1.1 k for X^N.  One launch: 2^20 extension coefficients in bit-reversed order take
// 33 us, base-field ones 16 us; a one-lane kernel for the common factor, extension-field inversions
// and a separate bit reverse took 83 and 59 us.
template <bool EXT>
__global__ __launch_bounds__(kThreads) void coeffs_kernel(gl::Tables tab, const u64 *x_ptr, u64 *common_ptr, u64 c,
                                                          u64 cn, u64 scale, u32 log_count, u32 log_k,
                                                          bool bit_reverse, u64 *coeffs) {
  constexpr int K = 1 << kLogInvBatch;
  const u32 log_t = log_count - log_k;
  const u32 t = blockIdx.x * kThreads + threadIdx.x;
  if (t >> log_t) return;
  const u64 a = gl::canon(x_ptr[0]), b = EXT ? gl::canon(x_ptr[1]) : 0;
  // the lane's first index and index step
  const u32 shift = gl::OMEGA_LOG_ORDER - log_count;
  const u32 i0 = bit_reverse ? gl::ntt::bitrev32(t, log_t) << log_k : t;
  const u64 step = gl::pow_w(tab, (bit_reverse ? 1u : 1u << log_t) << shift, true);
  u64 w[K], den[K], pre[K];
  w[0] = gl::pow_w(tab, i0 << shift, true);
  u64 alpha = 0, beta = 0, gamma = 0;
  if constexpr (EXT) {
    alpha = gl::sub(gl::sqr(a), gl::mul(gl::sqr(b), 7));
    beta = gl::mul(gl::add(a, a), c);
    gamma = gl::sqr(c);
  }
  u64 run = 1;
#pragma unroll
  for (int j = 0; j < K; j++) {
    if (j >> log_k) break;
    if (j) w[j] = gl::mul_lazy(w[j ? j - 1 : 0], step);
    // lazy: a lazy value minus, or plus, a canonical one stays a u64 residue
    den[j] = EXT ? gl::add_lazy(gl::mul_lazy(w[j], gl::sub(gl::mul_lazy(w[j], alpha), beta)), gamma)
                 : gl::sub(gl::mul_lazy(a, w[j]), c);
    pre[j] = run;  // product of den[0..j)
    run = gl::mul_lazy(run, den[j]);
  }
  u64 inv = gl::inv(run);
  // X^N and the common factor
  u64 e = a, f = b;
#pragma unroll 1
  for (u32 k = 0; k < log_count; k++) {
    if constexpr (EXT) {  // (e^2 + 7 f^2, 2 e f) on the words of the products
      using namespace gl::isa;
      const u64 ee = gl::mul_lazy(e, e), ff = gl::mul_lazy(f, f), ef = gl::mul_lazy(e, f);
      e = gl::fold_words((u64)lo(ff) * 7 + lo(ee), (u64)hi(ff) * 7 + hi(ee));
      f = gl::fold_words((u64)lo(ef) * 2, (u64)hi(ef) * 2);
    } else {
      e = gl::mul_lazy(e, e);
    }
  }
  e = gl::mul(gl::sub(gl::reduce1(e), cn), scale);
  f = gl::mul(f, scale);
  if (t == 0) {
    common_ptr[0] = e;
    if (EXT) common_ptr[1] = f;
  }
  u64 A = 0, B = 0, C = 0, D = 0;
  if constexpr (EXT) {
    A = gl::sub(gl::mul(e, a), gl::mul(gl::mul(f, b), 7));
    B = gl::mul(e, c);
    C = gl::sub(gl::mul(f, a), gl::mul(e, b));
    D = gl::mul(f, c);
  } else {
    inv = gl::mul(inv, e);
  }
#pragma unroll
  for (int j = K - 1; j >= 0; j--) {
    if (j >> log_k) continue;
    // 1 / den[j] (times common at a base point)
    const u64 v = EXT ? gl::mul_lazy(inv, pre[j]) : gl::mul(inv, pre[j]);
    const u32 m = bit_reverse ? gl::ntt::bitrev32(j, log_k) : j;
    u64 *out = coeffs + (t + (m << log_t));
    if constexpr (EXT) {
      out[0] = gl::mul(gl::sub(gl::mul_lazy(w[j], A), B), v);
      out[1ull << log_count] = gl::mul(gl::sub(gl::mul_lazy(w[j], C), D), v);
    } else {
      out[0] = v;
    }
    inv = gl::mul_lazy(inv, den[j]);
  }
}

// ---------------------------------------------------------------- batch evaluation
constexpr u32 kEvalThreads = 512;
constexpr int kRows = 8;                           // rows per lane per column
constexpr u32 kChunk = kEvalThreads * kRows;       // rows per workgroup
constexpr u32 kColsPerGroup = 8;                   // most columns a workgroup visits

// An exact sum of up to 2^16 products of u64 values: the partial products of equal weight (1, 2^32,
// 2^64) are summed in 64 bits with a count of the carries.  8 VALU per product, where a reduced
// product and a field addition take 20.
struct ProductSum {
  u64 z = 0, m = 0, w = 0;
  u32 cz = 0, cm = 0, cw = 0;
  __device__ __forceinline__ void add(u64 x, u64 y) {
    using namespace gl::isa;
    u64 c;
    z = mad(lo(x), lo(y), z, c);
    cz = addc0(cz, c);
    m = mad(hi(x), lo(y), m, c);
    cm = addc0(cm, c);
    m = mad(lo(x), hi(y), m, c);
    cm = addc0(cm, c);
    w = mad(hi(x), hi(y), w, c);
    cw = addc0(cw, c);
  }
  // The sum as a lazy residue: words r0..r4 with r4 < 2^17, reduced as [r0, r1] - [r3, r4] + r2 EPS
  // (2^64 = EPS, 2^96 = -1, 2^128 = -2^32); the borrow selects t - EPS (t > 2^64 - 2^50, no wrap),
  // the carry R + EPS (R < r2 EPS, no wrap).
  __device__ __forceinline__ u64 value() const {
    using namespace gl::isa;
    u64 k, b, c, dead;
    const u32 r1 = add_co(hi(z), lo(m), k);
    u32 r2 = addc(lo(w), hi(m), k, k);
    u32 r3 = addc0(hi(w), k, k);
    u32 r4 = addc0(cw, k);
    r2 = add_co(r2, cz, k);
    r3 = addc(r3, cm, k, k);
    r4 = addc0(r4, k);
    const u32 t0 = sub_co(lo(z), r3, b);
    const u32 t1 = subb(r1, r4, b, b);
    const u64 r = mad_eps(r2, minus_eps(t0, t1, b), c);
    return mad_eps(one_if(c), r, dead);
  }
};

// A residue cut into limbs of 22, 22 and 20 bits, so that sums over lanes are plain 32-bit additions.
struct Limbs {
  u32 l[3];
};
__device__ __forceinline__ Limbs limbs_of(u64 x) {
  return {{(u32)x & 0x3FFFFFu, (u32)(x >> 22) & 0x3FFFFFu, (u32)(x >> 44)}};
}
// l0 + l1 2^22 + l2 2^44, canonical
__device__ __forceinline__ u64 joined(const Limbs &v) {
  return gl::reduce1(gl::fold_words(v.l[0] + ((u64)v.l[1] << 22), (u64)v.l[2] << 12));
}

// lane 63 holds the sum of the wave's 64 values (six row shifts and broadcasts; the other lanes hold
// partial sums)
template <int CTRL, int ROWS>
__device__ __forceinline__ u32 plus_dpp(u32 x) {
  return x + (u32)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROWS, 0xF, true);
}
__device__ __forceinline__ u32 wave_sum(u32 x) {
  x = plus_dpp<0x111, 0xF>(x);  // row_shr:1, 2, 4, 8
  x = plus_dpp<0x112, 0xF>(x);
  x = plus_dpp<0x114, 0xF>(x);
  x = plus_dpp<0x118, 0xF>(x);
  x = plus_dpp<0x142, 0xA>(x);  // row_bcast:15 into rows 1 and 3
  x = plus_dpp<0x143, 0xC>(x);  // row_bcast:31 into rows 2 and 3
  return x;
}
__device__ __forceinline__ Limbs wave_sum(const Limbs &v) { return {{wave_sum(v.l[0]), wave_sum(v.l[1]), wave_sum(v.l[2])}}; }

// partial[chunk, col] = sum over the chunk's rows of L_row * y[row, col], for the chunk's rows and
// `cols_per_group` columns; with a single chunk, the evaluations themselves (`partial` = evals).
// XE: extension coefficients; YE: extension values.
// What bounds it: HBM (8 B per base value read once), with 32 KB of the next column in flight per
// workgroup.  64 x 2^20 base values at an extension point take 103 us with the sum over the chunks
// (5.2 TB/s), at a base point 94 us; reducing every product took 278 and 164 us, 52 of them in a
// final kernel with one lane per column.
template <bool XE, bool YE>
__global__ __launch_bounds__(kEvalThreads) void partial_kernel(const u64 *ys, const u64 *coeffs, u32 log_count,
                                                               u32 num_polys, u32 cols_per_group, u64 *partial,
                                                               u32 chunks) {
  constexpr int PL = XE ? 2 : 1, PY = YE ? 2 : 1;  // planes of a coefficient, of a value
  constexpr int WAVES = kEvalThreads / 64;
  const u64 count = 1ull << log_count;
  const u32 chunk = blockIdx.x;
  const u32 t = threadIdx.x;
  // rows past the end of a short column read row 0 with coefficient zero
  u32 row[kRows];
  u64 l[PL][kRows];
#pragma unroll
  for (int k = 0; k < kRows; k++) {
    const u32 r = chunk * kChunk + t + k * kEvalThreads;
    const bool in = !(r >> log_count);
    row[k] = in ? r : 0;
#pragma unroll
    for (int p = 0; p < PL; p++) {
      const u64 x = coeffs[row[k] + p * count];
      l[p][k] = in ? x : 0;
    }
  }
  __shared__ u64 sums[kColsPerGroup][PL][WAVES];
  const u32 col0 = blockIdx.y * cols_per_group;
  const u32 cols = min(num_polys - col0, cols_per_group);
  // the next column's values are loaded while the current column is accumulated
  u64 nxt[PY][kRows];
  auto fetch = [&](u32 col) {
    const u64 *y = ys + (u64)col * PY * count;
#pragma unroll
    for (int k = 0; k < kRows; k++)
#pragma unroll
      for (int p = 0; p < PY; p++) nxt[p][k] = y[row[k] + p * count];
  };
  fetch(col0);
  for (u32 i = 0; i < cols; i++) {
    u64 cur[PY][kRows];
#pragma unroll
    for (int k = 0; k < kRows; k++)
#pragma unroll
      for (int p = 0; p < PY; p++) cur[p][k] = nxt[p][k];
    if (i + 1 < cols) fetch(col0 + i + 1);
    Limbs out[PL];
    if constexpr (YE) {  // (l0 + l1 u)(y0 + y1 u) = l0 y0 + 7 l1 y1 + (l0 y1 + l1 y0) u
      ProductSum s00, s11, s01;
#pragma unroll
      for (int k = 0; k < kRows; k++) {
        s00.add(l[0][k], cur[0][k]);
        s11.add(l[1][k], cur[1][k]);
        s01.add(l[0][k], cur[1][k]);
        s01.add(l[1][k], cur[0][k]);
      }
      const Limbs p = limbs_of(s00.value()), q = limbs_of(s11.value());
#pragma unroll
      for (int j = 0; j < 3; j++) out[0].l[j] = p.l[j] + 7 * q.l[j];  // < 2^25, < 2^31 over a wave
      out[1] = limbs_of(s01.value());
    } else {
#pragma unroll
      for (int p = 0; p < PL; p++) {
        ProductSum s;
#pragma unroll
        for (int k = 0; k < kRows; k++) s.add(l[p][k], cur[0][k]);
        out[p] = limbs_of(s.value());
      }
    }
#pragma unroll
    for (int p = 0; p < PL; p++) {
      const u64 v = joined(wave_sum(out[p]));
      if ((t & 63) == 63) sums[i][p][t >> 6] = v;
    }
  }
  __syncthreads();
  // one lane per (column, plane) adds the waves' sums
  if (t < cols * PL) {
    const u32 i = t / PL, p = t % PL;
    u64 s = sums[i][p][0];
#pragma unroll
    for (int w = 1; w < WAVES; w++) s = gl::add(s, sums[i][p][w]);
    // partial sums: a column holds `chunks` values per plane; a single chunk's are its evaluations
    partial[((u64)(col0 + i) * PL + p) * chunks + chunk] = s;
  }
}

// evals[col] = sum over chunks of partial[chunk, col], one wave per (column, plane); extension results
// interleaved (c0, c1).  A lane sums the words of its chunks in 64 bits (2^31 values are 2^19 chunks, 2^13 a lane).
__global__ __launch_bounds__(64) void final_kernel(const u64 *partial, u32 chunks, u64 *evals) {
  const u64 *p = partial + (u64)blockIdx.x * chunks;
  u64 l = 0, h = 0;
  for (u32 k = threadIdx.x; k < chunks; k += 64) {
    const u64 x = p[k];
    l += gl::isa::lo(x);
    h += gl::isa::hi(x);
  }
  const u64 s = joined(wave_sum(limbs_of(gl::fold_words(l, h))));
  if (threadIdx.x == 63) evals[blockIdx.x] = s;
}

bool pow2(u64 x) { return x && !(x & (x - 1)); }
u32 log2u(u64 x) {
  u32 l = 0;
  while ((1ull << l) < x) l++;
  return l;
}

}  // namespace

extern "C" int ba_barycentric_precompute_lagrange_coeffs(int ext, const uint64_t *x, uint64_t *common_factor,
                                                         uint64_t coset, uint64_t *lagrange_coeffs, uint32_t count,
                                                         int bit_reverse, ba_stream_t stream) {
  if (!x || !common_factor || !lagrange_coeffs || !pow2(count) || (ext != 0 && ext != 1)) return BA_ERROR_INVALID_VALUE;
  const u32 log_count = log2u(count);
  if (log_count > gl::OMEGA_LOG_ORDER) return BA_ERROR_INVALID_VALUE;
  const ba_context *ctx = ba_context_for_current_device();
  if (!ctx) return BA_ERROR_NOT_INITIALIZED;
  hipStream_t s = (hipStream_t)stream;
  // 8 elements per lane once a workgroup's lanes have at least one each
  const u32 log_k = log_count > 8 ? std::min(kLogInvBatch, log_count - 8) : 0;
  const u32 grid = std::max(1u, (count >> log_k) / kThreads);
  const u64 c = gl::canon(coset), cn = gl_host::pow(c, count);
  const u64 scale = gl_host::mul(c, gl_host::inv(gl_host::mul(count, cn)));
  const auto kernel = ext ? coeffs_kernel<true> : coeffs_kernel<false>;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(kThreads), 0, s, ctx->tab, x, common_factor, c, cn, scale, log_count,
                     log_k, bit_reverse != 0, lagrange_coeffs);
  return (int)hipGetLastError();
}

extern "C" int ba_barycentric_batch_eval_temp_elems(int kind, uint32_t count, uint32_t num_polys, uint64_t *elems) {
  if (!elems || !pow2(count) || kind < 0 || kind > 2) return BA_ERROR_INVALID_VALUE;
  const u64 chunks = ((u64)count + kChunk - 1) / kChunk;
  *elems = chunks * num_polys * (kind == 0 ? 1 : 2);
  return BA_SUCCESS;
}

extern "C" int ba_barycentric_batch_eval(int kind, const uint64_t *ys, uint32_t count, uint32_t num_polys,
                                         const uint64_t *lagrange_coeffs, uint64_t *temp, uint64_t temp_elems,
                                         uint64_t *evals, ba_stream_t stream) {
  uint64_t need = 0;
  if (int rc = ba_barycentric_batch_eval_temp_elems(kind, count, num_polys, &need)) return rc;
  if (num_polys == 0) return BA_SUCCESS;
  if (!ys || !lagrange_coeffs || !evals || !temp || temp_elems < need) return BA_ERROR_INVALID_VALUE;
  const u32 log_count = log2u(count);
  const u32 chunks = (u32)(((u64)count + kChunk - 1) / kChunk);
  hipStream_t s = (hipStream_t)stream;
  if ((num_polys + kColsPerGroup - 1) / kColsPerGroup > 65535) return BA_ERROR_INVALID_VALUE;
  // Columns per workgroup: as many as give most CUs a workgroup.  Eight columns read the
  // coefficients once for all of them; with fewer workgroups than that, idle CUs cost more than
  // reading them again: 100 x 2^12 takes 5.6 us on 100 workgroups and 12.0 on 13, 100 x 2^16 17.1 us
  // on 800 and 15.8 on 208.
  u32 cols = kColsPerGroup;
  while (cols > 1 && (u64)chunks * ((num_polys + cols - 1) / cols) < 192) cols /= 2;
  const dim3 grid(chunks, (num_polys + cols - 1) / cols);
  u64 *sums = chunks == 1 ? evals : temp;
  // 0: base-field evaluations at a base-field point; 1: base-field evaluations at an extension point;
  // 2: extension evaluations at an extension point
  const auto kernel = kind == 0   ? partial_kernel<false, false>
                      : kind == 1 ? partial_kernel<true, false>
                                  : partial_kernel<true, true>;
  hipLaunchKernelGGL(kernel, grid, dim3(kEvalThreads), 0, s, ys, lagrange_coeffs, log_count, num_polys, cols, sums,
                     chunks);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess || chunks == 1) return (int)err;
  hipLaunchKernelGGL(final_kernel, dim3(num_polys * (kind ? 2 : 1)), dim3(64), 0, s, (const u64 *)temp, chunks, evals);
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------- batch evaluation, no allocation
// For callers that cannot allocate device memory (code under stream capture, tight serving loops):
// the partial sums live in this file-scope array instead of a caller workspace.  Every GPU the
// library runs on holds its own copy, at its own address, until the process ends.  The partial
// kernel writes every element the final kernel reads, so nothing has to start at zero; calls that
// overlap on one GPU share the array and race.
constexpr uint64_t kStaticTempElems = 1ull << 19;  // 4 MiB
static __device__ __align__(256) uint64_t scratch[kStaticTempElems];

namespace {
std::mutex g_scratch_mutex;
std::vector<uint64_t *> g_scratch_ptr;  // per device: the device address of `scratch`

// The device address of this GPU's copy of `scratch`, looked up once per device (with that device
// current) and kept; the array's name is a host-side stand-in and is never passed to a kernel.
int scratch_for_current_device(uint64_t **ptr) {
  int device = -1;
  hipError_t err = hipGetDevice(&device);
  if (err != hipSuccess) return (int)err;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if ((size_t)device >= g_scratch_ptr.size()) g_scratch_ptr.resize((size_t)device + 1, nullptr);
  if (!g_scratch_ptr[device]) {
    void *p = nullptr;
    err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (err != hipSuccess) return (int)err;
    if (!p) return BA_ERROR_NOT_INITIALIZED;
    g_scratch_ptr[device] = (uint64_t *)p;
  }
  *ptr = g_scratch_ptr[device];
  return BA_SUCCESS;
}
}  // namespace

extern "C" int ba_barycentric_batch_eval_noalloc(int kind, const uint64_t *ys, uint32_t count, uint32_t num_polys,
                                                 const uint64_t *lagrange_coeffs, uint64_t *evals,
                                                 ba_stream_t stream) {
  return ba_guarded([&]() -> int {
    uint64_t need = 0;
    if (int rc = ba_barycentric_batch_eval_temp_elems(kind, count, num_polys, &need)) return rc;
    if (num_polys == 0) return BA_SUCCESS;
    if (need > kStaticTempElems) return BA_ERROR_INVALID_VALUE;  // beyond the array's 2^19 elements
    if (!ys || !lagrange_coeffs || !evals) return BA_ERROR_INVALID_VALUE;
    uint64_t *temp = nullptr;
    if (int rc = scratch_for_current_device(&temp)) return rc;
    return ba_barycentric_batch_eval(kind, ys, count, num_polys, lagrange_coeffs, temp, kStaticTempElems, evals,
                                     stream);
  });
}
