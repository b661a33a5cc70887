// lde.hip -- batched coset low-degree extension (shivini's trace-commitment LDE).
//
// Reference composition (crates/shivini/src/data_structures/storage.rs:154-260,
// crates/shivini/src/primitives/ntt.rs:10-42,407-510): evaluations -> n2b inverse NTT -> bit
// reverse -> monomials (natural) -> for each coset c < B: n2b forward NTT with coset index
// bitrev_{log B}(c) and log_extension_degree = log B.
//
// Here the monomials stay in the bit-reversed order the inverse NTT leaves them in, and the
// first pass of every coset NTT gathers them (coalesced chunk reads staged through LDS), so the
// separate bit-reverse pass over the data disappears.  The coset NTTs of a call run pass by pass,
// every pass one launch over up to 8 cosets: passes(iNTT) + passes(NTT) launches, all on the
// caller's stream.
#include <algorithm>
#include <cstdlib>
#include <vector>

#include "api_internal.h"

namespace {

uint32_t bitrev_bits(uint32_t x, uint32_t bits) {
  uint32_t r = 0;
  for (uint32_t i = 0; i < bits; i++) r |= ((x >> i) & 1u) << (bits - 1 - i);
  return r;
}

// True when the n-element vectors starting at k s1 + c s2 (k < K, c < C) are pairwise disjoint.
// Two starts differ by dk s1 + dc s2 with |dk| < K, |dc| < C, not both zero.  Up to sign the
// index with the smaller count (outer) is >= 0; for each outer step the point of the inner
// progression closest to it is found by division, so no list of starts is built and the work
// is O(min(K, C)).
bool vectors_disjoint(uint64_t K, uint64_t s1, uint64_t C, uint64_t s2, uint64_t n) {
  typedef unsigned __int128 u128;
  uint64_t O = K, so = s1, I = C, si = s2;
  if (C < K) O = C, so = s2, I = K, si = s1;
  if (I > 1 && si < n) return false;  // outer step 0: neighbours along the inner stride
  for (uint64_t d = 1; d < O; d++) {
    const u128 x = (u128)d * so;  // distance to cancel with inner steps -e, 0 <= e <= I - 1
    u128 closest;
    if (si == 0) {
      closest = x;
    } else {
      const u128 q = x / si, r = x % si;
      if (q > I - 1) {
        closest = x - (u128)(I - 1) * si;
      } else {
        closest = r;
        if (q + 1 <= I - 1 && (u128)si - r < closest) closest = (u128)si - r;
      }
    }
    if (closest < n) return false;
  }
  return true;
}

}  // namespace

int ba_validate_lde(uint64_t *evals, uint64_t in_stride, uint64_t *monomials, uint64_t *out,
                    uint64_t out_col_stride, uint64_t out_coset_stride, uint32_t log_n,
                    uint32_t num_cols, uint32_t log_blowup) {
  if (log_n < 1 || log_n > BA_MAX_LOG_N || log_blowup < 1 || log_n + log_blowup > gl::OMEGA_LOG_ORDER)
    return BA_ERROR_INVALID_VALUE;
  const uint64_t n = 1ull << log_n;
  const uint64_t blowup = 1ull << log_blowup;
  if (num_cols == 0) return BA_SUCCESS;
  if (!evals || !out || in_stride < n) return BA_ERROR_INVALID_VALUE;
  // every buffer's extent must be addressable
  typedef unsigned __int128 u128;
  const u128 out_span = ((u128)(num_cols - 1) * out_col_stride + (u128)(blowup - 1) * out_coset_stride + n) * 8;
  const u128 ev_span = ((u128)(num_cols - 1) * in_stride + n) * 8;
  const u128 mono_span = (u128)num_cols * n * 8;
  if ((u128)(uintptr_t)out + out_span > ((u128)1 << 64) || (u128)(uintptr_t)evals + ev_span > ((u128)1 << 64) ||
      (monomials && (u128)(uintptr_t)monomials + mono_span > ((u128)1 << 64)))
    return BA_ERROR_INVALID_VALUE;
  // the B * num_cols output vectors of n elements must be pairwise disjoint
  if (!vectors_disjoint(num_cols, out_col_stride, blowup, out_coset_stride, n)) return BA_ERROR_INVALID_VALUE;
  // the outputs overlap neither the evaluations nor the monomials; monomials given separately
  // do not overlap the evaluations
  const char *out_end = (const char *)out + (size_t)out_span;
  const char *ev_end = (const char *)evals + (size_t)ev_span;
  auto overlap = [](const void *a0, const void *a1, const void *b0, const void *b1) {
    return a0 < b1 && b0 < a1;
  };
  if (overlap(out, out_end, evals, ev_end)) return BA_ERROR_INVALID_VALUE;
  if (monomials) {
    const char *mono_end = (const char *)monomials + (size_t)mono_span;
    if (overlap(out, out_end, monomials, mono_end) || overlap(evals, ev_end, monomials, mono_end))
      return BA_ERROR_INVALID_VALUE;
  }
  return BA_SUCCESS;
}

// BOOJUM_AMD_LDE_SERIAL=1 in the environment (read once) launches every coset's passes on their own,
// in order, so that a profiler's per-kernel figures are one transform's; so does launch tracing.  The
// kernels and their launch choices are those of the merged launches.
static bool lde_serial() {
  static const bool serial = [] {
    const char *e = std::getenv("BOOJUM_AMD_LDE_SERIAL");
    return e && e[0] == '1';
  }();
  return serial;
}

// Each pass of the coset NTTs is merged over the cosets.  A small LDE is a few launches of
// latency-shaped passes (13 x 2^14 at blowup 4: 29 us, 110 as ten launches of 52 workgroups over four
// streams); a large one reads the monomials once for 8 cosets; one of at most 2^3 points at blowup 64 is 9
// launches in place of 65.
int ba_launch_lde_cosets(const ba_context *ctx, const uint64_t *mono, uint64_t mono_stride, uint64_t *out,
                         uint64_t out_col_stride, uint64_t out_coset_stride, uint32_t log_n, uint32_t num_cols,
                         uint32_t log_blowup, bool apart, hipStream_t stream) {
  std::vector<BaPassLaunch> ls;
  const uint32_t blowup = 1u << log_blowup;
  static_assert(gl::ntt::MAX_COSETS == 8, "cosets of one launch");
  uint32_t log_merged = std::min(log_blowup, 3u);
  // a transform per thread: at most 2^31 threads a launch
  while (log_n < 4 && log_merged && ((uint64_t)num_cols << log_merged) > (1ull << 31)) log_merged--;
  const uint32_t log_at_once = apart ? 0 : log_merged, at_once = 1u << log_at_once;
  for (uint32_t c0 = 0; c0 < blowup; c0 += at_once) {
    ls.clear();
    int rc = ba_build_ntt(ctx, mono, out + (uint64_t)c0 * out_coset_stride, log_n, num_cols, mono_stride, out_col_stride,
                      false, false, log_blowup, bitrev_bits(c0, log_blowup), /*in_bitrev_gather=*/true, ls,
                      BA_LAT_AUTO, false, 1u << log_merged);
    if (rc) return rc;
    gl::ntt::CosetArgs first{};
    first.coset_stride = out_coset_stride;
    first.log_cosets = log_at_once;
    for (uint32_t y = 0; y < at_once; y++)
      ba_scale_factors(log_n, false, log_blowup, bitrev_bits(c0 + y, log_blowup), first.scale_tab[y],
                       first.coset_mul[y]);
    for (const BaPassLaunch &l : ls) {
      if (l.pass == 0) {
        first.a = l.args;
        // A short column's cosets share cache lines, and a workgroup its tile's monomials: a tile's cosets run
        // on one XCD if the tiles are a multiple of 8 (the last ones may be empty).  691802 columns of 2^1 at
        // blowup 2 take 19.8 us, 27.8 on the XCDs in turn; 1589344 at blowup 4 75 and 101.
        uint64_t tiles = l.grid;
        if (log_n < 4 && at_once > 1 && tiles > 8) tiles = (tiles + 7) & ~7ull;
        ba_trace_before(stream, l.coset_name);
        hipLaunchKernelGGL(l.coset_kernel, dim3((uint32_t)(tiles << log_at_once)), dim3(l.threads), 0, stream, first);
      } else {
        gl::ntt::PassArgs a = l.args;
        a.slice_stride = out_coset_stride;
        ba_trace_before(stream, l.name);
        hipLaunchKernelGGL(l.kernels.single, dim3((uint32_t)l.grid, at_once), dim3(l.threads), 0, stream, a);
      }
      ba_trace_after(stream);
      const hipError_t err = hipGetLastError();
      if (err != hipSuccess) return (int)err;
    }
  }
  return BA_SUCCESS;
}

// The LDE's launches on `stream`; with natural_monomials the monomials are bit-reversed in place once
// every coset has read them.
static int lde_run(ba_context_t ctx, uint64_t *evals, uint64_t in_stride, uint64_t *monomials,
                   uint64_t *out, uint64_t out_col_stride, uint64_t out_coset_stride, uint32_t log_n,
                   uint32_t num_cols, uint32_t log_blowup, bool natural_monomials, ba_stream_t stream) {
  // arguments first (host-only checks), then the context
  int rc = ba_validate_lde(evals, in_stride, monomials, out, out_col_stride, out_coset_stride, log_n,
                           num_cols, log_blowup);
  if (rc) return rc;
  if (!ctx) return BA_ERROR_NOT_INITIALIZED;
  if (num_cols == 0) return BA_SUCCESS;
  int device = -1;  // the context's tables live on its device
  if (hipGetDevice(&device) != hipSuccess || device != ctx->device) return BA_ERROR_INVALID_VALUE;
  uint64_t *mono = monomials ? monomials : evals;
  const uint64_t mono_stride = monomials ? (1ull << log_n) : in_stride;
  // The inverse NTT is latency-shaped by size alone: a tile_log of 10 says that plain NTTs of the class
  // take those passes whatever the batch, which costs a large LDE up to a third of its time (blowup 2,
  // 128 columns of 2^18: 1000 us against 754; 2048 of 2^14: 753 against 660).
  std::vector<BaPassLaunch> ls;
  rc = ba_build_ntt(ctx, evals, mono, log_n, num_cols, in_stride, mono_stride, false, true, 0, 0, false, ls,
                    ba_small_batch(num_cols, log_n) ? BA_LAT_AUTO : BA_LAT_NEVER);
  if (rc || (rc = ba_run_launches(ls, (hipStream_t)stream))) return rc;
  rc = ba_launch_lde_cosets(ctx, mono, mono_stride, out, out_col_stride, out_coset_stride, log_n, num_cols,
                            log_blowup, ba_trace_active() || lde_serial(), (hipStream_t)stream);
  if (rc || !natural_monomials) return rc;
  return ba_bit_reverse_in_place(mono, mono_stride, log_n, num_cols, stream);
}

extern "C" int ba_lde_batch(ba_context_t ctx, uint64_t *evals, uint64_t in_stride,
                            uint64_t *monomials, uint64_t *out, uint64_t out_col_stride,
                            uint64_t out_coset_stride, uint32_t log_n, uint32_t num_cols,
                            uint32_t log_blowup, ba_stream_t stream) {
  return ba_guarded([&]() -> int {
    return lde_run(ctx, evals, in_stride, monomials, out, out_col_stride, out_coset_stride, log_n, num_cols,
                   log_blowup, false, stream);
  });
}

extern "C" int ba_lde_batch_ex(ba_context_t ctx, uint64_t *evals, uint64_t in_stride,
                               uint64_t *monomials, uint64_t *out, uint64_t out_col_stride,
                               uint64_t out_coset_stride, uint32_t log_n, uint32_t num_cols,
                               uint32_t log_blowup, uint32_t flags, ba_stream_t stream) {
  return ba_guarded([&]() -> int {
    if (flags & ~(uint32_t)BA_LDE_NATURAL_MONOMIALS) return BA_ERROR_INVALID_VALUE;
    return lde_run(ctx, evals, in_stride, monomials, out, out_col_stride, out_coset_stride, log_n, num_cols,
                   log_blowup, (flags & BA_LDE_NATURAL_MONOMIALS) != 0, stream);
  });
}
