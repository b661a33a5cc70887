// ntt.hip -- batch NTT planner, launchers and the boojum_cuda::ntt entry points.
//
// Reference: crates/boojum-cuda/src/ntt.rs:57-369.  The reference plans 1-3 multi-stage
// kernels per log_n in 16..24 and falls back to log_n single-stage launches below 16
// (ntt.rs:201-241); here every size 1..30 runs in at most 1 + ceil((log_n - 12) / 8)
// passes of radix-16 register blocks (see ntt_kernels.h).
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "api_internal.h"
#include "gl_host.h"
#include "ntt_inst.h"
#include "ntt_lat.h"

using gl::ntt::PassArgs;

bool ba_plan_from_bits(uint32_t log_n, bool n2b, const uint32_t *bits, int num_passes, NttPlan &plan) {
  constexpr uint32_t T = gl::ntt::TILE_LOG;
  if (num_passes < 1 || num_passes > 8) return false;
  if (log_n < 4) {  // whole transform per thread
    if (num_passes != 1 || bits[0] != log_n) return false;
  } else if (log_n <= T) {  // one contiguous pass
    if (num_passes != 1 || bits[0] != log_n) return false;
  } else {
    // contiguous pass over 9..12 low bits (whole 4096-element tiles), strided passes of 4..10
    if (num_passes < 2 || bits[0] < 9 || bits[0] > T) return false;
    uint32_t sum = bits[0];
    for (int i = 1; i < num_passes; i++) {
      if (bits[i] < 4 || bits[i] > 10) return false;
      sum += bits[i];
    }
    if (sum != log_n) return false;
  }
  plan = NttPlan{};
  plan.num_passes = num_passes;
  uint32_t lo[8];
  uint32_t at = 0;
  for (int i = 0; i < num_passes; i++) lo[i] = at, at += bits[i];
  for (int i = 0; i < num_passes; i++) {
    const int src = n2b ? num_passes - 1 - i : i;  // n2b: top bits first
    plan.lo_bit[i] = lo[src];
    plan.bits[i] = bits[src];
    plan.contig[i] = src == 0;
  }
  return true;
}

NttPlan ba_plan_ntt(uint32_t log_n, bool n2b, bool gather) {
  // passes listed from the low bits up: a contiguous pass of 12 bits, then strided passes of
  // 8 bits, the last of 4..8 (bits borrowed from the pass below when fewer than 4 remain).
  // 2^21 takes one strided pass of 9 bits, in 64-byte runs, for two of 5 and 4 that each move every
  // element: 32 columns 704 -> 583 us (n2b), 703 -> 632 (b2n inverse), 716 -> 630 (coset), 13 columns
  // 269 -> 257, 275 -> 277, 287 -> 276, one column 46 -> 41.  A 10-bit one at 2^22, in 32-byte runs,
  // is no faster than 6 and 4 bits (16 columns 717 against 720, with a coset 800 against 720).  The
  // gathered pass of an LDE's coset NTT has no 9-bit build.
  uint32_t bits[8];
  int np = 0;
  if (log_n <= (uint32_t)gl::ntt::TILE_LOG) {
    bits[np++] = log_n;
  } else {
    uint32_t rest = log_n - gl::ntt::TILE_LOG;
    uint32_t sc = gl::ntt::TILE_LOG;
    if (rest < 4) {
      sc -= 4 - rest;
      rest = 4;
    }
    bits[np++] = sc;
    while (rest > 0) {
      uint32_t take = rest;
      if (rest > 8 && (log_n != 21 || gather)) take = (rest - 8 >= 4) ? 8 : rest - 4;
      bits[np++] = take;
      rest -= take;
    }
  }
  NttPlan plan{};
  (void)ba_plan_from_bits(log_n, n2b, bits, np, plan);
  return plan;
}

namespace {

using namespace gl::ntt;

// scale: 0 none, 1 one factor for every element, 2 per-element coset factors (the strided
// kernels fuse 1 and 2 alike)
// waves: the 9..12-bit contiguous pass's variant (3 or 4 waves per SIMD)
// shared: the launch shares the GPU with other streams' work (strided passes: three-waves builds)
BaKernels pick_kernel(bool contig, uint32_t S, bool n2b, bool inverse, bool top, int scale,
                      bool whole, bool gather, uint32_t waves, bool shared) {
  if (contig) {
    if (S <= 8) return ba_pick_contig_lo(S, n2b, inverse, scale, whole);
    return waves == 3 ? ba_pick_contig_hi3(S, n2b, inverse, scale, whole)
                      : ba_pick_contig_hi(S, n2b, inverse, scale, whole);
  }
  return ba_pick_strided(S, n2b, inverse, top, scale != 0, gather, shared);
}

// kernel names as rocprofv3 prints them, for launch tracing; the table is built once, by the
// first caller (a function-local static initialiser, so concurrent first calls are safe)
struct KernelNames {
  // [strided, contig, strided shared build][S][n2b][inverse][top or whole][scale][gather or 4-waves]
  char n[3][13][2][2][2][3][2][120];
  KernelNames() {
    static const char *tf[2] = {"false", "true"};
    for (int s = 0; s < 13; s++)
      for (int d = 0; d < 2; d++)
        for (int i = 0; i < 2; i++)
          for (int tp = 0; tp < 2; tp++)
            for (int sc = 0; sc < 3; sc++)
              for (int ga = 0; ga < 2; ga++) {
                snprintf(n[1][s][d][i][tp][sc][ga], sizeof(n[1][s][d][i][tp][sc][ga]),
                         "void gl::ntt::ntt_pass_contig<%d, %s, %s, %d, %s, %d>(gl::ntt::PassArgs)", s, tf[d],
                         tf[i], sc, tf[tp], ga ? 4 : 3);
                snprintf(n[0][s][d][i][tp][sc][ga], sizeof(n[0][s][d][i][tp][sc][ga]),
                         "void gl::ntt::ntt_pass_strided<%d, %s, %s, %s, %s, %s>(gl::ntt::PassArgs)", s,
                         tf[d], tf[i], tf[tp], tf[sc != 0], tf[ga]);
                snprintf(n[2][s][d][i][tp][sc][ga], sizeof(n[2][s][d][i][tp][sc][ga]),
                         "void gl::ntt::ntt_pass_strided_shared<%d, %s, %s, %s, %s, %s>(gl::ntt::PassArgs)", s,
                         tf[d], tf[i], tf[tp], tf[sc != 0], tf[ga]);
              }
  }
};

// shared_build: a strided pass's three-waves build for shared launches
const char *kernel_name(bool contig, uint32_t S, bool n2b, bool inverse, bool top, int scale,
                        bool gather, uint32_t waves, bool shared_build) {
  static const KernelNames names;
  return names.n[contig ? 1 : (shared_build ? 2 : 0)][S][n2b][inverse][top][scale][contig ? waves == 4 : gather];
}

// the same for the gathered first pass of an LDE's coset NTTs (4096-element tiles)
struct CosetNames {
  char n[3][13][80];  // strided, contiguous at 3 waves per SIMD, at 4
  CosetNames() {
    for (int s = 0; s < 13; s++) {
      snprintf(n[0][s], sizeof(n[0][s]), "void gl::ntt::ntt_pass_strided_cosets<%d>(gl::ntt::CosetArgs)", s);
      for (int w = 3; w <= 4; w++)
        snprintf(n[w - 2][s], sizeof(n[w - 2][s]), "void gl::ntt::ntt_pass_contig_cosets<%d, %s, %d>(gl::ntt::CosetArgs)",
                 s, s == TILE_LOG ? "true" : "false", w);
    }
  }
};
// and for whole transforms per thread
struct TinyNames {
  char n[4][2][2][80], cosets[4][80];  // [log_n][n2b][inverse]
  TinyNames() {
    static const char *tf[2] = {"false", "true"};
    for (int k = 0; k < 4; k++) {
      for (int d = 0; d < 2; d++)
        for (int i = 0; i < 2; i++)
          snprintf(n[k][d][i], sizeof(n[k][d][i]), "void gl::ntt::ntt_tiny<%d, %s, %s>(gl::ntt::PassArgs)", k, tf[d], tf[i]);
      snprintf(cosets[k], sizeof(cosets[k]), "void gl::ntt::ntt_tiny_cosets<%d>(gl::ntt::CosetArgs)", k);
    }
  }
};
const char *tiny_name(uint32_t log_n, bool n2b, bool inverse, bool cosets) {
  static const TinyNames names;
  return cosets ? names.cosets[log_n] : names.n[log_n][n2b][inverse];
}

const char *coset_name(bool contig, uint32_t S, uint32_t waves) {
  static const CosetNames names;
  return names.n[!contig ? 0 : waves == 4 ? 2 : 1][S];
}

constexpr uint64_t kMaxGrid = 0x7FFFFFFFull;

}  // namespace

// Columns (tile repeats) per workgroup, at most 8.  More of them spread the workgroup's set-up (round
// twiddles, scale factors) over more tiles, but leave fewer workgroups to even out the last ones:
// 1024 run at once (4 per CU).  `tiles` counts every tile of the launch, `cols` what a workgroup may
// repeat over.  The lines are measured; microseconds per launch, by columns per workgroup:
//   contiguous, 12 bits:  1792 tiles: 47 (1), 41 (2), 53 (4); 4096: 85, 85, 85, 104 (8); 6400: 127 (1),
//                         126 (2), 134 (4); 8192: 175, 158, 150 (3), 162 (8); 16384: 459 (1), 358 (2),
//                         307 (5), 313 (8).  From 14336 tiles on, 8 where that leaves a shorter last
//                         group (19 columns of 2^22: 340 against 356 by 5) and 5 where 8 divides the
//                         columns (16 of 2^22: 287 against 307 by 8; 32 of 2^21 282 against 294, inverse 283
//                         against 301; 240 of 2^18 284 against 296).  Where 5 divides too it is as good or
//                         better as well, within a run's noise (whole calls, 5 against 8: 80 of 2^20 629
//                         and 637, inverse 678 and 690; 120 of 2^20 933 and 941, inverse 1019 and 1002; 40
//                         of 2^21 708 and 709, inverse 738 and 751; 640 of 2^17 605 and 600, inverse 623
//                         and 633).  A transform's only pass (short columns) takes 8: 16384 columns of
//                         2^12 354 against 360 by 5.
//   contiguous, at most 8 bits: hardly any set-up.  4 bits: 1613 tiles 38 (1), 45 (2); 2100: 42, 47; 2600: 51,
//                         50; 3200: 64, 68; 4000: 78, 71; 7 bits: 47, 55; 54, 58; 64, 65; 80, 84; 97, 89.  With a
//                         factor per element the set-up is longer, and half as many workgroups run at once: 4
//                         bits, 1536 tiles 50 (1), 55 (2); 1700: 62, 56; 2048: 66, 58; 4096: 124, 109, 119 (3),
//                         110 (8); 8192: 342, 269, 318, 312; 7 bits, 1536 tiles 59, 66; 1700: 74, 68; 8192: 394,
//                         330, 355, 337; 11500: 560, 482, 485, 493; 16384: 796, 680, 680, 668; 8 bits, 1536 tiles
//                         51, 53; 1700: 59, 56.
//   strided, plain top pass: hardly any set-up (one round without twiddles) and HBM-bound:
//                         4 bits 2^26 elements: 180 (1), 189 (8); 5 bits 144 (1), 171 (4); 6 bits 184 (1),
//                         209 (8); 7 bits 204 (1), 199 (2), 213 (8); 8 bits 2^27: 439 (1), 424 (2), 450 (8);
//                         below the top, 6 bits: 198 (1), 181 (3), 191 (8).
//   strided, one factor for every element (n^-1): 4 bits 185 (1), 204 (8); 5 bits 177 (1), 158 (3), 176 (8);
//                         8 bits 257 (1), 242 (2..8).  Few tiles want all the workgroups (whole calls):
//                         6 bits, 384 tiles 33 (1), 41 (3); 1024: 48, 53; 1536: 65, 66; 2048: 79, 79; 8 bits,
//                         768 tiles 43, 50; 1536: 68, 70; 2048: 83, 78.
//   strided, 9 bits, any factor: 8192 tiles 336 (1), 330 (2), 345 (3), 333 (4), 355 (8); 6656: 274, 277,
//                         286, 289, 309; 12288: 491 (1), 477 (2), 473 (4), 485 (8); with a coset 532,
//                         500, 482, 486.
//   strided, a factor per element (coset, gathered coset pass): 16 factors of set-up.  4 bits 263 (1),
//                         252 (4), 272 (8); 5 bits 215 (1), 177 (5), 195 (8); 6 bits 290 (1), 222 (7);
//                         8 bits 341 (1), 256 (7).  At least 768 workgroups: 2^24 elements by 8 bits
//                         77 (3), 72 (5), 80 (8).
static uint32_t pick_reps(bool contig, uint32_t S, bool top, int scale, uint64_t tiles, uint32_t cols,
                          bool only_pass) {
  uint32_t reps;
  if (contig) {
    const uint32_t one = S > 8 ? 1536 : scale == 2 ? 1537 : 2560;  // below that many tiles
    const uint32_t two = S <= 7 && scale == 2 ? 14336 : 7168;
    reps = tiles < one ? 1 : tiles < two ? 2 : tiles < 14336 ? 3 : only_pass || cols % 8 ? 8 : 5;
  } else if (scale && S >= 9) {
    reps = tiles <= 8192 ? 2 : 4;
  } else if (scale == 2) {
    reps = std::min<uint32_t>(S == 4 ? 4 : S == 5 ? 5 : 7, (uint32_t)std::min<uint64_t>(8, tiles / 768));
  } else if (scale == 1) {
    reps = S == 4 || tiles < 2048 ? 1 : 3;
  } else {
    reps = !top ? 3 : S <= 6 ? 1 : 2;
  }
  return std::max(1u, std::min(reps, cols));
}

// Latency-shaped plan (ntt_lat.h): the bits of each pass from the low bits up (a contiguous
// pass of <= 10 bits, then a strided pass of <= 8), or 0 when the size has none.
static int lat_bits(uint32_t log_n, uint32_t *bits) {
  if (log_n < 4 || log_n > 18) return 0;
  if (log_n <= 10) {
    bits[0] = log_n;
    return 1;
  }
  bits[1] = std::min<uint32_t>(8, log_n / 2);
  bits[0] = log_n - bits[1];
  return 2;
}

// BOOJUM_AMD_LAT_MAX_LOG_ELEMS overrides the batch-size bound (read once; 0 turns the latency
// passes off)
static uint32_t lat_max_log_elems() {
  static const uint32_t v = [] {
    const char *e = std::getenv("BOOJUM_AMD_LAT_MAX_LOG_ELEMS");
    return e && *e ? (uint32_t)std::strtoul(e, nullptr, 10) : BA_LAT_MAX_LOG_ELEMS;
  }();
  return v;
}

// Columns that run a whole 2^11- or 2^12-element transform per workgroup (ntt_lat.h): every latency-
// shaped batch of 2^11, which as one launch beats the 4096-element tiles up to 2^21 elements (us per
// call, one launch / two / 4096-element tiles: 1 column 6.6 / 8.5, 256 7.7 / 11.0, 700 13.8 / 23 / 18,
// 2048 28.1 / - / 28.9); of 2^12, whose 1024-thread workgroup is one chain per CU, those that give the
// chip enough of them (1 column 9.5 / 8.5, 64 10.2 / 10.0, 128 10.7 / 11.5, 256 11.6 / 16.1).
static bool wide_columns(uint32_t log_n, uint64_t cols) { return log_n == 11 || (log_n == 12 && cols >= 96); }

bool ba_small_batch(uint64_t cols, uint32_t log_n) {
  const uint32_t m = lat_max_log_elems();
  return m > 0 && (cols << log_n) <= (1ull << std::min(m + (log_n == 11), 40u));
}

bool ba_latency_shape_exists(uint32_t log_n) {
  uint32_t bits[2];
  return lat_bits(log_n, bits) > 0;
}

bool ba_use_latency_passes(const ba_context *ctx, uint32_t log_n, bool n2b, uint32_t num_cols, BaLatPolicy lat) {
  if (lat == BA_LAT_NEVER || !ba_latency_shape_exists(log_n)) return false;
  // a tuned (or caller-set) tile choice for the size class, else the batch-size bound
  const BaTuned &t = ctx->tuned[n2b][log_n];
  if (t.valid && t.tile_log) return t.tile_log == LAT_TL;
  if (lat == BA_LAT_TUNED) return false;
  return ba_small_batch(num_cols, log_n);
}

void ba_scale_factors(uint32_t log_n, bool inverse, uint32_t log_ext, uint32_t coset_idx,
                      uint64_t (&scale_tab)[VALS], uint32_t &coset_mul) {
  coset_mul = log_ext > 0 ? coset_idx << (gl::OMEGA_LOG_ORDER - log_n - log_ext) : 0;
  // T[m] = Delta^m (times n^-1 for the inverse), Delta = s^(+-2^(L-4))
  uint64_t delta = 1;
  if (log_ext > 0 && log_n >= 4) {
    delta = gl_host::pow(gl_host::coset_shift(log_n, log_ext, coset_idx), 1ull << (log_n - 4));
    if (inverse) delta = gl_host::inv(delta);
  }
  uint64_t acc = inverse ? gl_host::inv_pow2(log_n) : 1;
  for (int m = 0; m < VALS; m++) {
    scale_tab[m] = acc;
    if (log_ext > 0) acc = gl_host::mul(acc, delta);
  }
}

int ba_build_ntt(const ba_context *ctx, const uint64_t *in, uint64_t *out, uint32_t log_n,
                 uint32_t num_cols, uint64_t stride_in, uint64_t stride_out, bool bitrev_inputs,
                 bool inverse, uint32_t log_ext, uint32_t coset_idx, bool in_bitrev_gather,
                 std::vector<BaPassLaunch> &launches, BaLatPolicy lat, bool shared, uint32_t cosets) {
  if (num_cols == 0) return BA_SUCCESS;
  const bool n2b = !bitrev_inputs;
  PassArgs base{};
  base.log_n = log_n;
  base.scale_coset = log_ext > 0;
  base.tab = ctx->tab;
  const bool pre = !inverse && log_ext > 0;
  ba_scale_factors(log_n, inverse, log_ext, coset_idx, base.scale_tab, base.coset_mul);

  if (log_n < 4) {
    BaPassLaunch l;
    l.args = base;
    l.args.in = in;
    l.args.out = out;
    l.args.stride_in = stride_in;
    l.args.stride_out = stride_out;
    l.args.num_cols = num_cols;
    l.args.scale = pre ? SCALE_PRE : (inverse ? SCALE_POST : SCALE_NONE);
    l.args.in_bitrev = in_bitrev_gather;
    l.kernels = ba_pick_tiny(log_n, n2b, inverse);
    l.grid = (num_cols + THREADS - 1) / THREADS;
    l.name = tiny_name(log_n, n2b, inverse, false);
    if (in_bitrev_gather) {
      l.coset_kernel = ba_pick_tiny_cosets(log_n);
      l.coset_name = tiny_name(log_n, n2b, inverse, true);
    }
    l.pass = 0;
    l.col0 = 0;
    launches.push_back(l);
    return BA_SUCCESS;
  }

  // an LDE call's coset NTTs: by the elements of all its cosets, unless they have a plan of their own
  // (whose passes are those of 4096-element tiles)
  const BaTuned &of_cosets = ctx->tuned[BA_TUNING_LDE_COSETS][log_n];
  const bool latency = in_bitrev_gather
                           ? lat == BA_LAT_AUTO && (!of_cosets.valid || of_cosets.small_by_size) &&
                                 ba_latency_shape_exists(log_n) && ba_small_batch((uint64_t)num_cols * cosets, log_n)
                           : ba_use_latency_passes(ctx, log_n, n2b, num_cols, lat);
  // single calls only: a batch plan's groups have 256 threads per workgroup
  if (latency && lat == BA_LAT_AUTO && wide_columns(log_n, (uint64_t)num_cols * cosets)) {
    BaPassLaunch l;
    PassArgs &a = l.args;
    a = base;
    a.in = in;
    a.out = out;
    a.stride_in = stride_in;
    a.stride_out = stride_out;
    a.num_cols = num_cols;
    a.reps = 1;
    a.in_canonical = in_bitrev_gather;
    a.in_bitrev = in_bitrev_gather;
    a.scale = pre ? SCALE_PRE : (inverse ? SCALE_POST : SCALE_NONE);
    l.grid = num_cols;
    a.tile_count = num_cols;
    l.threads = (uint32_t)wide_threads((int)log_n);
    l.kernels = {ba_pick_lat_wide(log_n, n2b, inverse, a.scale != SCALE_NONE), nullptr};
    l.name = ba_lat_wide_kernel_name(log_n, n2b, inverse, a.scale != SCALE_NONE);
    if (in_bitrev_gather) {
      l.coset_kernel = ba_pick_lat_wide_cosets(log_n);
      l.coset_name = ba_lat_wide_cosets_kernel_name(log_n);
    }
    l.pass = 0;
    l.col0 = 0;
    launches.push_back(l);
    return BA_SUCCESS;
  }
  if (latency) {
    uint32_t bits[2];
    const int np = lat_bits(log_n, bits);
    for (int p = 0; p < np; p++) {
      const int src = n2b ? np - 1 - p : p;  // n2b: top bits first
      const uint32_t S = bits[src], lo = src == 0 ? 0 : bits[0];
      const bool strided = src > 0, top = lo + S == log_n;
      BaPassLaunch l;
      PassArgs &a = l.args;
      a = base;
      a.in = p == 0 ? in : out;
      a.stride_in = p == 0 ? stride_in : stride_out;
      a.out = out;
      a.stride_out = stride_out;
      a.num_cols = num_cols;
      a.lo_bit = lo;
      a.reps = 1;
      a.in_canonical = p > 0 || in_bitrev_gather;
      a.in_bitrev = in_bitrev_gather && p == 0;
      a.scale = (pre && p == 0) ? SCALE_PRE : ((inverse && p == np - 1) ? SCALE_POST : SCALE_NONE);
      const bool scale = a.scale != SCALE_NONE;
      const uint64_t chunks = (uint64_t)num_cols << (log_n - S);
      l.grid = strided ? ((uint64_t)num_cols << (log_n - LAT_TL))
                       : (chunks + (1u << (LAT_TL - S)) - 1) >> (LAT_TL - S);
      a.tile_count = (uint32_t)l.grid;
      l.kernels = ba_pick_lat(S, strided, n2b, inverse, top, scale);
      if (a.in_bitrev) {
        l.coset_kernel = ba_pick_lat_cosets(S, strided);
        l.coset_name = ba_lat_cosets_kernel_name(S, strided);
      }
      l.name = ba_lat_kernel_name(S, strided, n2b, inverse, strided && top, scale);
      l.pass = p;
      l.col0 = 0;
      if (!l.kernels.single || (a.in_bitrev && !l.coset_kernel)) return BA_ERROR_INVALID_VALUE;
      launches.push_back(l);
    }
    return BA_SUCCESS;
  }

  // The size class's tuned plan, else the built-in one.  An LDE's coset NTTs (the gathered n2b
  // forward) have their own entry, timed on that transform: a plan tuned on plain NTTs does not
  // carry over (the gathered, scaled first pass has other costs; it has no 9- or 10-bit variant).
  const int kind = in_bitrev_gather ? BA_TUNING_LDE_COSETS : (n2b ? 1 : 0);
  const BaTuned &tuning = ctx->tuned[kind][log_n].valid ? ctx->tuned[kind][log_n] : BaTuned{};
  const NttPlan plan = tuning.valid ? tuning.plan : ba_plan_ntt(log_n, n2b, in_bitrev_gather);
  for (int p = 0; p < plan.num_passes; p++) {
    const uint32_t S = plan.bits[p];
    const bool contig = plan.contig[p];
    // tiles: L >= 12 -> 2^(L-12) per column, repeats stride over columns;
    //        L < 12  -> 2^(12-L) columns per tile (contiguous pass only), repeats adjacent
    const bool big = log_n >= (uint32_t)TILE_LOG;
    const uint32_t log_stride = big ? log_n - TILE_LOG : 0;
    const uint32_t cols_per_tile = big ? 1 : (1u << (TILE_LOG - log_n));
    // launch column groups small enough for 32-bit tile counts and grids
    const uint64_t max_cols = (big ? std::max<uint64_t>(1, (kMaxGrid >> log_stride)) : kMaxGrid) / cosets;
    for (uint64_t c0 = 0; c0 < num_cols; c0 += max_cols) {
      const uint32_t nc = (uint32_t)std::min<uint64_t>(max_cols, num_cols - c0);
      const uint64_t tiles = big ? ((uint64_t)nc << log_stride) : (nc + cols_per_tile - 1) / cols_per_tile;
      BaPassLaunch l;
      PassArgs &a = l.args;
      a = base;
      a.in = p == 0 ? in + c0 * stride_in : out + c0 * stride_out;
      a.stride_in = p == 0 ? stride_in : stride_out;
      a.out = out + c0 * stride_out;
      a.stride_out = stride_out;
      a.num_cols = nc;
      a.lo_bit = plan.lo_bit[p];
      a.tile_count = (uint32_t)tiles;
      a.log_tile_stride = log_stride;
      a.scale = (pre && p == 0) ? SCALE_PRE
                                : ((inverse && p == plan.num_passes - 1) ? SCALE_POST : SCALE_NONE);
      a.in_bitrev = in_bitrev_gather && p == 0;
      // later passes read this transform's own output, and the gathered LDE coset pass reads the
      // monomials the inverse NTT wrote: values < p
      a.in_canonical = p > 0 || in_bitrev_gather;
      const bool top = plan.lo_bit[p] + S == log_n;
      const int scale = a.scale == SCALE_NONE ? 0 : (a.scale_coset ? 2 : 1);
      const uint32_t tuned_reps = tuning.valid ? tuning.reps[p] : 0;
      const uint32_t most = big ? nc : (uint32_t)tiles;
      a.reps = std::max(1u, tuned_reps ? std::min(tuned_reps, most)
                                       : pick_reps(contig, S, top, scale, tiles * cosets, most, log_n == S));
      const uint64_t groups = big ? (nc + a.reps - 1) / a.reps : (tiles + a.reps - 1) / a.reps;
      l.grid = groups << log_stride;
      const bool gather = !contig && a.in_bitrev;
      // the 9..12-bit contiguous pass: as tuned, else 4 waves per SIMD.  (The three-waves build with its
      // prefetch takes as long on up to 512 tiles, 18 and 22 us, and longer above: 34.6 against 29.9 us
      // on 1024 tiles, 146 against 127 on 6400.)
      const uint32_t waves = S < 9 ? 3 : tuning.valid && tuning.contig_waves ? tuning.contig_waves : 4;
      l.kernels = pick_kernel(contig, S, n2b, inverse, top, scale, big, gather, waves, shared);
      const bool shared_build =
          shared && !contig && l.kernels.group != pick_kernel(contig, S, n2b, inverse, top, scale, big, gather, waves, false).group;
      l.name = kernel_name(contig, S, n2b, inverse, contig ? big : top, scale, gather, waves, shared_build);
      if (a.in_bitrev) {
        l.coset_kernel = !contig      ? ba_pick_strided_cosets(S)
                         : S <= 8     ? ba_pick_contig_lo_cosets(S)
                         : waves == 3 ? ba_pick_contig_hi3_cosets(S)
                                      : ba_pick_contig_hi_cosets(S);
        l.coset_name = coset_name(contig, S, waves);
      }
      l.pass = p;
      l.col0 = c0;
      if (!l.kernels.group || (a.in_bitrev && !l.coset_kernel)) return BA_ERROR_INVALID_VALUE;
      launches.push_back(l);
    }
  }
  return BA_SUCCESS;
}

int ba_run_launches(const std::vector<BaPassLaunch> &launches, hipStream_t stream) {
  for (const BaPassLaunch &l : launches) {
    ba_trace_before(stream, l.name);
    hipLaunchKernelGGL(l.kernels.single, dim3((uint32_t)l.grid), dim3(l.threads), 0, stream, l.args);
    ba_trace_after(stream);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return (int)err;
  }
  return BA_SUCCESS;
}

int ba_launch_ntt(const ba_context *ctx, const uint64_t *in, uint64_t *out, uint32_t log_n,
                  uint32_t num_cols, uint64_t stride_in, uint64_t stride_out, bool bitrev_inputs,
                  bool inverse, uint32_t log_ext, uint32_t coset_idx, hipStream_t stream) {
  std::vector<BaPassLaunch> launches;
  const int rc = ba_build_ntt(ctx, in, out, log_n, num_cols, stride_in, stride_out, bitrev_inputs,
                              inverse, log_ext, coset_idx, false, launches, BA_LAT_AUTO);
  if (rc) return rc;
  return ba_run_launches(launches, stream);
}

int ba_validate_ntt(uint32_t log_n, uint64_t stride_in, uint64_t stride_out, uint32_t log_ext,
                    uint32_t coset_idx) {
  // ntt.rs:192-200; in addition a column holds at most 2^28 elements (the reference's plans
  // stop at 2^24, ntt.rs:74-169, and index past them for larger sizes)
  if (log_n < 1 || log_n > BA_MAX_LOG_N || log_n + log_ext > gl::OMEGA_LOG_ORDER)
    return BA_ERROR_INVALID_VALUE;
  const uint64_t n = 1ull << log_n;
  if (n > stride_in || n > stride_out) return BA_ERROR_INVALID_VALUE;
  if (coset_idx > 0 && (log_ext == 0 || coset_idx >= (1u << log_ext))) return BA_ERROR_INVALID_VALUE;
  return BA_SUCCESS;
}

extern "C" int ba_batch_ntt_ctx(ba_context_t ctx, const uint64_t *inputs, uint64_t *outputs,
                                uint32_t log_n, uint32_t num_ntts, uint64_t stride_in,
                                uint64_t stride_out, int bitrev_inputs, int inverse,
                                uint32_t log_extension_degree, uint32_t coset_index,
                                ba_stream_t stream) {
  return ba_guarded([&]() -> int {
    if (!ctx) return BA_ERROR_NOT_INITIALIZED;
    int rc = ba_validate_ntt(log_n, stride_in, stride_out, log_extension_degree, coset_index);
    if (rc) return rc;
    if (num_ntts && (!inputs || !outputs)) return BA_ERROR_INVALID_VALUE;
    return ba_launch_ntt(ctx, inputs, outputs, log_n, num_ntts, stride_in, stride_out,
                         bitrev_inputs != 0, inverse != 0, log_extension_degree, coset_index,
                         (hipStream_t)stream);
  });
}

extern "C" int ba_batch_ntt_internal(const uint64_t *inputs, uint64_t *outputs, uint32_t log_n,
                                     uint32_t num_ntts, uint32_t stride_between_input_arrays,
                                     uint32_t stride_between_output_arrays, int bitrev_inputs,
                                     int inverse, uint32_t log_extension_degree,
                                     uint32_t coset_index, ba_stream_t stream) {
  return ba_guarded([&]() -> int {
    return ba_batch_ntt_ctx(ba_context_for_current_device(), inputs, outputs, log_n, num_ntts,
                            stride_between_input_arrays, stride_between_output_arrays,
                            bitrev_inputs, inverse, log_extension_degree, coset_index, stream);
  });
}

extern "C" int ba_batch_ntt_out_of_place(const uint64_t *inputs_matrix, size_t inputs_len,
                                         uint64_t *outputs_matrix, size_t outputs_len,
                                         uint32_t log_n, uint32_t num_ntts, uint32_t inputs_offset,
                                         uint32_t outputs_offset,
                                         uint32_t stride_between_input_arrays,
                                         uint32_t stride_between_output_arrays, int bitrev_inputs,
                                         int inverse, uint32_t log_extension_degree,
                                         uint32_t coset_index, ba_stream_t stream) {
  return ba_guarded([&]() -> int {
    // ntt.rs:309-320, with 64-bit arithmetic in place of the reference's u32 products
    if (log_n < 1 || log_n > BA_MAX_LOG_N) return BA_ERROR_INVALID_VALUE;
    const uint64_t n = 1ull << log_n;
    if ((uint64_t)inputs_offset + n > stride_between_input_arrays) return BA_ERROR_INVALID_VALUE;
    if ((uint64_t)outputs_offset + n > stride_between_output_arrays) return BA_ERROR_INVALID_VALUE;
    if ((uint64_t)inputs_len < (uint64_t)num_ntts * stride_between_input_arrays) return BA_ERROR_INVALID_VALUE;
    if ((uint64_t)outputs_len < (uint64_t)num_ntts * stride_between_output_arrays) return BA_ERROR_INVALID_VALUE;
    // the reference's slices are distinct borrows (ntt.rs:317,320): no overlap at all
    if (inputs_len && outputs_len && inputs_matrix < outputs_matrix + outputs_len &&
        outputs_matrix < inputs_matrix + inputs_len)
      return BA_ERROR_INVALID_VALUE;
    const uint64_t *in = inputs_matrix + inputs_offset;
    uint64_t *out = outputs_matrix + outputs_offset;
    if ((const void *)in == (const void *)out) return BA_ERROR_INVALID_VALUE;
    return ba_batch_ntt_internal(in, out, log_n, num_ntts, stride_between_input_arrays,
                                 stride_between_output_arrays, bitrev_inputs, inverse,
                                 log_extension_degree, coset_index, stream);
  });
}

extern "C" int ba_batch_ntt_in_place(uint64_t *inputs_matrix, size_t inputs_len, uint32_t log_n,
                                     uint32_t num_ntts, uint32_t inputs_offset,
                                     uint32_t stride_between_input_arrays, int bitrev_inputs,
                                     int inverse, uint32_t log_extension_degree,
                                     uint32_t coset_index, ba_stream_t stream) {
  return ba_guarded([&]() -> int {
    // ntt.rs:350-352
    if (log_n < 1 || log_n > BA_MAX_LOG_N) return BA_ERROR_INVALID_VALUE;
    const uint64_t n = 1ull << log_n;
    if ((uint64_t)inputs_offset + n > stride_between_input_arrays) return BA_ERROR_INVALID_VALUE;
    if ((uint64_t)inputs_len < (uint64_t)num_ntts * stride_between_input_arrays) return BA_ERROR_INVALID_VALUE;
    uint64_t *io = inputs_matrix + inputs_offset;
    return ba_batch_ntt_internal(io, io, log_n, num_ntts, stride_between_input_arrays,
                                 stride_between_input_arrays, bitrev_inputs, inverse,
                                 log_extension_degree, coset_index, stream);
  });
}
