// ntt_lat.hip -- instantiations of the latency-shaped NTT passes (see ntt_lat.h) and their
// kernel names for launch tracing.
#include <cstdio>

#include "ntt_inst.h"
#include "ntt_lat.h"

using namespace gl::ntt;

template <int S, bool N2B, bool INV, bool STRIDED, bool TOP, bool SCALE>
static BaKernels one() {
  return {ntt_pass_lat<S, N2B, INV, STRIDED, TOP, SCALE>, ntt_pass_lat_group<S, N2B, INV, STRIDED, TOP, SCALE>};
}

template <int S, bool N2B, bool INV>
static BaKernels pick3(bool strided, bool top, bool scale) {
  if (!strided) {
    if constexpr (S >= BA_LAT_MIN_CONTIG && S <= BA_LAT_MAX_CONTIG)
      return scale ? one<S, N2B, INV, false, false, true>() : one<S, N2B, INV, false, false, false>();
  } else {
    if constexpr (S >= BA_LAT_MIN_STRIDED && S <= BA_LAT_MAX_STRIDED) {
      if (!top) return scale ? BaKernels{nullptr, nullptr} : one<S, N2B, INV, true, false, false>();
      return scale ? one<S, N2B, INV, true, true, true>() : one<S, N2B, INV, true, true, false>();
    }
  }
  return {nullptr, nullptr};
}

template <int S>
static BaKernels pick(bool strided, bool n2b, bool inverse, bool top, bool scale) {
  if (n2b) return inverse ? pick3<S, true, true>(strided, top, scale) : pick3<S, true, false>(strided, top, scale);
  return inverse ? pick3<S, false, true>(strided, top, scale) : pick3<S, false, false>(strided, top, scale);
}

BaKernels ba_pick_lat(uint32_t S, bool strided, bool n2b, bool inverse, bool top, bool scale) {
  switch (S) {
    case 4: return pick<4>(strided, n2b, inverse, top, scale);
    case 5: return pick<5>(strided, n2b, inverse, top, scale);
    case 6: return pick<6>(strided, n2b, inverse, top, scale);
    case 7: return pick<7>(strided, n2b, inverse, top, scale);
    case 8: return pick<8>(strided, n2b, inverse, top, scale);
    case 9: return pick<9>(strided, n2b, inverse, top, scale);
    case 10: return pick<10>(strided, n2b, inverse, top, scale);
  }
  return {nullptr, nullptr};
}

template <int S>
static BaCosetKernel pick_cosets(bool strided) {
  if (strided) {
    if constexpr (S >= BA_LAT_MIN_STRIDED && S <= BA_LAT_MAX_STRIDED) return ntt_pass_lat_cosets<S, true>;
  } else {
    if constexpr (S >= BA_LAT_MIN_CONTIG && S <= BA_LAT_MAX_CONTIG) return ntt_pass_lat_cosets<S, false>;
  }
  return nullptr;
}

BaCosetKernel ba_pick_lat_cosets(uint32_t S, bool strided) {
  switch (S) {
    case 4: return pick_cosets<4>(strided);
    case 5: return pick_cosets<5>(strided);
    case 6: return pick_cosets<6>(strided);
    case 7: return pick_cosets<7>(strided);
    case 8: return pick_cosets<8>(strided);
    case 9: return pick_cosets<9>(strided);
    case 10: return pick_cosets<10>(strided);
  }
  return nullptr;
}

template <int S, bool N2B, bool INV>
static BaPassKernel wide(bool scale) {
  return scale ? ntt_pass_lat_wide<S, N2B, INV, true> : ntt_pass_lat_wide<S, N2B, INV, false>;
}
template <int S>
static BaPassKernel wide(bool n2b, bool inverse, bool scale) {
  if (n2b) return inverse ? wide<S, true, true>(scale) : wide<S, true, false>(scale);
  return inverse ? wide<S, false, true>(scale) : wide<S, false, false>(scale);
}

BaPassKernel ba_pick_lat_wide(uint32_t S, bool n2b, bool inverse, bool scale) {
  return S == 11 ? wide<11>(n2b, inverse, scale) : S == 12 ? wide<12>(n2b, inverse, scale) : nullptr;
}
BaCosetKernel ba_pick_lat_wide_cosets(uint32_t S) {
  return S == 11 ? ntt_pass_lat_wide_cosets<11> : S == 12 ? ntt_pass_lat_wide_cosets<12> : nullptr;
}

namespace {
// as rocprofv3 prints them; built by the first caller (a function-local static initialiser, so
// concurrent first calls are safe)
struct LatNames {
  char n[11][2][2][2][2][2][100];  // [S][n2b][inverse][strided][top][scale]
  char cosets[11][2][80];          // [S][strided]
  char wide[2][2][2][2][80];       // [S - 11][n2b][inverse][scale]
  char wide_cosets[2][80];         // [S - 11]
  LatNames() {
    static const char *tf[2] = {"false", "true"};
    for (int s = 0; s < 11; s++)
      for (int d = 0; d < 2; d++)
        for (int i = 0; i < 2; i++)
          for (int st = 0; st < 2; st++)
            for (int tp = 0; tp < 2; tp++)
              for (int sc = 0; sc < 2; sc++)
                snprintf(n[s][d][i][st][tp][sc], sizeof(n[s][d][i][st][tp][sc]),
                         "void gl::ntt::ntt_pass_lat<%d, %s, %s, %s, %s, %s>(gl::ntt::PassArgs)", s, tf[d], tf[i],
                         tf[st], tf[tp], tf[sc]);
    for (int s = 0; s < 11; s++)
      for (int st = 0; st < 2; st++)
        snprintf(cosets[s][st], sizeof(cosets[s][st]), "void gl::ntt::ntt_pass_lat_cosets<%d, %s>(gl::ntt::CosetArgs)",
                 s, tf[st]);
    for (int s = 0; s < 2; s++) {
      for (int d = 0; d < 2; d++)
        for (int i = 0; i < 2; i++)
          for (int sc = 0; sc < 2; sc++)
            snprintf(wide[s][d][i][sc], sizeof(wide[s][d][i][sc]),
                     "void gl::ntt::ntt_pass_lat_wide<%d, %s, %s, %s>(gl::ntt::PassArgs)", s + 11, tf[d], tf[i], tf[sc]);
      snprintf(wide_cosets[s], sizeof(wide_cosets[s]), "void gl::ntt::ntt_pass_lat_wide_cosets<%d>(gl::ntt::CosetArgs)",
               s + 11);
    }
  }
};
const LatNames &lat_names() {
  static const LatNames names;
  return names;
}
}  // namespace

const char *ba_lat_kernel_name(uint32_t S, bool strided, bool n2b, bool inverse, bool top, bool scale) {
  return S <= 10 ? lat_names().n[S][n2b][inverse][strided][top][scale] : "ntt_pass_lat";
}
const char *ba_lat_cosets_kernel_name(uint32_t S, bool strided) {
  return S <= 10 ? lat_names().cosets[S][strided] : "ntt_pass_lat_cosets";
}
const char *ba_lat_wide_kernel_name(uint32_t S, bool n2b, bool inverse, bool scale) {
  return S == 11 || S == 12 ? lat_names().wide[S - 11][n2b][inverse][scale] : "ntt_pass_lat_wide";
}
const char *ba_lat_wide_cosets_kernel_name(uint32_t S) {
  return S == 11 || S == 12 ? lat_names().wide_cosets[S - 11] : "ntt_pass_lat_wide_cosets";
}
