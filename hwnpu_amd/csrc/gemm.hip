// Prefill / verify GEMM (K3) on gfx950: the kernels of hwk_i8_gemm and hwk_mxfp4_gemm and the choice
// of tile shape (the device code is in gemm_kernels.h).
#include "gemm_kernels.h"
#include "hwk_common.h"

namespace {

using namespace hwk_gemm;

template <int BM, int BN, bool MX, int WM, int WN, int KG>
__global__ __launch_bounds__(64 * WM * WN * KG) __attribute__((amdgpu_waves_per_eu(MX && WM * WN * KG == 4 ? 2 : 1))) void k_gemm(
    const u32x4 *__restrict__ X, const uint8_t *__restrict__ W, const uint8_t *__restrict__ E,
    const uint16_t *__restrict__ S, void *__restrict__ Y, uint32_t M, uint32_t N, uint32_t K, int mode, bool equads) {
  __shared__ __attribute__((aligned(16))) u32x4 lds[2 * BM * CH];
  gemm_wg<BM, BN, MX, WM, WN, KG>(blockIdx.x, X, W, E, S, Y, M, N, K, mode, equads, lds);
}

// Up to 16 waves a CU: as many registers as that leaves a wave.
template <int BM, int BN, bool MX, int WM, int WN, int KG, int RS, int RES>
__global__ __launch_bounds__(64 * WM * WN * KG) __attribute__((amdgpu_waves_per_eu(WM * WN * KG * RES / 4))) void k_gemm_pair(
    const u32x4 *__restrict__ X, const uint8_t *__restrict__ W, const uint8_t *__restrict__ E,
    const uint16_t *__restrict__ S, void *__restrict__ Y, uint32_t M, uint32_t N, uint32_t K, int mode, bool equads) {
  __shared__ __attribute__((aligned(16))) u32x4 lds[PairCfg<BM, BN, MX, WM, WN, KG, RS>::LDS];
  gemm_pair_wg<BM, BN, MX, WM, WN, KG, RS>(blockIdx.x, X, W, E, S, Y, M, N, K, mode, equads, lds);
}

// The general form's tile shape for (m, n): the fewest rounds of workgroups over the CUs, a round weighted by the
// tile's work and its per-tile overheads (larger tiles reuse their loads more). When every tile
// gets a CU of its own, 8 waves (2 x 4, two a SIMD: one computes while the other waits) beat 4 by
// 5-12 % on the prompt's shapes; with several tiles a CU, 4-wave workgroups fill the SIMDs as well.
// An int8 tile of 2 x 2 waves can be doubled into two k groups (8 waves) instead: its SIMDs then
// split the tile's k, which lets a smaller tile use 8 waves (128 x 96 fills the 256 CUs at 512 x 6144).
struct Shape {
  int bm, bn, wm, wn, kg;  // tile, waves over its rows and columns, k groups
};
constexpr Shape kShapes[] = {{128, 128, 2, 2, 1}, {128, 96, 2, 2, 1}, {128, 64, 2, 2, 1}, {64, 128, 2, 2, 1},
                             {128, 128, 2, 4, 1}, {128, 64, 2, 4, 1}, {128, 96, 2, 2, 2}};
Shape pick_shape(uint32_t m, uint32_t n, int cus, bool mx) {
  Shape best = kShapes[0];
  double best_cost = 1e300;
  for (const Shape &s : kShapes) {
    if (mx && s.kg != 1) continue;
    const uint64_t tiles = (uint64_t)((m + s.bm - 1) / s.bm) * ((n + s.bn - 1) / s.bn);
    const uint64_t rounds = (tiles + cus - 1) / cus;
    const bool eight = s.wm * s.wn * s.kg == 8;
    if (eight && tiles > (uint64_t)cus) continue;
    const double cost = (double)rounds * s.bm * s.bn * (1.0 + 32.0 / s.bm + 32.0 / s.bn) * (eight ? 0.75 : 1.0);
    if (cost < best_cost) {
      best_cost = cost;
      best = s;
    }
  }
  return best;
}

int device_cus() {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) !=
                                              hipSuccess || cus <= 0)
    cus = 256;
  return cus;
}

template <bool MX>
char *launch(hipStream_t st, const void *x, const void *w, const void *e, const void *s, void *y, uint32_t m,
             uint32_t n, uint32_t k, int mode, const char *what) {
  const bool equads = MX && (k / 32) % 16 == 0 && hwk::aligned(e, 16);
  const u32x4 *X = (const u32x4 *)x;
  const uint8_t *W = (const uint8_t *)w, *E = (const uint8_t *)e;
  const uint16_t *S = (const uint16_t *)s;
  if (pair_takes(MX, m, n, k, e)) {
    int i = pick_pair(MX, m, n, k);
#define HWK_PAIR(BM, BN, WM, WN, KG, RS, RES, PS)                                                                  \
  if (i-- == 0) {                                                                                                  \
    const uint32_t tiles = ((m + BM - 1) / BM) * ((n + BN - 1) / BN);                                              \
    hipLaunchKernelGGL((k_gemm_pair<BM, BN, MX, WM, WN, KG, RS, RES>), dim3(pair_grid(tiles)), dim3(64 * WM * WN * KG), \
                       0, st, X, W, E, S, y, m, n, k, mode, equads);                                               \
    return hwk::launched(what);                                                                                    \
  }
    if constexpr (MX) {
      HWK_PAIR_MX(HWK_PAIR)
    } else {
      HWK_PAIR_I8(HWK_PAIR)
    }
#undef HWK_PAIR
    HWK_CHECK(false, "%s: no kernel for %ux%ux%u", what, m, n, k);
  }
  static const int cus = device_cus();
  const Shape sh = pick_shape(m, n, cus, MX);
  const dim3 grid(((m + sh.bm - 1) / sh.bm) * ((n + sh.bn - 1) / sh.bn));
#define HWK_GEMM_IF(BMv, BNv, WMv, WNv, KGv)                                                                   \
  if (sh.bm == BMv && sh.bn == BNv && sh.wm == WMv && sh.wn == WNv && sh.kg == KGv)                               \
    hipLaunchKernelGGL((k_gemm<BMv, BNv, MX, WMv, WNv, KGv>), grid, dim3(64 * WMv * WNv * KGv), 0, st, X, W, E, S, \
                       y, m, n, k, mode, equads);                                                                 \
  else
  HWK_GEMM_IF(128, 128, 2, 2, 1)
  HWK_GEMM_IF(128, 96, 2, 2, 1)
  HWK_GEMM_IF(128, 64, 2, 2, 1)
  HWK_GEMM_IF(64, 128, 2, 2, 1)
  HWK_GEMM_IF(128, 128, 2, 4, 1)
  HWK_GEMM_IF(128, 64, 2, 4, 1)
  if constexpr (!MX) {
    HWK_GEMM_IF(128, 96, 2, 2, 2)
    HWK_CHECK(false, "%s: no kernel for the %dx%d tile", what, sh.bm, sh.bn);
  } else {
    HWK_CHECK(false, "%s: no kernel for the %dx%d tile", what, sh.bm, sh.bn);
  }
#undef HWK_GEMM_IF
  return hwk::launched(what);
}

}  // namespace

extern "C" {

HWK_API char *hwk_i8_gemm(void *stream, const void *x, const void *q, const void *scale16, void *y, uint32_t m,
                          uint32_t n, uint32_t k, int out_mode) {
  HWK_CHECK(x && q && scale16 && y, "hwk_i8_gemm: null pointer");
  HWK_CHECK(k % 32 == 0 && k > 0, "hwk_i8_gemm: k=%u is not a positive multiple of 32", k);
  HWK_CHECK(out_mode >= HWK_OUT_F32 && out_mode <= HWK_OUT_SWIGLU_F16, "hwk_i8_gemm: out_mode %d", out_mode);
  HWK_CHECK(out_mode != HWK_OUT_SWIGLU_F16 || n % 16 == 0, "hwk_i8_gemm: SwiGLU output needs n %% 16 == 0 (n=%u)", n);
  HWK_CHECK(hwk::aligned(x, 16) && hwk::aligned(q, 16), "hwk_i8_gemm: x and q must be 16-byte aligned");
  if (m == 0 || n == 0) return nullptr;
  return launch<false>((hipStream_t)stream, x, q, nullptr, scale16, y, m, n, k, out_mode, "hwk_i8_gemm");
}

HWK_API char *hwk_mxfp4_gemm(void *stream, const void *x, const void *w, const void *e, void *y, uint32_t m,
                             uint32_t n, uint32_t k, int out_mode) {
  HWK_CHECK(x && w && e && y, "hwk_mxfp4_gemm: null pointer");
  HWK_CHECK(k % 32 == 0 && k > 0, "hwk_mxfp4_gemm: k=%u is not a positive multiple of 32", k);
  HWK_CHECK(out_mode >= HWK_OUT_F32 && out_mode <= HWK_OUT_SWIGLU_F16, "hwk_mxfp4_gemm: out_mode %d", out_mode);
  HWK_CHECK(out_mode != HWK_OUT_SWIGLU_F16 || n % 16 == 0, "hwk_mxfp4_gemm: SwiGLU output needs n %% 16 == 0 (n=%u)", n);
  HWK_CHECK(hwk::aligned(x, 16) && hwk::aligned(w, 16), "hwk_mxfp4_gemm: x and w must be 16-byte aligned");
  if (m == 0 || n == 0) return nullptr;
  return launch<true>((hipStream_t)stream, x, w, e, nullptr, y, m, n, k, out_mode, "hwk_mxfp4_gemm");
}

}  // extern "C"
