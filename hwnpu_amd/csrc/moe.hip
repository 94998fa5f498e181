// MoE on gfx950: the kernels of hwk_moe_route, hwk_moe_experts and hwk_moe_layer and their launch
// choices (the device code is in moe_kernels.h).
#include <atomic>

#include "hwk_common.h"
#include "moe_kernels.h"

#define HWK_Q(call)                  \
  do {                               \
    if (char *e_ = (call)) return e_; \
  } while (0)

namespace {

using namespace hwk_moe;

// hwk_moe_route: one wave a row.
__global__ __launch_bounds__(256) void k_moe_route(const float *__restrict__ logits, const float *__restrict__ bias,
                                                   int32_t *__restrict__ idx, float *__restrict__ w, uint32_t rows,
                                                   uint32_t E, uint32_t k, int score, int norm, float scale) {
  const uint32_t row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  choose_wave(logits + (size_t)row * E, bias, E, k, score, norm, scale, idx + (size_t)row * k, w + (size_t)row * k);
}

template <int LPR, int BPL, int PPW, bool ROUTE>
__global__ __launch_bounds__(256) void k_moe_gate_up(const uint4 *__restrict__ x, const float *__restrict__ logits,
                                                     const float *__restrict__ rbias, int32_t *__restrict__ idx,
                                                     float *__restrict__ wout, const uint4 *__restrict__ gw,
                                                     const uint8_t *__restrict__ ge, const float *__restrict__ gb,
                                                     float *__restrict__ act, MoeArgs a) {
  extern __shared__ __attribute__((aligned(16))) char xs[];
  moe_gate_up_wg<LPR, BPL, PPW, ROUTE>(blockIdx.x, blockIdx.y, x, logits, rbias, idx, wout, gw, ge, gb, act, a, xs);
}

template <int LPR, int BPL, int R, int NW>
__global__ __launch_bounds__(64 * NW) void k_moe_down(const float *__restrict__ act, const int32_t *__restrict__ idx,
                                                      const float *__restrict__ w, const uint4 *__restrict__ dw,
                                                      const uint8_t *__restrict__ de, const float *__restrict__ db,
                                                      float *__restrict__ out, MoeArgs a) {
  moe_down_wg<LPR, BPL, R, NW>(blockIdx.x, act, idx, w, dw, de, db, out, a);
}

// The waves of a down workgroup, by the most experts chosen: a wave an expert, up to 8 while the staged
// activations fit 128 KB of LDS; 16 for short rows while the grid is one workgroup a CU (a layer of 5 tokens:
// 21.4 µs, with 8 waves 22.8; of 3: 15.3 and 16.8).
template <int LPR, int BPL, int R>
void launch_down(hipStream_t st, const float *act, const int32_t *idx, const float *w, const void *dw, const void *de,
                 const float *db, float *out, const MoeArgs &a) {
  constexpr int RS = R * 64 / LPR;
  const dim3 grid((a.H + RS - 1) / RS);
  const uint32_t n = a.T * a.k < a.E ? a.T * a.k : a.E;
#define HWK_DN(NW)                                                                                             \
  hipLaunchKernelGGL((k_moe_down<LPR, BPL, R, NW>), grid, dim3(64 * NW), 0, st, act, idx, w, (const uint4 *)dw, \
                     (const uint8_t *)de, db, out, a)
  if constexpr (LPR == 8) {
    if (n > 8 && a.H <= 256 * RS) {
      HWK_DN(16);
      return;
    }
  }
  if constexpr (DownCfg<LPR, BPL, R, 8>::kActs * 8 <= 128 * 1024) {
    if (n > 4) {
      HWK_DN(8);
      return;
    }
  }
  HWK_DN(4);
#undef HWK_DN
}

char *check_params(const char *what, const hwk_moe_params *p) {
  HWK_CHECK(p, "%s: null params", what);
  HWK_CHECK(p->tokens >= 1 && p->tokens <= 8, "%s: %u tokens (1..8)", what, p->tokens);
  HWK_CHECK(p->experts >= 1 && p->experts <= 64, "%s: %u experts (1..64)", what, p->experts);
  HWK_CHECK(p->k >= 1 && p->k <= p->experts && p->tokens * p->k <= 64, "%s: k=%u", what, p->k);
  HWK_CHECK(p->hidden % 32 == 0 && p->hidden > 0 && p->hidden <= 8192, "%s: hidden %u", what, p->hidden);
  HWK_CHECK(p->inter % 32 == 0 && p->inter > 0 && p->inter <= 8192, "%s: inter %u", what, p->inter);
  HWK_CHECK(p->out_mode == HWK_OUT_F32 || p->out_mode == HWK_OUT_ADD_F32, "%s: out_mode %u", what, p->out_mode);
  HWK_CHECK(p->act == HWK_ACT_SILU || p->act == HWK_ACT_GPTOSS, "%s: act %u", what, p->act);
  return nullptr;
}

MoeArgs args_of(const hwk_moe_params *p) {
  MoeArgs a;
  a.T = p->tokens;
  a.H = p->hidden;
  a.I = p->inter;
  a.E = p->experts;
  a.k = p->k;
  a.act = (int)p->act;
  a.alpha = hwk::f32_of_bits(p->alpha_bits);
  a.limit = hwk::f32_of_bits(p->limit_bits);
  a.score = (int)p->score;
  a.norm = (int)p->norm;
  a.scale = hwk::f32_of_bits(p->scale_bits);
  a.mode = (int)p->out_mode;
  a.span = 1;
  return a;
}

// Allows a kernel its dynamic LDS past 64 KB on the current device (done: the kernel's devices so far, a bit each).
char *allow_lds(const void *kernel, std::atomic<uint64_t> &done) {
  int dev = 0;
  HWK_TRY("hipGetDevice", hipGetDevice(&dev));
  const uint64_t bit = dev < 64 ? 1ull << dev : 0;
  if (done.load(std::memory_order_relaxed) & bit) return nullptr;
  HWK_TRY("hwk_moe (LDS)", hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024));
  done.fetch_or(bit, std::memory_order_relaxed);
  return nullptr;
}

template <int PPW, bool ROUTE>
char *launch_gate_up(hipStream_t st, const void *x, const float *logits, const float *rbias, int32_t *idx, float *w,
                    const void *gu_w, const void *gu_e, const float *gu_b, float *act, MoeArgs a) {
  const uint32_t unique_max = a.T * a.k < a.E ? a.T * a.k : a.E, nb = a.H / 32;
  // tiles a workgroup: one until the grid has twice what the chip holds (four workgroups a CU), then as many as
  // leave that, so that the choice, x and the gated unit are shared by more rows (a layer of 8 tokens of 64
  // experts at k = 8, I = 1,408: 110 µs with one tile a workgroup, 74 with 8; goals of 512 and 2,048: 74 and 83)
  const uint32_t wgs = gate_up_wgs(a.I, 4 * PPW) * unique_max, goal = 4 * 256;
  a.span = wgs < 2 * goal ? 1 : wgs / goal < kMoeSpan ? wgs / goal : kMoeSpan;
  // with the route folded in, one more column of workgroups: the route's own (moe_gate_up_wg)
  const dim3 g1(gate_up_wgs(a.I, 4 * PPW * a.span) + (ROUTE ? 1 : 0), unique_max);
  const uint32_t lds = a.T * x_bytes(a.H);  // 8 tokens of H = 8,192 take 128 KB
#define HWK_GU(L, B)                                                                                              \
  do {                                                                                                            \
    static std::atomic<uint64_t> done{0};                                                                         \
    if (lds > 64 * 1024) HWK_Q(allow_lds((const void *)k_moe_gate_up<L, B, PPW, ROUTE>, done));                   \
    hipLaunchKernelGGL((k_moe_gate_up<L, B, PPW, ROUTE>), g1, dim3(256), lds, st, (const uint4 *)x, logits, rbias, \
                       idx, w, (const uint4 *)gu_w, (const uint8_t *)gu_e, gu_b, act, a);                         \
  } while (0)
  // lanes a row: 32 up to H = 4,096 (a row sum is then half the steps, and one load takes gate and up)
  if (nb <= 32) HWK_GU(32, 1);
  else if (nb <= 64) HWK_GU(32, 2);
  else if (nb <= 96) HWK_GU(32, 3);
  else if (nb <= 128) HWK_GU(32, 4);
  else if (nb <= 192) HWK_GU(64, 3);
  else HWK_GU(64, 4);
#undef HWK_GU
  return nullptr;
}

// K5b: gate_up (with the route folded in when ROUTE), then down with the ordered combine.
template <bool ROUTE>
char *run_experts(hipStream_t st, const void *x, const float *logits, const float *rbias, int32_t *idx, float *w,
                  const void *gu_w, const void *gu_e, const float *gu_b, const void *dn_w, const void *dn_e,
                  const float *dn_b, float *out, float *act, const MoeArgs &a, const char *what) {
  if (a.T <= 2) HWK_Q((launch_gate_up<2, ROUTE>(st, x, logits, rbias, idx, w, gu_w, gu_e, gu_b, act, a)));
  else HWK_Q((launch_gate_up<4, ROUTE>(st, x, logits, rbias, idx, w, gu_w, gu_e, gu_b, act, a)));
  if (char *err = hwk::launched(what)) return err;
  // down: lanes a row by I/32 blocks, the fewest idle slots (8 lanes x 3 blocks for I = 768), and row sets enough
  // that a workgroup has 8 rows to share the staged activations; 2 rows up to H = 512, where 8 leave most CUs idle
  // (a layer of H = 256, I = 3,200, 1 token: 8.0 µs, with 8 rows 9.6; 8 tokens on 3 experts 34 and 46; at H = 768 2
  // rows lose, 8 tokens of I = 6,144 0.46 against 0.38 of the time before)
  const uint32_t nbi = a.I / 32;
  const bool narrow = a.H <= 512;
  if (nbi <= 8) launch_down<8, 1, 1>(st, act, idx, w, dn_w, dn_e, dn_b, out, a);
  else if (nbi <= 16) launch_down<8, 2, 1>(st, act, idx, w, dn_w, dn_e, dn_b, out, a);
  else if (nbi <= 24) launch_down<8, 3, 1>(st, act, idx, w, dn_w, dn_e, dn_b, out, a);
  else if (nbi <= 32) launch_down<16, 2, 2>(st, act, idx, w, dn_w, dn_e, dn_b, out, a);
  else if (nbi <= 48) launch_down<16, 3, 2>(st, act, idx, w, dn_w, dn_e, dn_b, out, a);
  else if (nbi <= 64 && narrow) launch_down<32, 2, 1>(st, act, idx, w, dn_w, dn_e, dn_b, out, a);
  else if (nbi <= 64) launch_down<32, 2, 4>(st, act, idx, w, dn_w, dn_e, dn_b, out, a);
  else if (nbi <= 96 && narrow) launch_down<32, 3, 1>(st, act, idx, w, dn_w, dn_e, dn_b, out, a);
  else if (nbi <= 96) launch_down<32, 3, 4>(st, act, idx, w, dn_w, dn_e, dn_b, out, a);
  else if (nbi <= 128 && narrow) launch_down<64, 2, 2>(st, act, idx, w, dn_w, dn_e, dn_b, out, a);
  else if (nbi <= 128) launch_down<64, 2, 8>(st, act, idx, w, dn_w, dn_e, dn_b, out, a);
  else if (nbi <= 192 && narrow) launch_down<64, 3, 2>(st, act, idx, w, dn_w, dn_e, dn_b, out, a);
  else if (nbi <= 192) launch_down<64, 3, 4>(st, act, idx, w, dn_w, dn_e, dn_b, out, a);
  else if (narrow) launch_down<64, 4, 2>(st, act, idx, w, dn_w, dn_e, dn_b, out, a);
  else launch_down<64, 4, 4>(st, act, idx, w, dn_w, dn_e, dn_b, out, a);
  return hwk::launched(what);
}

// Whether hwk_moe_layer folds the route into the gate_up launch: up to 2 tokens always, and up to 5 where the
// choice can be read off the logits (k wave maxima a token and wave; Choose in every workgroup costs more than
// the launch it saves). A layer of 3, 4, 5, 6 and 8 tokens folded against a route launch, µs: 15.3 and 18.2,
// 22.9 and 26.6 (k = 8 of 64), 21.4 and 22.8, 43.4 and 43.3 (k = 8), 30.9 and 28.7.
bool folds_route(const hwk_moe_params *p, const void *router_bias) {
  return p->tokens <= 2 || (p->tokens <= 5 && p->score == HWK_SCORE_SOFTMAX && !router_bias);
}

}  // namespace

extern "C" {

HWK_API char *hwk_moe_route(void *stream, const void *logits, const void *bias, void *idx, void *w, uint32_t rows,
                            uint32_t experts, uint32_t k, int score, int norm, uint32_t scale_bits) {
  HWK_CHECK(logits && idx && w, "hwk_moe_route: null pointer");
  HWK_CHECK(experts >= 1 && experts <= 64, "hwk_moe_route: %u experts (1..64)", experts);
  HWK_CHECK(k >= 1 && k <= experts, "hwk_moe_route: k=%u of %u experts", k, experts);
  HWK_CHECK(score == HWK_SCORE_SOFTMAX || score == HWK_SCORE_SIGMOID, "hwk_moe_route: score %d", score);
  if (rows == 0) return nullptr;
  hipLaunchKernelGGL(k_moe_route, dim3((rows + 3) / 4), dim3(256), 0, (hipStream_t)stream, (const float *)logits,
                     (const float *)bias, (int32_t *)idx, (float *)w, rows, experts, k, score, norm,
                     hwk::f32_of_bits(scale_bits));
  return hwk::launched("hwk_moe_route");
}

// Layout: act (tokens, k, I) fp32.
HWK_API size_t hwk_moe_workspace_bytes(const hwk_moe_params *p) {
  if (!p) return 0;
  return (size_t)p->tokens * p->k * p->inter * sizeof(float);
}

HWK_API char *hwk_moe_experts(void *stream, const void *x, const void *idx, const void *w, const void *gu_w,
                              const void *gu_e, const void *gu_b, const void *dn_w, const void *dn_e,
                              const void *dn_b, void *out, void *workspace, size_t workspace_bytes,
                              const hwk_moe_params *p) {
  HWK_Q(check_params("hwk_moe_experts", p));
  HWK_CHECK(x && idx && w && gu_w && gu_e && dn_w && dn_e && out && workspace, "hwk_moe_experts: null pointer");
  HWK_CHECK(hwk::aligned(x, 16) && hwk::aligned(gu_w, 16) && hwk::aligned(dn_w, 16) && hwk::aligned(workspace, 16),
            "hwk_moe_experts: x, weights and workspace must be 16-byte aligned");
  HWK_CHECK(workspace_bytes >= hwk_moe_workspace_bytes(p), "hwk_moe_experts: workspace %zu bytes, %zu needed",
            workspace_bytes, hwk_moe_workspace_bytes(p));
  return run_experts<false>((hipStream_t)stream, x, nullptr, nullptr, (int32_t *)idx, (float *)w, gu_w, gu_e,
                            (const float *)gu_b, dn_w, dn_e, (const float *)dn_b, (float *)out, (float *)workspace,
                            args_of(p), "hwk_moe_experts");
}

HWK_API char *hwk_moe_layer(void *stream, const void *x, const void *logits, const void *router_bias, void *idx,
                            void *w, const void *gu_w, const void *gu_e, const void *gu_b, const void *dn_w,
                            const void *dn_e, const void *dn_b, void *out, void *workspace, size_t workspace_bytes,
                            const hwk_moe_params *p) {
  HWK_Q(check_params("hwk_moe_layer", p));
  HWK_CHECK(x && logits && idx && w && gu_w && gu_e && dn_w && dn_e && out && workspace,
            "hwk_moe_layer: null pointer");
  HWK_CHECK(p->score == HWK_SCORE_SOFTMAX || p->score == HWK_SCORE_SIGMOID, "hwk_moe_layer: score %u", p->score);
  HWK_CHECK(hwk::aligned(x, 16) && hwk::aligned(gu_w, 16) && hwk::aligned(dn_w, 16) && hwk::aligned(workspace, 16),
            "hwk_moe_layer: x, weights and workspace must be 16-byte aligned");
  HWK_CHECK(workspace_bytes >= hwk_moe_workspace_bytes(p), "hwk_moe_layer: workspace %zu bytes, %zu needed",
            workspace_bytes, hwk_moe_workspace_bytes(p));
  const MoeArgs a = args_of(p);
  hipStream_t st = (hipStream_t)stream;
  if (folds_route(p, router_bias))
    return run_experts<true>(st, x, (const float *)logits, (const float *)router_bias, (int32_t *)idx, (float *)w,
                             gu_w, gu_e, (const float *)gu_b, dn_w, dn_e, (const float *)dn_b, (float *)out,
                             (float *)workspace, a, "hwk_moe_layer");
  hipLaunchKernelGGL(k_moe_route, dim3((p->tokens + 3) / 4), dim3(256), 0, st, (const float *)logits,
                     (const float *)router_bias, (int32_t *)idx, (float *)w, p->tokens, p->experts, p->k,
                     (int)p->score, (int)p->norm, a.scale);
  HWK_Q(hwk::launched("hwk_moe_layer (route)"));
  return run_experts<false>(st, x, nullptr, nullptr, (int32_t *)idx, (float *)w, gu_w, gu_e, (const float *)gu_b,
                            dn_w, dn_e, (const float *)dn_b, (float *)out, (float *)workspace, a, "hwk_moe_layer");
}

}  // extern "C"
