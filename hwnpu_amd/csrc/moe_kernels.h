// The device code of the MoE path (K5a routing, K5b experts), shared by libhwk's kernels (moe.hip) and
// the kernels of the library's code object (co/hwk_co.hip), so that both run the same instructions.
//
// MoE on gfx950: the router's top-k choice (K5a) and the chosen experts' gated FFNs (K5b).
//
// K5a restates the reference's Routing.Choose operation for operation (float64 exp rounded to
// float32, a sequential float32 sum, a stable descending order) in one wave per token with lane j
// holding expert j, so that the chosen expert ids are the reference's bit for bit.
//
// K5b is two launches and needs nothing from the host between them. The gate_up kernel gives each
// (chosen expert, row-pair tile) to a workgroup: with the route folded in (hwk_moe_layer) every
// workgroup derives the tokens' choice from the router logits itself (read off the logits' order
// where that provably equals Choose's, so that its weight loads issue before Choose has run, in a
// workgroup of its own that writes idx and w; else by Choose first); otherwise it reads the given
// idx. It reads the expert's rows once for all tokens that chose it, adds the gate/up biases,
// and writes the gated unit (SiLU, or gpt-oss's clamped one) in fp32 (it overflows fp16 at the
// benchmark's scales). The down kernel gives each workgroup a tile of output rows for every chosen
// expert (its waves take the experts in turn, all their rows' loads issued at once) and then adds,
// for each token, w * (y + down bias) in ascending expert id, the reference's summation order
// (host.go:566-578,866-881), with no atomics.
#pragma once

#include "hwk_common.h"

namespace hwk_moe {


// ---- K5a ----

// A lane's float as a wave-uniform value (v_readlane: no LDS round trip).
__device__ __forceinline__ float lane_f(float v, uint32_t j) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), (int)j));
}

// Routing.Choose (internal/llm/experts/weights.go:33-81) of one row of E <= 64 logits by one wave,
// lane j holding expert j, reading other lanes' values with v_readlane only (no LDS, no barrier):
// softmax scores in float32 (exp in float64 rounded to float32, the sum taken in expert order), or
// sigmoid; the rank of each expert in a stable descending sort of score + bias (ties to the lower
// index); the first k (idx, w) with w the chosen scores over their float32 sum + 1e-6 (norm), times
// scale unless 0. Lanes < k write idx_out/w_out.
__device__ void choose_wave(const float *__restrict__ logits, const float *__restrict__ bias, uint32_t E, uint32_t k,
                            int score, int norm, float scale, int32_t *idx_out, float *w_out) {
#pragma clang fp contract(off)
  const uint32_t lane = threadIdx.x & 63;
  const bool live = lane < E;
  const float v = live ? logits[lane] : -__builtin_inff();
  const float bl = bias && live ? bias[lane] : 0.0f;
  float s;
  if (score == HWK_SCORE_SOFTMAX) {
    const float m = group_max_dpp<64>(v);
    const float ex = live ? (float)exp((double)(v - m)) : 0.0f;
    float total = 0.0f;
    for (uint32_t j = 0; j < E; j++) total += lane_f(ex, j);
    s = ex / total;
  } else {
    s = 1.0f / (1.0f + (float)exp((double)(-v)));
  }
  const float kv = bias && live ? s + bl : s;
  uint32_t rank = 0;
  for (uint32_t j = 0; j < E; j++) {
    const float kj = lane_f(kv, j);
    rank += (kj > kv) || (kj == kv && j < lane);
  }
  // the k chosen in rank order: lane r learns the expert of rank r and its score
  int my_e = -1;
  float my_w = 0.0f, sum = 0.0f;
  for (uint32_t r = 0; r < k; r++) {
    const uint64_t who = __ballot(live && rank == r);
    const uint32_t src = who ? (uint32_t)__builtin_ctzll(who) : 0u;  // no such rank only with NaN scores
    const float wr = lane_f(s, src);
    sum += wr;
    if (lane == r) {
      my_e = (int)src;
      my_w = wr;
    }
  }
  if (lane < k) {
    float wj = my_w;
    if (norm) wj /= sum + 1e-6f;
    if (scale != 0.0f) wj *= scale;
    idx_out[lane] = my_e;
    w_out[lane] = wj;
  }
}

// Routing.Choose's choice of one token read off the logits alone, where that provably gives Choose's experts
// in Choose's order (softmax scores, no bias): the k largest in turn (a wave maximum each), ties to the lower
// index. With d = logit - max (the float32 difference Choose exponentiates; softmax is monotone in it) the
// choice is Choose's when the d of consecutive ranks 0 .. min(k, E-1) differ by at least 2^-20 (their
// float64 exps then differ by a factor above 1 + 9.5e-7, so their float32 roundings, and the roundings of
// those over the same sum, differ: a float32 rounding moves a value by at most 2^-24 of it) and the last
// chosen has d >= -80 (every chosen score a normal float32). Returns that (wave-uniform) and writes the
// choice in rank order to ch[0, k).
__device__ __forceinline__ bool choice_of_logits(const float *__restrict__ logits, uint32_t E, uint32_t k, int32_t *ch) {
  const uint32_t lane = threadIdx.x & 63;
  float v = lane < E ? logits[lane] : -__builtin_inff();
  bool ok = !__ballot(v != v);
  float top = 0.0f, prev = 0.0f;
  for (uint32_t r = 0; r <= k && r < E; r++) {
    const float m = group_max_dpp<64>(v);
    const uint64_t who = __ballot(v == m);
    const uint32_t src = who ? (uint32_t)__builtin_ctzll(who) : 0u;  // (none only with NaN logits)
    if (r == 0) top = m;
    const float d = m - top;  // NaN for an infinite top: every comparison below then fails
    ok = ok && (r == 0 ? d == 0.0f : prev - d >= 0x1p-20f) && (r + 1 != k || d >= -80.0f);
    prev = d;
    if (r < k && lane == 0) ch[r] = (int32_t)src;
    if (lane == src) v = -__builtin_inff();
  }
  return ok;
}

// ---- K5b helpers ----

// The choice as each lane holds it: lane j < n (n = T*k) the expert of (token, slot) j, -1 for an id outside
// [0, E) and in the lanes past n.
__device__ __forceinline__ int lane_choice(const int32_t *idx, uint32_t n, uint32_t E) {
  const uint32_t lane = threadIdx.x & 63;
  const int e = lane < n ? idx[lane] : -1;
  return (uint32_t)e < E ? e : -1;
}

// The set of the experts chosen, from lane_choice.
__device__ __forceinline__ uint64_t chosen_set(int my, uint32_t n) {
  uint64_t set = 0;
  for (uint32_t j = 0; j < n; j++) {
    const int e = __builtin_amdgcn_readlane(my, (int)j);
    set |= e >= 0 ? 1ull << e : 0ull;
  }
  return set;
}

// The u-th expert of a set with more than u, by ascending id.
__device__ __forceinline__ int expert_at(uint64_t set, uint32_t u) {
  for (uint32_t i = 0; i < u; i++) set &= set - 1;
  return __builtin_ctzll(set);
}

// PPW (gate, up) pairs' row sums at once: v[p] holds pair p's partial sums, the gate's in lanes 0..31 and
// the up's in lanes 32..63. Each step adds a lane and its partner and, while there are pairs left, leaves
// half the lanes to each of two pairs, so that all pairs take little more than one sum (and the sum's order
// is the same for any PPW). Lane L ends with the sum of pair pair_of_lane(L), gate for L < 32.
template <int PPW>
__device__ __forceinline__ uint32_t pair_of_lane(uint32_t lane) {
  return ((lane >> 4) & 1) + (PPW >= 4 ? 2 * ((lane >> 3) & 1) : 0);
}
template <int PPW>
__device__ __forceinline__ float pair_sums(float (&v)[PPW]) {
  static_assert(PPW == 2 || PPW == 4, "pairs a wave");
  const uint32_t lane = threadIdx.x & 63;
  float a[PPW / 2];
#pragma unroll
  for (int i = 0; i < PPW / 2; i++) {
    swap_rows16(v[2 * i], v[2 * i + 1]);  // rows of 16: (first, second, first, second) of both pairs
    a[i] = v[2 * i] + v[2 * i + 1];
  }
  float s;
  if constexpr (PPW == 4) {
    const float x = lane & 8 ? a[1] : a[0], y = lane & 8 ? a[0] : a[1];
    s = x + HWK_DPP_ALL(y, 0x128);  // row_ror:8
  } else {
    s = a[0] + HWK_DPP_ALL(a[0], 0x128);
  }
  s += HWK_DPP_ALL(s, 0x141);  // row_half_mirror
  s += HWK_DPP_ALL(s, 0x4e);  // quad_perm [2, 3, 0, 1]
  s += HWK_DPP_ALL(s, 0xb1);  // quad_perm [1, 0, 3, 2]
  return s;
}

// c as it stands at this point: the compiler cannot move its conversions out of the loop over the tokens around
// it (a block's 32 converted values take four times its registers, which then spill).
__device__ __forceinline__ void keep_codes(uint4 &c) { asm volatile("" : "+v"(c.x), "+v"(c.y), "+v"(c.z), "+v"(c.w)); }

// sum over a 32-value block: codes (16 bytes) as fp16 pairs against x in fp16 pairs (v_dot2)
__device__ __forceinline__ float dot_block_f16(uint4 c, const uint4 (&x)[4]) {
  const uint32_t cw[4] = {c.x, c.y, c.z, c.w};
  float d0 = 0.0f, d1 = 0.0f;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    d0 = __builtin_amdgcn_fdot2(fp4x2_to_h2<0>(cw[q]), h2_of_bits(x[q].x), d0, false);
    d1 = __builtin_amdgcn_fdot2(fp4x2_to_h2<1>(cw[q]), h2_of_bits(x[q].y), d1, false);
    d0 = __builtin_amdgcn_fdot2(fp4x2_to_h2<2>(cw[q]), h2_of_bits(x[q].z), d0, false);
    d1 = __builtin_amdgcn_fdot2(fp4x2_to_h2<3>(cw[q]), h2_of_bits(x[q].w), d1, false);
  }
  return d0 + d1;
}

// the same against fp32 activations a[32] (mixed-precision multiply-adds)
__device__ __forceinline__ float dot_block_f32(uint4 c, const float4 (&a)[8]) {
  const uint32_t cw[4] = {c.x, c.y, c.z, c.w};
  float d0 = 0.0f, d1 = 0.0f;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const h2 p0 = fp4x2_to_h2<0>(cw[q]), p1 = fp4x2_to_h2<1>(cw[q]);
    const h2 p2 = fp4x2_to_h2<2>(cw[q]), p3 = fp4x2_to_h2<3>(cw[q]);
    const float4 a0 = a[2 * q], a1 = a[2 * q + 1];
    d0 = fmaf((float)p0.x, a0.x, d0);
    d1 = fmaf((float)p0.y, a0.y, d1);
    d0 = fmaf((float)p1.x, a0.z, d0);
    d1 = fmaf((float)p1.y, a0.w, d1);
    d0 = fmaf((float)p2.x, a1.x, d0);
    d1 = fmaf((float)p2.y, a1.y, d1);
    d0 = fmaf((float)p3.x, a1.z, d0);
    d1 = fmaf((float)p3.y, a1.w, d1);
  }
  return d0 + d1;
}

// ---- K5b stage 1: route (optional), gate_up + bias, the gated unit ----

constexpr uint32_t kMoeSpan = 8;
__host__ __device__ __forceinline__ uint32_t gate_up_wgs(uint32_t I, uint32_t pairs) { return (I + pairs - 1) / pairs; }

struct MoeArgs {
  uint32_t T, H, I, E, k;
  int act;  // HWK_ACT_SILU or HWK_ACT_GPTOSS
  int score, norm;
  float alpha, limit, scale;
  int mode;  // out_mode of the down stage
  uint32_t span;  // row-pair tiles of a gate_up workgroup, at most kMoeSpan
};

// The gated unit of one (gate, up) pair (host.go:516-527): SiLU g/(1+e^-g)*u, or gpt-oss's
// min(g, L)/(1+e^(-a*min(g, L))) * (clamp(u, -L, L) + 1), exp in float64 rounded to float32, every
// other step a float32 operation of its own.
__device__ __forceinline__ float gated(float g, float u, const MoeArgs &a) {
#pragma clang fp contract(off)
  if (a.act == HWK_ACT_GPTOSS) {
    g = fminf(g, a.limit);
    u = fminf(fmaxf(u, -a.limit), a.limit);
    return g / (1.0f + (float)exp((double)(-(a.alpha * g)))) * (u + 1.0f);
  }
  return g / (1.0f + (float)exp((double)(-g))) * u;
}

// A token's x in LDS: whole 1 KB loads, the four 16-byte chunks of block b in the order q ^ (b/4 & 3), so that one
// chunk of 16 neighbouring blocks fills the banks.
__host__ __device__ __forceinline__ uint32_t x_bytes(uint32_t H) { return (H * 2 + 1023) / 1024 * 1024; }

// Workgroup (a.span row-pair tiles of 4*PPW pairs from tile bx*a.span on, chosen expert number by in ascending
// id), PPW pairs (gate row 2j, up row 2j+1) a wave and tile. LPR lanes a row: 32 (the wave's halves take a pair's
// gate and up row) or 64 (each row in turn), BPL blocks a lane (nb = H/32 <= LPR*BPL). ROUTE: the workgroup reads
// every token's choice off the logits (waves over tokens), and a column of workgroups of its own runs Choose for
// idx and w; where the logits do not settle the choice, every workgroup runs Choose first, and workgroup (0, 0)
// writes idx and w. Else idx is given. The row sums meet in LDS and the gated unit, an exp in float64 and the
// longest stretch of the vector ALUs a result, runs once a workgroup with full lanes. xs: LDS for the x of the
// tokens that chose the expert, x_bytes each (all T may).
// Bound by the vector ALUs once a few tokens share an expert, and by the choice, the weights' latency and the
// gated unit in turn below that: 5 tokens of hidden 2048, 32 experts, k = 4, I = 768 took 17 µs with x from
// memory, the choice launched before it and the gated unit in each wave, and take 13; 8 tokens of hidden 2880,
// I = 2880, 142 and 65.
template <int LPR, int BPL, int PPW, bool ROUTE>
__device__ __forceinline__ void moe_gate_up_wg(uint32_t bx, uint32_t by, const uint4 *__restrict__ x,
                                               const float *__restrict__ logits, const float *__restrict__ rbias,
                                               int32_t *__restrict__ idx, float *__restrict__ wout,
                                               const uint4 *__restrict__ gw, const uint8_t *__restrict__ ge,
                                               const float *__restrict__ gb, float *__restrict__ act, MoeArgs a,
                                               char *xs) {
  static_assert(LPR == 32 || LPR == 64, "lanes a row");
  constexpr int RR = LPR / 32;  // rows of a pair in turn
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t n = a.T * a.k;
  if (ROUTE && bx == gate_up_wgs(a.I, 4 * PPW * a.span) && by > 0) return;
  int my;
  if constexpr (ROUTE) {
    __shared__ int32_t sidx[64];
    __shared__ float sw[64];
    __shared__ uint32_t sure[4];
    bool spec = !rbias && a.score == HWK_SCORE_SOFTMAX;
    if (spec) {
      bool ok = true;
      for (uint32_t t = wave; t < a.T; t += 4)
        ok = choice_of_logits(logits + (size_t)t * a.E, a.E, a.k, sidx + t * a.k) && ok;
      if (lane == 0) sure[wave] = ok;
      __syncthreads();
      spec = sure[0] && sure[1] && sure[2] && sure[3];
    }
    if (bx == gate_up_wgs(a.I, 4 * PPW * a.span)) {
      // the route's own workgroup (one column past the experts' tiles): Choose's idx and w, beside the experts'
      // loads; without the logits' choice the experts' workgroups route themselves
      if (spec)
        for (uint32_t t = wave; t < a.T; t += 4)
          choose_wave(logits + (size_t)t * a.E, rbias, a.E, a.k, a.score, a.norm, a.scale, idx + t * a.k,
                      wout + t * a.k);
      return;
    }
    if (!spec) {
      __syncthreads();  // every wave is done with the logits' choice
      for (uint32_t t = wave; t < a.T; t += 4)
        choose_wave(logits + (size_t)t * a.E, rbias, a.E, a.k, a.score, a.norm, a.scale, sidx + t * a.k,
                    sw + t * a.k);
      __syncthreads();
      if (bx == 0 && by == 0 && threadIdx.x < n) {
        idx[threadIdx.x] = sidx[threadIdx.x];
        wout[threadIdx.x] = sw[threadIdx.x];
      }
    }
    my = lane_choice(sidx, n, a.E);
  } else {
    my = lane_choice(idx, n, a.E);
  }
  const uint64_t set = chosen_set(my, n);
  if (by >= (uint32_t)__builtin_popcountll(set)) return;
  const int e = expert_at(set, by);
  uint64_t who = __ballot(my == e);  // the (token, slot)s that chose it
  const uint32_t nb = a.H / 32, I = a.I, l = lane % LPR;
  const uint32_t xrow = x_bytes(a.H);
  const size_t erow = (size_t)e * 2 * I;  // the expert's first row
  __shared__ float2 sums[kMoeSpan * 4 * PPW * 8];  // (gate, up) of (token, tile, pair); a token chooses once
  const uint32_t spanned = a.span * 4 * PPW;      // pairs of the workgroup
  // x of the tokens, the j-th of them from LDS byte j * xrow on; each wave a quarter of a row's loads
  uint64_t slots = 0;  // the first slot of each token that chose e
  for (uint64_t m = who; m; m &= m - 1)
    if (!slots || (uint32_t)__builtin_ctzll(m) / a.k != (63 - (uint32_t)__builtin_clzll(slots)) / a.k)
      slots |= m & -m;
  const uint32_t cols = (uint32_t)__builtin_popcountll(slots), xl = lds_at(xs);
  for (uint32_t tile = 0; tile < a.span; tile++) {
    const uint32_t pair0 = ((bx * a.span + tile) * 4 + wave) * PPW;
    // every load issued unconditionally from a clamped row / block (a load under a branch is waited
    // for where the branches join): terms of blocks past nb are dropped, rows past I not written
    uint4 c[PPW][RR][BPL];
    uint32_t s[PPW][RR][BPL];
#pragma unroll
    for (int p = 0; p < PPW; p++)
#pragma unroll
      for (int r = 0; r < RR; r++)
#pragma unroll
        for (int j = 0; j < BPL; j++) {
          const uint32_t pair = min(pair0 + p, I - 1), b = min((uint32_t)(j * LPR) + l, nb - 1);
          const size_t blk = (erow + 2 * pair + (RR == 2 ? (uint32_t)r : lane >> 5)) * nb + b;
          c[p][r][j] = load_stream(&gw[blk]);
          s[p][r][j] = ge[blk];
        }
    if (tile == 0) {
      issue_order();
      uint32_t row = xl;
      for (uint64_t m = slots; m; m &= m - 1, row += xrow) {
        const uint32_t t = (uint32_t)__builtin_ctzll(m) / a.k;
        for (uint32_t o = __builtin_amdgcn_readfirstlane(wave) * 1024; o < nb * 64; o += 4096) {
          const uint32_t ch = o / 16 + lane;
          to_lds16(x, t * nb * 64 + min(((ch & ~3u) | ((ch ^ ch >> 4) & 3)) * 16, nb * 64 - 16), row + o);
        }
      }
      wait_loads<0>();  // the weights and the wave's part of x
      __syncthreads();
    }
    for (uint32_t col = 0; col < cols; col++) {
#pragma unroll
      for (int p = 0; p < PPW; p++)
#pragma unroll
        for (int r = 0; r < RR; r++)
#pragma unroll
          for (int j = 0; j < BPL; j++) keep_codes(c[p][r][j]);
      uint4 xr[BPL][4];
#pragma unroll
      for (int j = 0; j < BPL; j++) {
        const uint32_t b = min((uint32_t)(j * LPR) + l, nb - 1);
#pragma unroll
        for (uint32_t q = 0; q < 4; q++) xr[j][q] = *(const uint4 *)(xs + col * xrow + b * 64 + (q ^ (b >> 2 & 3)) * 16);
      }
      float v[PPW];
#pragma unroll
      for (int p = 0; p < PPW; p++) {
        float gu[RR];
#pragma unroll
        for (int r = 0; r < RR; r++) {
          gu[r] = 0.0f;
#pragma unroll
          for (int j = 0; j < BPL; j++) {
            const float term = dot_block_f16(c[p][r][j], xr[j]) * e8m0_scale(s[p][r][j]);
            gu[r] += (uint32_t)(j * LPR) + l < nb ? term : 0.0f;
          }
        }
        if constexpr (RR == 2) {
          swap_rows32(gu[0], gu[1]);  // (gate's, up's) lower halves and upper halves
          v[p] = gu[0] + gu[1];
        } else {
          v[p] = gu[0];
        }
      }
      const float y = pair_sums<PPW>(v);
      if ((lane & (PPW == 4 ? 7 : 15)) == 0)  // a gate in lanes below 32, the up in those from it on
        ((float *)&sums[col * spanned + tile * 4 * PPW + wave * PPW + pair_of_lane<PPW>(lane)])[lane >> 5] = y;
    }
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < cols * spanned; i += 256) {
    const uint32_t col = i / spanned, pair = bx * spanned + i % spanned;
    uint64_t m = slots;
    for (uint32_t j = 0; j < col; j++) m &= m - 1;
    if (pair < I) {
      const float *pb = gb + erow + 2 * pair;
      act[(size_t)__builtin_ctzll(m) * I + pair] =
          gb ? gated(sums[i].x + pb[0], sums[i].y + pb[1], a) : gated(sums[i].x, sums[i].y, a);
    }
  }
}

// ---- K5b stage 2: down for every chosen expert, then the ordered combine ----

// Workgroup: RS = R * 64/LPR output rows, NW waves; wave wv takes the chosen experts u = wv, wv+NW, ...
// (ascending id), R row sets of 64/LPR rows with LPR lanes a row and BPL blocks a lane (nb = I/32 <=
// LPR*BPL), all loads of an expert's rows issued at once, each read once for every token that chose it. The
// activations (fp32) of each (token, slot) go into LDS of the wave's own, whole lines straight from memory
// with 16-byte chunk q of block b at chunk q ^ (b & 7), so that the reads of 8 lanes (one block each, the same
// chunk) fall in distinct banks; a lane's blocks are the same in all R row sets. Each expert's unweighted y is
// kept in LDS by (token slot, row); then one thread a (token, row) adds w * (y + down bias) over the token's
// experts in ascending expert id.
// Bound by the weights' latency and the LDS reads of the activations: 5 tokens of the sizes above 8 µs (10 with
// the activations of all tokens copied by every workgroup through registers), 8 tokens of 2880 x 2880 49 (115).
template <int LPR, int BPL, int R, int NW>
struct DownCfg {
  static constexpr uint32_t kActs = LPR * BPL * 128;  // bytes of one (token, slot)'s activations
  static constexpr int kBufs = 2 * NW * kActs <= 128 * 1024 ? 2 : 1;  // the next one's loads under this one's products
};
template <int LPR, int BPL, int R, int NW>
__device__ __forceinline__ void moe_down_wg(uint32_t bx, const float *__restrict__ act, const int32_t *__restrict__ idx,
                                            const float *__restrict__ w, const uint4 *__restrict__ dw,
                                            const uint8_t *__restrict__ de, const float *__restrict__ db,
                                            float *__restrict__ out, MoeArgs a) {
  using C = DownCfg<LPR, BPL, R, NW>;
  constexpr int SR = 64 / LPR, RS = R * SR;
  __shared__ __attribute__((aligned(16))) char acts[NW * C::kBufs * C::kActs];
  __shared__ float ys[64 * RS];   // (token slot, row)
  __shared__ int32_t order[64];   // (token, rank): the slot of the token's rank-th expert by id, -1 past its last
  __shared__ float sw[64];
  const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = lane % LPR;
  const uint32_t n = a.T * a.k, H = a.H, nb = a.I / 32;
  const int my = lane_choice(idx, n, a.E);
  const float mw = wave == 0 && lane < n ? w[lane] : 0.0f;
  const uint64_t set = chosen_set(my, n);
  const uint32_t U = (uint32_t)__builtin_popcountll(set);
  const uint32_t row0 = bx * RS;
  const uint32_t lds0 = lds_at(acts) + wave * C::kBufs * C::kActs;
  // the lane's source of load i: unit p = 64 i + lane holds chunk (p % 8) ^ (block & 7) of block p / 8
  auto stage = [&](uint32_t slot, uint32_t buf) __attribute__((always_inline)) {
    const float *src = act + (size_t)slot * a.I;
#pragma unroll
    for (int i = 0; i < LPR * BPL / 8; i++) {
      const uint32_t blk = min((uint32_t)i * 8 + (lane >> 3), nb - 1), ch = (lane & 7) ^ ((lane >> 3) & 7);
      to_lds16(src, blk * 128 + ch * 16, lds0 + buf * C::kActs + i * 1024);
    }
  };
  for (uint32_t u = wave; u < U; u += NW) {
    const int e = expert_at(set, u);
    uint64_t who = __ballot(my == e);
    uint4 c[R][BPL];
    uint32_t sc[R][BPL];
    // every load issued unconditionally (a load under a branch is waited for where the branches join):
    // rows past H and blocks past nb read the last one, their terms are dropped
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
      for (int j = 0; j < BPL; j++) {
        const uint32_t row = min(row0 + r * SR + lane / LPR, H - 1), b = min((uint32_t)(j * LPR) + l, nb - 1);
        const size_t blk = ((size_t)e * H + row) * nb + b;
        c[r][j] = load_stream(&dw[blk]);
        sc[r][j] = de[blk];
      }
    issue_order();
    uint32_t buf = 0;
    stage((uint32_t)__builtin_ctzll(who), 0);
    while (who) {
      const uint32_t slot = (uint32_t)__builtin_ctzll(who);
      who &= who - 1;
      wait_loads<0>();  // the weights and this slot's activations
      issue_order();
      if (C::kBufs == 2 && who) stage((uint32_t)__builtin_ctzll(who), buf ^ 1);
      const char *av0 = acts + (wave * C::kBufs + buf) * C::kActs;
      float v[R];
#pragma unroll
      for (int r = 0; r < R; r++) v[r] = 0.0f;
#pragma unroll
      for (int j = 0; j < BPL; j++) {
        const uint32_t b = (uint32_t)(j * LPR) + l;
        float4 av[8];
#pragma unroll
        for (int q = 0; q < 8; q++) av[q] = *(const float4 *)(av0 + b * 128 + (((uint32_t)q ^ (b & 7)) * 16));
#pragma unroll
        for (int r = 0; r < R; r++) {
          keep_codes(c[r][j]);
          const float term = dot_block_f32(c[r][j], av) * e8m0_scale(sc[r][j]);
          v[r] += b < nb ? term : 0.0f;
        }
      }
#pragma unroll
      for (int r = 0; r < R; r++) {
        const float y = group_sum<LPR>(v[r]);
        if (l == 0) ys[slot * RS + r * SR + lane / LPR] = y;
      }
      if (C::kBufs == 1 && who) {
        wait_lds();  // this slot's reads done
        stage((uint32_t)__builtin_ctzll(who), 0);
      }
      if (C::kBufs == 2) buf ^= 1;
    }
    wait_lds();  // the reads done before the next expert's loads
  }
  if (wave == 0) {
    // the slots of each token by ascending expert id (ids outside [0, E) and repeated ids left out)
    const uint32_t t = lane / a.k;
    uint32_t rank = 0;
    bool first = my >= 0;
    for (uint32_t j = 0; j < n; j++) {
      const int e = __builtin_amdgcn_readlane(my, (int)j);
      const bool same = j / a.k == t && e >= 0;
      const bool repeat = (__ballot(lane < j && lane / a.k == j / a.k && my == e) != 0);  // an earlier slot's expert
      rank += same && !repeat && e < my;
      if (lane == j) first = first && !repeat;
    }
    if (lane < n) order[lane] = -1;
    if (lane < n && first) order[t * a.k + rank] = (int32_t)lane;
    sw[lane] = mw;
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < a.T * RS; i += 64 * NW) {
#pragma clang fp contract(off)
    const uint32_t t = i / RS, r = i % RS, orow = row0 + r;
    if (orow >= H) continue;
    float acc = a.mode == HWK_OUT_ADD_F32 ? out[(size_t)t * H + orow] : 0.0f;
    for (uint32_t q = 0; q < a.k; q++) {
      const int slot = order[t * a.k + q];
      if (slot < 0) break;
      const float bias = db ? db[(size_t)idx[slot] * H + orow] : 0.0f;
      acc += sw[slot] * (ys[slot * RS + r] + bias);
    }
    out[(size_t)t * H + orow] = acc;
  }
}

}  // namespace hwk_moe
