// Causal attention of a prompt (prefill) on gfx950: T query rows at positions start .. start+T-1
// per head over an fp16 KV cache that already holds their keys, GQA (head j on kv head
// j/(heads/kv_heads)). This is the prompt form of the reference's per-chunk program with its
// causal mask (internal/llm/paged/paged.go:70-203 at tokens > 1, internal/llm/blocks/blocks.go:
// 516-540): every query sees the keys at or before its own position.
//
// The query rows of a kv head are its (position, query head) pairs, in that order; a workgroup takes 64 of
// them (16 a wave, four waves) and a chunk of the keys they see, in tiles of 32 keys in key order. The kv
// head is the workgroup index modulo kv_heads, so that with 8 kv heads every workgroup of a head runs on the
// same XCD and the head's K and V stay in that XCD's L2. Tiles go straight from memory into three LDS stages
// two tiles ahead (16-byte chunks of a row placed at chunk ^ (key & 15) for K, and at chunk ^ 2 (key & 7)
// for V, so that the operand reads of 16 lanes fall in distinct banks), small enough for three workgroups a
// CU, whose softmax runs beside the others' MFMAs.
// On the fp16 MFMA (v_mfma_f32_16x16x32_f16) a wave computes the scores transposed, S^T = K Q^T, so
// that a lane holds eight scores of one query: the online softmax (fp32, base 2) reduces them
// in-lane and across its four lane groups (permlane swaps), and the probabilities already sit where
// the B operand of O^T = V^T P^T wants them (the MFMA's k index is permuted to the keys the lane
// holds, consistently in A and B); V^T's operand comes from the row-major tile by LDS transpose reads
// (ds_read_b64_tr_b16). P is split into an fp16 high part and an fp16 residual, two MFMAs, so that
// P.V keeps the precision of fp32 probabilities.
// With a workspace the keys of a block of rows are split into chunks that workgroups of their own take, each
// leaving its state (m, l, O) in fp32 for a second launch that merges them by the Merge rule: a few rows
// behind a long cache, or a prompt whose last rows see many times the keys of its first, then fill the chip.
// Without one, a workgroup of up to three key groups of four waves takes all of a block's keys.
#include <algorithm>

#include "hwk_common.h"
#include "internal.h"

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int KT = 32;  // keys a tile
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLift = 8.0f;
constexpr uint32_t kFold = 16;
constexpr int NST = 3;                          // LDS stages
constexpr uint32_t KBYTES = KT * 256;           // a stage: K rows, then V rows
constexpr uint32_t STAGE = 2 * KBYTES;
constexpr int LOADS = STAGE / (4 * 64 * 16);    // loads into LDS a lane a tile
constexpr uint32_t kRows = 64;                  // query rows a workgroup
constexpr uint32_t kPart = kRows * (128 + 2);   // floats of a chunk's state: O (rows, 128) | m (rows) | l (rows)

__device__ __forceinline__ half8 half8_of(u32x4 u) { return __builtin_bit_cast(half8, u); }

// LDS transpose read: in each 16-lane group, lane 4a + c receives element c of the 8-byte
// segments addressed by lanes a, a + 4, a + 8, a + 12 of the group.
__device__ __forceinline__ short4v tr_read(const lds_char *p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)p);
}

// The larger of two and the largest of three, NaNs left out (fmaxf would first quiet each operand in an
// instruction of its own). max3 is inline assembly, which the compiler does not keep away from an MFMA that
// still writes its operand: the scores go through max2, its own instruction, first.
__device__ __forceinline__ float max2(float a, float b) { return __builtin_amdgcn_fmed3f(a, b, __builtin_inff()); }
__device__ __forceinline__ float max3(float a, float b, float c) {
  float d;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
  return d;
}

// How a prompt's attention is cut up: blocks of 64 rows a kv head, and chunks of `tiles` key tiles, at most
// `chunks` a block (1: not split).
struct Cut {
  uint32_t blocks, tiles, chunks;
};

struct PrefillArgs {
  int mode;
  uint32_t T, start, heads, kvh, cap, gs;  // gs: log2 of the query heads a kv head
  float scale_log2;
  Cut cut;
};

// The keys [0, last) that block qb's rows see.
__device__ __forceinline__ uint32_t block_last(const PrefillArgs &a, uint32_t qb) {
  return a.start + min(((qb + 1) * kRows - 1) >> a.gs, a.T - 1) + 1;
}

// The first block with a chunk c: with keys past the first c chunks (the grid holds no chunk past the last).
__host__ __device__ __forceinline__ uint32_t first_block(const PrefillArgs &a, uint32_t c) {
  const uint32_t x = c * a.cut.tiles * KT;
  return x < a.start ? 0u : min((x - a.start) >> (6 - a.gs), a.cut.blocks);
}

// S key groups of four waves: group gi takes the chunk's tiles gi, gi + S, ... with stages of its own; the
// other groups' (m, l, O^T) then meet the first's in LDS (the Merge rule in base 2). ZERO: the scale is 0.
template <int S, bool ZERO>
__global__ __launch_bounds__(256 * S) __attribute__((amdgpu_waves_per_eu(3))) void k_attn_prefill(
    const u32x4 *__restrict__ q, const u32x4 *__restrict__ kc, const u32x4 *__restrict__ vc, void *__restrict__ out,
    float *__restrict__ ws, PrefillArgs a) {
  static_assert(S >= 1 && S <= 3, "one to three key groups");
  __shared__ __attribute__((aligned(16))) char lds_all[S * NST * STAGE];
  const int wg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int gi = wg >> 2, wave = wg & 3, lane = threadIdx.x & 63;
  const int n = lane & 15, grp = lane >> 4;
  const uint32_t h = blockIdx.x % a.kvh;  // consecutive workgroups go to different XCDs
  // the first chunks of all blocks, then the second ones of the blocks that have them, ..., in each the longest
  // block first
  uint32_t r = blockIdx.x / a.kvh, c = 0;
  for (uint32_t n; r >= (n = a.cut.blocks - first_block(a, c)); c++) r -= n;
  const uint32_t qb = a.cut.blocks - 1 - r;
  const uint32_t last = block_last(a, qb), tiles = (last + KT - 1) / KT;
  const uint32_t it0 = c * a.cut.tiles, it1 = min(it0 + a.cut.tiles, tiles);  // the chunk's tiles
  const uint32_t r0 = qb * kRows + wave * 16, row = r0 + n;  // the wave's first row, the lane's
  const uint32_t p0 = r0 >> a.gs;                            // the wave's first position
  const bool wlive = p0 < a.T;
  const uint32_t tq = min(row >> a.gs, a.T - 1), head = (h << a.gs) + (row & ((1u << a.gs) - 1));
  const bool qlive = (row >> a.gs) < a.T;
  const uint32_t qpos = a.start + tq;
  const uint32_t wmax = a.start + min((r0 + 15) >> a.gs, a.T - 1);  // the wave's last position
  const uint32_t wfull = a.start + p0;  // keys up to here are seen by every row of the wave
  const u32x4 *kh = kc + (size_t)h * a.cap * 16, *vh = vc + (size_t)h * a.cap * 16;

  // the scale's sign (exactly) into q, and a zero scale as q times 0 (NaN of a NaN or infinity), in a kernel of its own
  // (in the others its instructions cost 33 rows behind 8,000 keys 18.0 -> 18.7 µs): the scores' largest is then that
  // of the products
  const uint32_t flip = a.scale_log2 < 0.0f ? 0x80008000u : 0u;
  const float scale = ZERO ? 1.0f : fabsf(a.scale_log2);
  half8 qv[4];
#pragma unroll
  for (int s = 0; s < 4; s++) {
    const u32x4 v = qlive ? q[((size_t)tq * a.heads + head) * 16 + s * 4 + grp] : (u32x4){0u, 0u, 0u, 0u};
    qv[s] = half8_of(v ^ flip);
    if constexpr (ZERO) qv[s] *= (f16)0.0f;
  }

  // the group's stages; the lane's loads of a tile: slot p = (i * 4 + wave) * 64 + lane holds chunk p % 16 of
  // key p / 16, swizzled on the source side. Keys past the block's read its last key (masked), tiles past the
  // chunk its last tile.
  const uint32_t lds0 = lds_at(lds_all) + gi * NST * STAGE;
  constexpr int HALF = LOADS / 2;
  uint32_t lkey[HALF], lk[HALF], lv[HALF];
#pragma unroll
  for (int i = 0; i < HALF; i++) {
    const uint32_t p = (i * 4 + wave) * 64 + lane, key = p / 16, ch = p % 16;
    lkey[i] = key;
    lk[i] = (ch ^ (key & 15)) * 16;
    lv[i] = (ch ^ ((key & 7) << 1)) * 16;
  }
  auto load = [&](uint32_t j, uint32_t stage) __attribute__((always_inline)) {
    const uint32_t key0 = min(it0 + j * S + gi, it1 - 1) * KT, st = lds0 + stage * STAGE + wave * 1024;
    const u32x4 *kt = kh + (size_t)key0 * 16, *vt = vh + (size_t)key0 * 16;
#pragma unroll
    for (int i = 0; i < HALF; i++) {
      const uint32_t at = min(lkey[i], last - 1 - key0) * 256;
      to_lds16(kt, at + lk[i], st + i * 4096);
      to_lds16(vt, at + lv[i], st + KBYTES + i * 4096);
    }
  };
  // the lane's operands in a stage: K row n, chunk (s*4 + grp) ^ n; V^T transpose reads: source lane of group
  // grp addresses key grp*4 + n/4 (+16 for the second read), dims d*16 + 4*(n%4) .. +3
  const uint32_t ka = n * 256 + ((grp ^ n) & 15) * 16;
  const uint32_t vkey = grp * 4 + n / 4;
  const uint32_t va = KBYTES + vkey * 256 + (vkey & 7) * 32 + (n % 4) * 8;

  floatx4 acc[8];
#pragma unroll
  for (int d = 0; d < 8; d++) acc[d] = (floatx4){0.0f, 0.0f, 0.0f, 0.0f};
  float m = -__builtin_inff(), l = 0.0f;
  // one key group walks all of a block's tiles: its sums go to a second level every kFold tiles, so that they
  // keep the precision of the shorter sums that several groups (or chunks) add up
  floatx4 tot[S == 1 ? 8 : 1];
  float ltot = 0.0f;
  if constexpr (S == 1) {
#pragma unroll
    for (int d = 0; d < 8; d++) tot[d] = (floatx4){0.0f, 0.0f, 0.0f, 0.0f};
  }

  auto attend = [&](uint32_t it, uint32_t stage) __attribute__((always_inline)) {
    const uint32_t key0 = it * KT;
    if (it >= it1 || !wlive || key0 > wmax) return;
    const lds_char *st = (const lds_char *)lds_all + (gi * NST + stage) * STAGE;
    // S^T: keys key0 + kt*16 + grp*4 + r of the lane's query n; then V^T's operands, read under the softmax
    typedef const __attribute__((address_space(3))) u32x4 lds_u32x4;
    u32x4 kv[2][4];
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int kt = 0; kt < 2; kt++) kv[kt][s] = *(lds_u32x4 *)(st + (ka ^ (s << 6)) + kt * 4096);
    issue_order();
    short4v vv[4][2];  // dims 0..63; the others are read when these are used
#pragma unroll
    for (int d = 0; d < 4; d++)
#pragma unroll
      for (int u = 0; u < 2; u++) vv[d][u] = tr_read(st + (va ^ (d << 5)) + u * 4096);
    issue_order();
    floatx4 sc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int kt = 0; kt < 2; kt++)
        sc[kt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(half8_of(kv[kt][s]), qv[s], sc[kt], 0, 0, 0);
    if (key0 + KT - 1 > wfull) {
#pragma unroll
      for (int kt = 0; kt < 2; kt++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (key0 + kt * 16 + grp * 4 + r > qpos) sc[kt][r] = -__builtin_inff();
    }
    const float t0 = max2(sc[0][0], sc[0][1]), t1 = max2(sc[0][2], sc[0][3]);
    const float t2 = max2(sc[1][0], sc[1][1]), t3 = max2(sc[1][2], sc[1][3]);
    float tmax = max3(max3(t0, t1, t2), t3, t3);
    {
      float x = tmax, y = tmax;
      swap_rows16(x, y);
      tmax = max3(x, y, y);
      x = y = tmax;
      swap_rows32(x, y);
      tmax = max3(x, y, y) * scale;
    }
    // m, the exponent that the row's sums are taken against, moves only when a score passes it by kLift: the
    // sums are then rescaled (any m gives the same quotient; p stays below 2^kLift, far inside fp16)
    if (__ballot(tmax > m + kLift)) {
      const float mnew = tmax > m + kLift ? tmax : m;
      const float alpha = mnew == -__builtin_inff() ? 1.0f : __builtin_amdgcn_exp2f(m - mnew);
      m = mnew;
      l *= alpha;
#pragma unroll
      for (int d = 0; d < 8; d++) acc[d] *= alpha;
      if constexpr (S == 1) {
        ltot *= alpha;
#pragma unroll
        for (int d = 0; d < 8; d++) tot[d] *= alpha;
      }
    }
    const float base = m == -__builtin_inff() ? 0.0f : m;  // no key seen yet: every p is exp2(-inf) = 0
    // v_exp_f32 alone: exp2f's further steps only keep results below 2^-126, beside a largest p of 1 or more
    float p[2][4];
#pragma unroll
    for (int kt = 0; kt < 2; kt++)
#pragma unroll
      for (int r = 0; r < 4; r++) p[kt][r] = __builtin_amdgcn_exp2f(fmaf(sc[kt][r], scale, -base));
    // the lane's own keys: the four lane groups are summed once, at the end
    l += ((p[0][0] + p[0][1]) + (p[0][2] + p[0][3])) + ((p[1][0] + p[1][1]) + (p[1][2] + p[1][3]));
    half8 bhi, blo;
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      typedef float f2 __attribute__((ext_vector_type(2)));
      const f2 pv = {p[i / 4][i % 4], p[i / 4][i % 4 + 1]};
      const h2 hi = __builtin_convertvector(pv, h2);
      const f2 rest = {fmaf((float)hi.x, -1.0f, pv.x), fmaf((float)hi.y, -1.0f, pv.y)};  // exact
      const h2 lo = __builtin_convertvector(rest, h2);
      bhi[i] = hi.x;
      bhi[i + 1] = hi.y;
      blo[i] = lo.x;
      blo[i + 1] = lo.y;
    }
#pragma unroll
    for (int d = 0; d < 8; d++) {
      const half8 av =
          __builtin_bit_cast(half8, __builtin_shufflevector(vv[d % 4][0], vv[d % 4][1], 0, 1, 2, 3, 4, 5, 6, 7));
      if (d < 4) {
#pragma unroll
        for (int u = 0; u < 2; u++) vv[d][u] = tr_read(st + (va ^ ((d + 4) << 5)) + u * 4096);
      }
      acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bhi, acc[d], 0, 0, 0);
      acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, blo, acc[d], 0, 0, 0);
    }
  };

  // Step j: every wave's loads of tile j landed and every wave done with tile j-1's stage, which tile
  // j + NST-1 takes. All groups run as many steps as group 0.
  const uint32_t steps = (it1 - it0 + S - 1) / S;
#pragma unroll
  for (int s = 0; s < NST - 1; s++) load(s, s);
  for (uint32_t j0 = 0; j0 < steps; j0 += NST) {
#pragma unroll
    for (int s = 0; s < NST; s++) {
      const uint32_t j = j0 + s;
      if (j >= steps) break;
      wait_loads<LOADS * (NST - 2)>();
      wait_lds();
      bare_barrier();
      load(j + NST - 1, (s + NST - 1) % NST);
      attend(it0 + j * S + gi, s);
      if constexpr (S == 1) {
        if (j % kFold == kFold - 1) {
          ltot += l;
          l = 0.0f;
#pragma unroll
          for (int d = 0; d < 8; d++) {
            tot[d] += acc[d];
            acc[d] = (floatx4){0.0f, 0.0f, 0.0f, 0.0f};
          }
        }
      }
    }
  }
  if constexpr (S == 1) {
    l += ltot;
#pragma unroll
    for (int d = 0; d < 8; d++) acc[d] += tot[d];
  }
  wait_loads<0>();  // no load into LDS may land in a stage put to another use
  l = row_groups_sum(l);
  if constexpr (S > 1) {
    // groups 1 .. S-1's states to group 0 through the stages, group 0 merges: weights 2^(m - top)
    wait_lds();
    bare_barrier();
    float *xo = (float *)lds_all + (size_t)(wave * 64 + lane) * 34;
    constexpr size_t GX = 256 * 34;  // floats a group's states take
    if (gi > 0) {
      float *xg = xo + (gi - 1) * GX;
#pragma unroll
      for (int d = 0; d < 8; d++)
#pragma unroll
        for (int r = 0; r < 4; r++) xg[d * 4 + r] = acc[d][r];
      xg[32] = m;
      xg[33] = l;
    }
    __syncthreads();
    if (gi > 0) return;
    float mg[S], ag[S];
    mg[0] = m;
    float top = m;
#pragma unroll
    for (int g = 1; g < S; g++) {
      mg[g] = xo[(g - 1) * GX + 32];
      top = fmaxf(top, mg[g]);
    }
#pragma unroll
    for (int g = 0; g < S; g++) ag[g] = top == -__builtin_inff() ? 0.0f : exp2f(mg[g] - top);
    l = l * ag[0];
#pragma unroll
    for (int g = 1; g < S; g++) l = l + xo[(g - 1) * GX + 33] * ag[g];
#pragma unroll
    for (int d = 0; d < 8; d++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        float v = acc[d][r] * ag[0];
#pragma unroll
        for (int g = 1; g < S; g++) v = v + xo[(g - 1) * GX + d * 4 + r] * ag[g];
        acc[d][r] = v;
      }
    m = top;
  }
  if (!qlive) return;
  if (tiles > a.cut.tiles) {  // one chunk of several: the state, for k_attn_prefill_merge
    float *part = ws + ((size_t)(h * a.cut.blocks + qb) * a.cut.chunks + c) * kPart;
#pragma unroll
    for (int d = 0; d < 8; d++) *(floatx4 *)(part + (wave * 16 + n) * 128 + d * 16 + grp * 4) = acc[d];
    if (grp == 0) {
      part[kRows * 128 + wave * 16 + n] = m;
      part[kRows * 129 + wave * 16 + n] = l;
    }
    return;
  }
  const float inv = l > 0.0f ? 1.0f / l : 0.0f;
  const size_t o0 = ((size_t)tq * a.heads + head) * 128;
#pragma unroll
  for (int d = 0; d < 8; d++) {
    const uint32_t dim = d * 16 + grp * 4;
    if (a.mode == HWK_OUT_F16) {
      half4 o;
#pragma unroll
      for (int r = 0; r < 4; r++) o[r] = (f16)f32_value(acc[d][r] * inv);
      *(half4 *)((f16 *)out + o0 + dim) = o;
    } else {
#pragma unroll
      for (int r = 0; r < 4; r++) ((float *)out)[o0 + dim + r] = acc[d][r] * inv;
    }
  }
}

// The chunks' states of each row whose keys were split, merged: one wave a row, lane c holding chunk c's m and l
// (at most 64 chunks), then two dims a lane, eight chunks' loads at once. A chunk none of whose keys the row saw (l
// exactly 0) adds nothing; every other one is weighed by 2^(m - top), its NaN or infinite l or O included, so that a
// NaN or +Inf score makes the row NaN as it does in one workgroup's sums.
constexpr uint32_t kMaxSplit = 64;
__global__ __launch_bounds__(256) void k_attn_prefill_merge(const float *__restrict__ ws, void *__restrict__ out,
                                                            PrefillArgs a) {
  const uint32_t lane = threadIdx.x & 63, i = blockIdx.x * 4 + (threadIdx.x >> 6);
  const uint32_t rw = i % kRows, b = i / kRows, qb = b % a.cut.blocks, h = b / a.cut.blocks;
  const uint32_t row = qb * kRows + rw, t = row >> a.gs;
  const uint32_t tiles = (block_last(a, qb) + KT - 1) / KT;
  if (h >= a.kvh || t >= a.T || tiles <= a.cut.tiles) return;
  const uint32_t chunks = (tiles + a.cut.tiles - 1) / a.cut.tiles;
  const float *part = ws + (size_t)b * a.cut.chunks * kPart;
  const uint32_t cl = min(lane, chunks - 1);
  const float mc = part[cl * kPart + kRows * 128 + rw], lc = part[cl * kPart + kRows * 129 + rw];
  const bool some = lane < chunks && lc != 0.0f;
  const float top = group_max_dpp<64>(some ? mc : -__builtin_inff());
  const float w = some ? exp2f(mc - top) : 0.0f;
  const float den = group_sum<64>(w * (some ? lc : 0.0f));
  const int keep = some ? -1 : 0;  // a mask and no selects: the compiler moves loads into a select's branch
  float n0 = 0.0f, n1 = 0.0f;
  for (uint32_t c0 = 0; c0 < chunks; c0 += 8) {
    uint2 o[8];
#pragma unroll
    for (int u = 0; u < 8; u++)
      o[u] = *(const uint2 *)(part + (size_t)min(c0 + u, chunks - 1) * kPart + rw * 128 + 2 * lane);
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const float wc = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w), (int)(c0 + u)));
      const uint32_t k = (uint32_t)__builtin_amdgcn_readlane(keep, (int)(c0 + u));
      n0 += wc * __uint_as_float(o[u].x & k);
      n1 += wc * __uint_as_float(o[u].y & k);
    }
  }
  const size_t o0 = ((size_t)t * a.heads + (h << a.gs) + (row & ((1u << a.gs) - 1))) * 128 + 2 * lane;
  store_out(out, o0, den == 0.0f ? 0.0f : n0 / den, a.mode);
  store_out(out, o0 + 1, den == 0.0f ? 0.0f : n1 / den, a.mode);
}

// How the rows of `tokens` positions from start on are cut. Unsplit (no workspace) a chunk is all of a
// block's keys. With one, when the blocks are too few for the chip and their keys many, chunks of
//   max(4, min(one workgroup a CU, max(16, three a CU))) tiles
// if a block then has at least four: below that the second launch, the states written and read again and
// the last chunks' idle time cost more than the split gains (measured over chunks of 1..128 tiles, us, start
// -> unsplit -> split: 33 rows of 16 heads behind 8,000 keys 159 -> 91 -> 18; 5 behind 1,024 25.4 -> 15.1 ->
// 8.7; 128 behind 4,000 86 -> 50 -> 22; 200 rows of 32 heads behind 8,000 170 -> 94 -> 57; but 1,000 behind
// 1,000 45 -> 27.8 -> 28.8 and the 1,024-token prompt 28.8 -> 18.1 -> 26).
constexpr uint32_t kCus = 256, kSplitBlocks = 256;
Cut cut_of(uint32_t tokens, uint32_t start, const hwk_attn_params *p, bool split) {
  Cut c;
  c.blocks = (uint32_t)(((uint64_t)tokens * (p->heads / p->kv_heads) + kRows - 1) / kRows);
  const uint32_t most = (uint32_t)(((uint64_t)start + tokens + KT - 1) / KT);
  c.tiles = most;
  const uint64_t units = (uint64_t)c.blocks * p->kv_heads;
  if (split && units < kSplitBlocks) {
    const uint64_t one = (units * most + kCus - 1) / kCus, three = (units * most + 3 * kCus - 1) / (3 * kCus);
    const uint64_t least = (most + kMaxSplit - 1) / kMaxSplit;
    const uint64_t t = std::max({(uint64_t)4, least, std::min(one, std::max((uint64_t)16, three))});
    if (most >= 4 * t) c.tiles = (uint32_t)t;
  }
  c.chunks = (most + c.tiles - 1) / c.tiles;
  return c;
}

template <int S>
char *launch_prefill(hipStream_t st, const void *q, const void *k, const void *v, void *out, float *ws,
                     const PrefillArgs &a) {
  uint32_t units = 0;
  for (uint32_t c = 0; c < a.cut.chunks; c++) units += a.cut.blocks - first_block(a, c);
  auto *kernel = a.scale_log2 == 0.0f ? k_attn_prefill<S, true> : k_attn_prefill<S, false>;
  hipLaunchKernelGGL(kernel, dim3(units * a.kvh), dim3(256 * S), 0, st, (const u32x4 *)q, (const u32x4 *)k,
                     (const u32x4 *)v, out, ws, a);
  if (char *err = hwk::launched("hwk_attn_prefill")) return err;
  if (a.cut.chunks == 1) return nullptr;
  hipLaunchKernelGGL(k_attn_prefill_merge, dim3(a.cut.blocks * a.kvh * (kRows / 4)), dim3(256), 0, st, ws, out, a);
  return hwk::launched("hwk_attn_prefill (merge)");
}

char *run_prefill(hipStream_t st, const void *q, const void *k, const void *v, void *out, float *ws, uint32_t tokens,
                  uint32_t start, const hwk_attn_params *p, const Cut &cut) {
  PrefillArgs a;
  a.mode = (int)p->out_mode;
  a.T = tokens;
  a.start = start;
  a.heads = p->heads;
  a.kvh = p->kv_heads;
  a.cap = p->capacity;
  const uint32_t G = p->heads / p->kv_heads;
  a.gs = G == 4 ? 2 : G == 2 ? 1 : 0;
  a.scale_log2 = hwk::f32_of_bits(p->scale_bits) * kLog2e;
  a.cut = cut;
  // one key group a workgroup when the key chunks or the blocks alone fill the chip with three workgroups a CU
  // (4,096 rows of 32 heads: 219 us against 245 in three groups); else two once the longest block has a few
  // tiles, three past 256 keys (1,024 rows of 16 heads: 22.9 us in one group, 18.4 in two, 18.1 in three)
  if (cut.chunks > 1 || (uint64_t)cut.blocks * p->kv_heads >= 6 * kCus || start + tokens <= 128)
    return launch_prefill<1>(st, q, k, v, out, ws, a);
  if (start + tokens <= 256) return launch_prefill<2>(st, q, k, v, out, ws, a);
  return launch_prefill<3>(st, q, k, v, out, ws, a);
}

char *check_prefill(const char *what, const void *q, const void *k, const void *v, const void *out, uint32_t tokens,
                    uint32_t start, const hwk_attn_params *p) {
  HWK_CHECK(p, "%s: null params", what);
  HWK_CHECK(q && k && v && out, "%s: null pointer", what);
  HWK_CHECK(p->head_dim == 128, "%s: head_dim %u (128 only)", what, p->head_dim);
  HWK_CHECK(!p->kv_int8, "%s: fp16 caches only", what);
  HWK_CHECK(p->kv_heads > 0 && p->heads % p->kv_heads == 0, "%s: %u heads over %u kv heads", what, p->heads, p->kv_heads);
  const uint32_t G = p->heads / p->kv_heads;
  HWK_CHECK(G == 1 || G == 2 || G == 4, "%s: %u query heads a kv head (1, 2 or 4)", what, G);
  HWK_CHECK((uint64_t)start + tokens <= p->capacity, "%s: positions %u+%u past capacity %u", what, start, tokens,
            p->capacity);
  HWK_CHECK(p->len == start + tokens, "%s: len %u is not start + tokens = %u", what, p->len, start + tokens);
  HWK_CHECK(p->out_mode == HWK_OUT_F32 || p->out_mode == HWK_OUT_F16, "%s: out_mode %u", what, p->out_mode);
  HWK_CHECK(hwk::aligned(q, 16) && hwk::aligned(k, 16) && hwk::aligned(v, 16) && hwk::aligned(out, 8),
            "%s: q, k, v 16-byte and out 8-byte aligned", what);
  return nullptr;
}

}  // namespace

extern "C" {

HWK_API size_t hwk_attn_prefill_workspace_bytes(uint32_t tokens, uint32_t start, const hwk_attn_params *p) {
  if (!p || p->kv_heads == 0 || p->heads % p->kv_heads || tokens == 0) return 0;
  const Cut c = cut_of(tokens, start, p, true);
  return c.chunks == 1 ? 0 : (size_t)c.blocks * p->kv_heads * c.chunks * kPart * sizeof(float);
}

HWK_API char *hwk_attn_prefill_ws(void *stream, const void *q, const void *k, const void *v, void *out, void *workspace,
                                  size_t workspace_bytes, uint32_t tokens, uint32_t start, const hwk_attn_params *p) {
  if (char *err = check_prefill("hwk_attn_prefill_ws", q, k, v, out, tokens, start, p)) return err;
  if (tokens == 0) return nullptr;
  const size_t need = hwk_attn_prefill_workspace_bytes(tokens, start, p);
  HWK_CHECK(need == 0 || (workspace && hwk::aligned(workspace, 16) && workspace_bytes >= need),
            "hwk_attn_prefill_ws: a 16-byte aligned workspace of %zu bytes needed, %zu given", need, workspace_bytes);
  return run_prefill((hipStream_t)stream, q, k, v, out, (float *)workspace, tokens, start, p,
                     cut_of(tokens, start, p, true));
}

HWK_API char *hwk_attn_prefill(void *stream, const void *q, const void *k, const void *v, void *out, uint32_t tokens,
                               uint32_t start, const hwk_attn_params *p) {
  if (char *err = check_prefill("hwk_attn_prefill", q, k, v, out, tokens, start, p)) return err;
  if (tokens == 0) return nullptr;
  return run_prefill((hipStream_t)stream, q, k, v, out, nullptr, tokens, start, p, cut_of(tokens, start, p, false));
}

}  // extern "C"

// cut_of's chunks take a block's keys in at least 16 tiles, with at most three workgroups a CU and one more
// chunk a block.
size_t hwk::attn_prefill_most_bytes(uint32_t max_ctx) {
  return max_ctx <= 15 * KT ? 0 : (3 * kCus + kSplitBlocks) * kPart * sizeof(float);
}
