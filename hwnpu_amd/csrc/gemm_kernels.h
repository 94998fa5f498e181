// The device code of K3, the prefill / verify GEMM, shared by libhwk's kernels (gemm.hip) and the
// kernels of the library's code object (co/hwk_co.hip), so that both run the same instructions.
//
// Prefill / verify GEMM (K3) on gfx950: Y (M, N) = X (M, K) W^T, X fp16, W int8 per output channel
// or MXFP4, fp32 accumulation on the fp16 MFMA (v_mfma_f32_16x16x32_f16). Weights are converted next to
// the MFMAs that take them: int8 exactly to fp16 (the channel scale applied to the fp32 result), MXFP4 by
// the hardware fp4 conversion with the block scale folded in.
//
// Two forms. The paired form (gemm_pair_wg, K a multiple of 64) takes nearly everything: operands straight
// from memory into LDS rings, one barrier a step of 64 values, tiles from 16 x 32 to 128 x 256 and, for tiles
// that would leave CUs or waves idle, several k groups of waves a workgroup (pick_pair chooses). The general
// form (gemm_wg) takes any K that is a multiple of 32, operands past 4 GiB and odd scale addresses: a
// BM x BN tile, K 128 at a time with X through LDS (two buffers, one barrier a step) and the weights loaded
// into registers two steps ahead.
//
// MXFP4 exactness: a code times its block scale is an fp16 value when the scale's exponent is in
// [-23, 13]. A row (output channel) whose finite block exponents leave that range is shifted by a
// power of two s0 chosen per row (the largest exponent mapped to 13) and its fp32 result scaled back
// by 2^s0, which is exact; rows whose exponents span more than 36 lose the low bits of their
// smallest blocks (values below 2^-24 of the shifted scale). Scale e = 0 is 0 and e = 255 is +Inf,
// as in the reference's Dequantize (internal/mxfp4/mxfp4.go:77).
#pragma once

#include <type_traits>

#include "hwk_common.h"

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

namespace hwk_gemm {

constexpr int KS = 128;     // K a step
constexpr int CH = KS / 8;  // 16-byte chunks of an X row a step
constexpr int KK = KS / 32;  // MFMAs a step for one (16-row, 16-column) tile
constexpr int NS = 2;       // register stages: loads run NS steps ahead
constexpr int kOutSwiGLU = HWK_OUT_SWIGLU_F16;

// 4 int8 codes (one dword) as 4 exact fp16 values (two dwords).
__device__ __forceinline__ uint2 i8x4_to_f16x4(uint32_t w) {
  const uint32_t u = w ^ 0x80808080u;
  const h2 bias = {(f16)1152.0f, (f16)1152.0f};
  const h2 lo = h2_of_bits(__builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) - bias;
  const h2 hi = h2_of_bits(__builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) - bias;
  return make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
}

// 8 int8 codes (two dwords) as a half8 operand.
__device__ __forceinline__ half8 i8x8_to_half8(uint32_t a, uint32_t b) {
  const uint2 p = i8x4_to_f16x4(a), q = i8x4_to_f16x4(b);
  const u32x4 v = {p.x, p.y, q.x, q.y};
  return __builtin_bit_cast(half8, v);
}

// 8 e2m1 codes (one dword, even element in the low nibble) times scale s as a half8 operand.
__device__ __forceinline__ half8 fp4x8_to_half8(uint32_t w, float s) {
  const u32x4 v = {__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, s, 0)),
                   __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, s, 1)),
                   __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, s, 2)),
                   __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, s, 3))};
  return __builtin_bit_cast(half8, v);
}

__device__ __forceinline__ u32x4 load16(const void *p) { return *(const u32x4 *)p; }

// The X chunk (of CH a row a step) that MFMA kk of lane group q reads: the k offsets of a lane's
// operands in the step. int8: two 16-byte weight loads a lane at q*16 and 64 + q*16 (each 16 rows x 64
// contiguous bytes a load instruction); MXFP4: one 32-value block a lane at q*32 (one code load and one scale
// byte: the paired form's order, 16 values of each 64, took two of each and 1.1-1.28 times as long here).
template <bool MX>
__device__ __forceinline__ int xchunk(int q, int kk) {
  if constexpr (MX) return 4 * q + kk;
  return kk < 2 ? 2 * q + kk : 8 + 2 * q + (kk - 2);
}

// The first 128-value step of segment g when the S steps of K go to KG segments.
__host__ __device__ __forceinline__ uint32_t seg_first(uint32_t S, uint32_t KG, uint32_t g) {
  return (uint32_t)((uint64_t)g * S / KG);
}

// KG k groups of WM x WN waves: group g takes MFMAs g*KK/KG .. of every step of the whole tile, and
// the groups' accumulators are summed at the end (int8 only: 2 groups make an 8-wave workgroup of a
// tile that 4 waves would hold, so that a CU's SIMDs split the tile's k as well as its columns).
template <int BM, int BN, bool MX, int WM, int WN, int KG>
struct Cfg {
  static constexpr int NT = 64 * WM * WN * KG;              // threads: KG groups of WM x WN waves
  static constexpr int TM = BM / WM / 16, TN = BN / WN / 16;  // 16 x 16 tiles a wave
  static constexpr int AL = BM * CH / NT;                   // X chunks a thread stages a step
  static constexpr int BL = MX ? 1 : 2 / KG;                // 16-byte weight loads a lane a step a tile
  static constexpr int KKG = KK / KG;                       // MFMAs a tile a step a wave
  static_assert(BM * CH % NT == 0 && TM * WM * 16 == BM && TN * WN * 16 == BN, "tile shape");
  static_assert(KG == 1 || KG == 2, "one or two k groups");
};

template <int BM, int BN, bool MX, int WM, int WN, int KG>
struct Stage {
  u32x4 a[Cfg<BM, BN, MX, WM, WN, KG>::AL];
  u32x4 b[Cfg<BM, BN, MX, WM, WN, KG>::TN][Cfg<BM, BN, MX, WM, WN, KG>::BL];
  uint32_t e[Cfg<BM, BN, MX, WM, WN, KG>::TN];  // MXFP4 block scale bytes
  uint32_t k0;                                  // the step's K offset
};

// Issue the global loads of the step at K offset k0 into s: X (load_x) and the weights (load_w).
// Out-of-range rows and columns read the last row/column (their results are not stored); K past the
// end reads in-range data, which zero_tail clears when the stage is consumed (a select here would wait
// for the load at once). Every load is issued unconditionally (a load under a branch would be waited
// for at the join).
template <int BM, int BN, bool MX, int WM, int WN, int KG>
__device__ __forceinline__ void load_x(Stage<BM, BN, MX, WM, WN, KG> &s, const u32x4 *__restrict__ X, uint32_t M,
                                       uint32_t K, uint32_t m0, uint32_t k0, int t) {
  using C = Cfg<BM, BN, MX, WM, WN, KG>;
  s.k0 = k0;
#pragma unroll
  for (int i = 0; i < C::AL; i++) {
    const int c = t + C::NT * i, row = c / CH, ch = c % CH;
    const uint32_t m = min(m0 + row, M - 1);
    s.a[i] = X[((size_t)m * K + min(k0 + ch * 8, K - 8)) / 8];
  }
}

// (int8: a k group's half of the step's 128 codes a row, h = g, when KG = 2)
template <int BM, int BN, bool MX, int WM, int WN, int KG>
__device__ __forceinline__ void load_w(Stage<BM, BN, MX, WM, WN, KG> &s, const uint8_t *__restrict__ W,
                                       const uint8_t *__restrict__ E, uint32_t K, uint32_t k0,
                                       const uint32_t (&brow)[Cfg<BM, BN, MX, WM, WN, KG>::TN], int q, int g) {
  using C = Cfg<BM, BN, MX, WM, WN, KG>;
  if constexpr (MX) {
    const uint32_t blk = min(k0 + q * 32, K - 32) / 32;
#pragma unroll
    for (int j = 0; j < C::TN; j++) {
      const size_t bi = (size_t)brow[j] * (K / 32) + blk;
      s.b[j][0] = load16(W + bi * 16);
      s.e[j] = E[bi];
    }
  } else {
#pragma unroll
    for (int h = 0; h < C::BL; h++) {
      const uint32_t kc = min(k0 + (KG == 1 ? h : g) * 64 + q * 16, K - 16);
#pragma unroll
      for (int j = 0; j < C::TN; j++) s.b[j][h] = load16(W + (size_t)brow[j] * K + kc);
    }
  }
}

// A step reaching past K: its X chunks and weight loads past K become zeros (MXFP4: scale 0).
template <int BM, int BN, bool MX, int WM, int WN, int KG>
__device__ __forceinline__ void zero_tail(Stage<BM, BN, MX, WM, WN, KG> &s, uint32_t K, int t, int q, int g) {
  using C = Cfg<BM, BN, MX, WM, WN, KG>;
  const u32x4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int i = 0; i < C::AL; i++)
    if (s.k0 + ((t + C::NT * i) % CH) * 8 >= K) s.a[i] = zero;
#pragma unroll
  for (int j = 0; j < C::TN; j++) {
    if constexpr (MX) {
      if (s.k0 + q * 32 >= K) {
        s.b[j][0] = zero;
        s.e[j] = 0u;
      }
    } else {
#pragma unroll
      for (int h = 0; h < C::BL; h++)
        if (s.k0 + (KG == 1 ? h : g) * 64 + q * 16 >= K) s.b[j][h] = zero;
    }
  }
}

// The block scale of exponent byte e in a row shifted by 2^-s0 (see the header): 0 for e = 0 or a
// shifted exponent below the float range, +Inf for e = 255.
__device__ __forceinline__ float shifted_scale(uint32_t e, int s0) {
  const float v = __uint_as_float((uint32_t)max((int)e - s0, 0) << 23);  // below the float range: +0
  return e == 255u ? __builtin_inff() : e == 0u ? 0.0f : v;
}

// The row shifts s0 of the tile's BN weight rows (n0 .. n0+BN-1, clamped to N-1): 0 for a row whose
// finite, nonzero block exponents are all in [-23, 13]; else the largest mapped to 13. The workgroup's
// threads scan the rows' scale bytes (16-byte chunks when every row starts 16-byte aligned, all of a
// thread's loads issued before any is used; bytes otherwise) and combine per row in LDS (hs: the
// largest exponent byte other than 255, ls: the smallest other than 0 and 255). hs and ls are set
// to 0 and 255 by the caller before a barrier; another barrier follows before they are read.
template <int BN, int NT>
__device__ __forceinline__ void scan_shifts(const uint8_t *__restrict__ E, uint32_t n0, uint32_t N, uint32_t nb,
                                            bool quads, int t, int *hs, int *ls) {
  auto take = [&](uint32_t e, uint32_t &h, uint32_t &l) {
    h = max(h, e == 255u ? 0u : e);
    l = min(l, (e == 0u || e == 255u) ? 255u : e);
  };
  if (quads) {
    const uint32_t nch = nb / 16, total = BN * nch;
    for (uint32_t base = 0; base < total; base += 4 * NT) {
      u32x4 v[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t c = min(base + t + NT * i, total - 1), row = c / nch;
        v[i] = *(const u32x4 *)(E + (size_t)min(n0 + row, N - 1) * nb + (c % nch) * 16);
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t c = base + t + NT * i;
        if (c >= total) continue;
        uint32_t h = 0, l = 255;
#pragma unroll
        for (int w = 0; w < 4; w++)
#pragma unroll
          for (int b = 0; b < 4; b++) take((v[i][w] >> (8 * b)) & 255u, h, l);
        atomicMax(&hs[c / nch], (int)h);
        atomicMin(&ls[c / nch], (int)l);
      }
    }
  } else {
    for (uint32_t c = t; c < BN * nb; c += NT) {
      const uint32_t row = c / nb;
      uint32_t h = 0, l = 255;
      take(E[(size_t)min(n0 + row, N - 1) * nb + c % nb], h, l);
      atomicMax(&hs[row], (int)h);
      atomicMin(&ls[row], (int)l);
    }
  }
}

// The shift of a row from its scanned bytes.
__device__ __forceinline__ int shift_of(int hi, int lo) {
  if (hi == 0) return 0;  // no finite nonzero scale
  const int emax = hi - 127, emin = lo - 127;
  return (emax <= 13 && emin >= -23) ? 0 : emax - 13;
}

// Workgroup id -> tile: consecutive ids go round the XCDs, so ids x, x+8, x+16, ... share an XCD;
// those take the M tiles of one N panel in turn.
__device__ __forceinline__ void tile_of(uint32_t id, uint32_t mt, uint32_t nt, uint32_t &tm, uint32_t &tn) {
  const uint32_t total = mt * nt;
  const uint32_t xcd = id % 8, j = id / 8;
  uint32_t lin = id;
  if (total % 8 == 0) {
    const uint32_t per = total / 8;  // tiles an XCD runs
    lin = xcd * per + j;
  }
  tn = lin / mt;
  tm = lin % mt;
}

// The tile's store: D of MFMA tile (i, j) of the wave, lane (r16, q) holding rows q*4 + r of column
// r16; int8 results take the column's scale, MXFP4 results the row shift back (2^s0, exact).
// KG > 1: the 16-row tiles i = own, own + KG, ... only.
template <int BM, int WM, int TM, int TN, bool MX, int KG = 1>
__device__ __forceinline__ void store_tile(const floatx4 (&acc)[TM][TN], const int (&s0)[TN],
                                           const uint16_t *__restrict__ S, void *__restrict__ Y, uint32_t M,
                                           uint32_t N, uint32_t m0, uint32_t nw, int wm, int r16, int q, int mode,
                                           int own = 0) {
  if (mode == kOutSwiGLU) {
    // columns (2c, 2c+1) are (gate, up) of output c, held by lanes r16 and r16 ^ 1 for the same four
    // rows: the gate lane takes the up values of rows 0, 1 and computes those outputs, the up lane
    // takes the gate values of rows 2, 3 and computes those. Every lane joins the swaps; columns past
    // N (a tile wider than N) store nothing, and with N % 16 == 0 a pair is wholly below N or not.
    const bool gate = (r16 & 1) == 0;
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const uint32_t n = nw + j * 16 + r16, c = n / 2;
      const float sc = MX ? 1.0f : (float)__builtin_bit_cast(f16, S[min(n, N - 1)]);
#pragma unroll
      for (int i = 0; i < TM; i++) {
        if (KG > 1 && i % KG != own) continue;
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] = MX ? ldexpf(acc[i][j][r], s0[j]) : acc[i][j][r] * sc;
        const float o0 = __shfl_xor(gate ? v[2] : v[0], 1, 64), o1 = __shfl_xor(gate ? v[3] : v[1], 1, 64);
        const uint32_t mr = m0 + wm * (BM / WM) + i * 16 + q * 4 + (gate ? 0 : 2);  // the lane's first row
        const float y0 = gate ? swiglu_value(v[0], o0) : swiglu_value(o0, v[2]);
        const float y1 = gate ? swiglu_value(v[1], o1) : swiglu_value(o1, v[3]);
        if (n < N && mr < M) ((f16 *)Y)[(size_t)mr * (N / 2) + c] = (f16)y0;
        if (n < N && mr + 1 < M) ((f16 *)Y)[(size_t)(mr + 1) * (N / 2) + c] = (f16)y1;
      }
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < TN; j++) {
    const uint32_t n = nw + j * 16 + r16;
    if (n >= N) continue;
    const float sc = MX ? 1.0f : (float)__builtin_bit_cast(f16, S[n]);
#pragma unroll
    for (int i = 0; i < TM; i++) {
      if (KG > 1 && i % KG != own) continue;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const uint32_t m = m0 + wm * (BM / WM) + i * 16 + q * 4 + r;
        if (m < M) store_out(Y, (size_t)m * N + n, MX ? ldexpf(acc[i][j][r], s0[j]) : acc[i][j][r] * sc, mode);
      }
    }
  }
}

// The tile's store through LDS, 16 rows of the wave's block at a time (a strip): the values as stored
// (fp16 rounded, SwiGLU'd pairs, or scaled fp32), then 16-byte pieces of the rows to Y, since an MFMA
// tile's lanes hold one column each. Every value is rounded and combined as store_tile does it. st: the
// wave's 16 x (TN*16 + 4) floats of LDS. For staged(Y, N, mode).
__device__ __forceinline__ bool staged(const void *Y, uint32_t N, int mode) {
  const uint32_t piece = mode == kOutSwiGLU ? 16 : mode == HWK_OUT_F16 ? 8 : 4;
  return ((uintptr_t)Y & 15) == 0 && N % piece == 0;
}
// KG > 1: strips own, own + KG, ... only.
template <int TM, int TN, bool MX, int KG = 1>
__device__ __forceinline__ void store_strips(const floatx4 (&acc)[TM][TN], const int (&s0)[TN], bool shift,
                                             const uint16_t *__restrict__ S, void *__restrict__ Y, uint32_t M,
                                             uint32_t N, uint32_t r0, uint32_t nw, int lane, int mode, float *st,
                                             int own = 0) {
  constexpr int CW = TN * 16, P32 = CW + 4, P16 = CW + 8, PH = CW / 2 + 8;
  const int r16 = lane & 15, q = lane >> 4;
  float sc[TN];
#pragma unroll
  for (int j = 0; j < TN; j++) sc[j] = MX ? 1.0f : (float)__builtin_bit_cast(f16, S[min(nw + j * 16 + r16, N - 1)]);
  auto value = [&](int i, int j, int r) __attribute__((always_inline)) {
    if constexpr (MX) return shift ? ldexpf(acc[i][j][r], s0[j]) : acc[i][j][r];
    else return acc[i][j][r] * sc[j];
  };
  f16 *h = (f16 *)st;
  if (mode == kOutSwiGLU) {
    // the pairs as store_tile makes them: gate lane rows 0, 1 of its quad, up lane rows 2, 3
    const bool gate = (r16 & 1) == 0;
#pragma unroll
    for (int i = 0; i < TM; i++) {
      if (KG > 1 && i % KG != own) continue;
#pragma unroll
      for (int j = 0; j < TN; j++) {
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] = value(i, j, r);
        const float o0 = __shfl_xor(gate ? v[2] : v[0], 1, 64), o1 = __shfl_xor(gate ? v[3] : v[1], 1, 64);
        const int row = q * 4 + (gate ? 0 : 2), c = (j * 16 + r16) / 2;
        h[row * PH + c] = (f16)swiglu_value(gate ? v[0] : o0, gate ? o0 : v[2]);
        h[(row + 1) * PH + c] = (f16)swiglu_value(gate ? v[1] : o1, gate ? o1 : v[3]);
      }
      wait_lds();
      constexpr int CPR = CW / 16;  // pieces of 8 outputs a row
      for (int c = lane; c < 16 * CPR; c += 64) {
        const int row = c / CPR, k = c % CPR;
        const uint32_t m = r0 + i * 16 + row, n = nw + k * 16;
        if (m < M && n < N) *(u32x4 *)((f16 *)Y + (size_t)m * (N / 2) + n / 2) = *(const u32x4 *)(h + row * PH + k * 8);
      }
    }
  } else if (mode == HWK_OUT_F16) {
#pragma unroll
    for (int i = 0; i < TM; i++) {
      if (KG > 1 && i % KG != own) continue;
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int r = 0; r < 4; r++) h[(q * 4 + r) * P16 + j * 16 + r16] = (f16)f32_value(value(i, j, r));
      wait_lds();
      constexpr int CPR = CW / 8;
      for (int c = lane; c < 16 * CPR; c += 64) {
        const int row = c / CPR, k = c % CPR;
        const uint32_t m = r0 + i * 16 + row, n = nw + k * 8;
        if (m < M && n < N) *(u32x4 *)((f16 *)Y + (size_t)m * N + n) = *(const u32x4 *)(h + row * P16 + k * 8);
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < TM; i++) {
      if (KG > 1 && i % KG != own) continue;
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int r = 0; r < 4; r++) st[(q * 4 + r) * P32 + j * 16 + r16] = value(i, j, r);
      wait_lds();
      constexpr int CPR = CW / 4;
      for (int c = lane; c < 16 * CPR; c += 64) {
        const int row = c / CPR, k = c % CPR;
        const uint32_t m = r0 + i * 16 + row, n = nw + k * 4;
        if (m >= M || n >= N) continue;
        floatx4 v = *(const floatx4 *)(st + row * P32 + k * 4);
        floatx4 *y = (floatx4 *)((float *)Y + (size_t)m * N + n);
        if (mode == HWK_OUT_ADD_F32) v = *y + v;
        *y = v;
      }
    }
  }
}

// The general form's store through LDS: the wave's whole block (RW x CW) into its region st, the values as
// store_strips has them, then 16-byte pieces of its rows to Y (in strips the 128 x 128 MXFP4 tile of four waves
// spills registers). The fp32 rows are padded (P32 = CW + 4 floats) so that the 4 row groups of a write land in
// different banks (P32 = CW where the padded block does not fit); the fp16 rows are not (padding them measured no
// faster: their reads of 16 bytes a lane then conflict). For staged(Y, N, mode).
template <int TM, int TN, int P32>
struct StageRows {
  static constexpr int RW = TM * 16, CW = TN * 16;
  static constexpr int P16 = CW, PH = CW / 2 + 8;  // fp16 rows: full width, SwiGLU half width (padded)
  static constexpr int FLOATS = RW * P32;              // a region, in floats (the largest of the three)
  static_assert(P32 == CW || P32 == CW + 4, "fp32 row stride");
  static_assert(RW * P16 * 2 <= FLOATS * 4 && RW * PH * 2 <= FLOATS * 4, "fp16 rows fit the region");
};
template <int BM, int WM, int TM, int TN, bool MX, int P32>
__device__ __forceinline__ void store_tile_staged(const floatx4 (&acc)[TM][TN], const int (&s0)[TN],
                                                  const uint16_t *__restrict__ S, void *__restrict__ Y, uint32_t M,
                                                  uint32_t N, uint32_t m0, uint32_t nw, int wm, int lane, int mode,
                                                  float *st) {
  using G = StageRows<TM, TN, P32>;
  constexpr int RW = G::RW, CW = G::CW;
  const int r16 = lane & 15, q = lane >> 4;
  const uint32_t r0 = m0 + wm * RW;
  auto value = [&](int i, int j, int r) __attribute__((always_inline)) {
    const float sc = MX ? 1.0f : (float)__builtin_bit_cast(f16, S[min(nw + j * 16 + r16, N - 1)]);
    return MX ? ldexpf(acc[i][j][r], s0[j]) : acc[i][j][r] * sc;
  };
  if (mode == kOutSwiGLU) {
    // the pairs as store_tile makes them: gate lane rows 0, 1 of its quad, up lane rows 2, 3
    f16 *h = (f16 *)st;
    const bool gate = (r16 & 1) == 0;
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int i = 0; i < TM; i++) {
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] = value(i, j, r);
        const float o0 = __shfl_xor(gate ? v[2] : v[0], 1, 64), o1 = __shfl_xor(gate ? v[3] : v[1], 1, 64);
        const int row = i * 16 + q * 4 + (gate ? 0 : 2), c = (j * 16 + r16) / 2;
        h[row * G::PH + c] = (f16)(gate ? swiglu_value(v[0], o0) : swiglu_value(o0, v[2]));
        h[(row + 1) * G::PH + c] = (f16)(gate ? swiglu_value(v[1], o1) : swiglu_value(o1, v[3]));
      }
    wait_lds();
    constexpr int CPR = CW / 16;  // 8 outputs a piece
    for (int c = lane; c < RW * CPR; c += 64) {
      const int row = c / CPR, k = c % CPR;
      const uint32_t m = r0 + row, n = nw + k * 16;
      if (m < M && n < N)
        *(u32x4 *)((f16 *)Y + (size_t)m * (N / 2) + n / 2) = *(const u32x4 *)(h + row * G::PH + k * 8);
    }
  } else if (mode == HWK_OUT_F16) {
    f16 *h = (f16 *)st;
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) h[(i * 16 + q * 4 + r) * G::P16 + j * 16 + r16] = (f16)f32_value(value(i, j, r));
    wait_lds();
    constexpr int CPR = CW / 8;
    for (int c = lane; c < RW * CPR; c += 64) {
      const int row = c / CPR, k = c % CPR;
      const uint32_t m = r0 + row, n = nw + k * 8;
      if (m < M && n < N) *(u32x4 *)((f16 *)Y + (size_t)m * N + n) = *(const u32x4 *)(h + row * G::P16 + k * 8);
    }
  } else {
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) st[(i * 16 + q * 4 + r) * P32 + j * 16 + r16] = value(i, j, r);
    wait_lds();
    constexpr int CPR = CW / 4;
    for (int c = lane; c < RW * CPR; c += 64) {
      const int row = c / CPR, k = c % CPR;
      const uint32_t m = r0 + row, n = nw + k * 4;
      if (m >= M || n >= N) continue;
      floatx4 v = *(const floatx4 *)(st + row * P32 + k * 4);
      floatx4 *y = (floatx4 *)((float *)Y + (size_t)m * N + n);
      if (mode == HWK_OUT_ADD_F32) v = *y + v;
      *y = v;
    }
  }
}

// lds: 2 * BM * CH 16-byte slots of LDS (the X buffers).
template <int BM, int BN, bool MX, int WM, int WN, int KG = 1>
__device__ __forceinline__ void gemm_wg(uint32_t bx, const u32x4 *__restrict__ X, const uint8_t *__restrict__ W,
                                        const uint8_t *__restrict__ E, const uint16_t *__restrict__ S,
                                        void *__restrict__ Y, uint32_t M, uint32_t N, uint32_t K, int mode,
                                        bool equads, u32x4 *lds) {
  using C = Cfg<BM, BN, MX, WM, WN, KG>;
  constexpr int TM = C::TM, TN = C::TN, NT = C::NT, KKG = C::KKG;
  static_assert(KG == 1 || !MX, "k groups here: int8 only");
  static_assert(KG == 1 || BM * BN * 4 <= 2 * BM * CH * 16, "the k groups' sum goes through the X buffers");
  __shared__ int hs[MX ? BN : 1], ls[MX ? BN : 1];  // the row shift scan (MXFP4)
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int g = wave / (WM * WN), wl = wave % (WM * WN);  // k group, wave in the group
  const int wm = wl / WN, wn = wl % WN;
  const int r16 = lane & 15, q = lane >> 4;
  uint32_t tm, tn;
  tile_of(bx, (M + BM - 1) / BM, (N + BN - 1) / BN, tm, tn);
  const uint32_t m0 = tm * BM, n0 = tn * BN;
  const uint32_t nw = n0 + wn * (BN / WN);  // the wave's first column
  uint32_t brow[TN];
#pragma unroll
  for (int j = 0; j < TN; j++) brow[j] = min(nw + j * 16 + r16, N - 1);

  const uint32_t steps = (K + KS - 1) / KS;
  auto kofs = [&](uint32_t j) -> uint32_t { return min(j, steps) * KS; };  // past the end: reads zeros
  Stage<BM, BN, MX, WM, WN, KG> st[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) {
    load_x<BM, BN, MX, WM, WN, KG>(st[s], X, M, K, m0, kofs(s), t);
    load_w<BM, BN, MX, WM, WN, KG>(st[s], W, E, K, kofs(s), brow, q, g);
  }
  int s0[TN];
#pragma unroll
  for (int j = 0; j < TN; j++) s0[j] = 0;
  if constexpr (MX) {
    if (t < BN) {
      hs[t] = 0;
      ls[t] = 255;
    }
    __syncthreads();
    scan_shifts<BN, NT>(E, n0, N, K / 32, equads, t, hs, ls);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const uint32_t r = brow[j] - n0;
      s0[j] = shift_of(hs[r], ls[r]);
    }
  }

  floatx4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) acc[i][j] = (floatx4){0.0f, 0.0f, 0.0f, 0.0f};

  // Steps in groups of NS (a partial last group multiplies zeros: its loads read past K). A step:
  // its X slab into LDS, barrier, the next X loads of its stage, then for each kk its weight operands
  // converted next to the MFMAs that take them (the VALU work overlaps the matrix core), then the
  // next weight loads of its stage. Issue order is pinned: the wait counter is in order, so a stage
  // consumed before the loads behind it is waited for without waiting for them.
  for (uint32_t j0 = 0; j0 < steps; j0 += NS) {
#pragma unroll
    for (int s = 0; s < NS; s++) {
      const uint32_t j = j0 + s;
      u32x4 *buf = lds + (s & 1) * (BM * CH);  // NS is even: step j uses buffer j & 1
      if (st[s].k0 + KS > K) zero_tail<BM, BN, MX, WM, WN, KG>(st[s], K, t, q, g);  // uniform: only a ragged step
#pragma unroll
      for (int i = 0; i < C::AL; i++) {
        const int c = t + NT * i, row = c / CH, ch = c % CH;
        buf[row * CH + (ch ^ (row & 15))] = st[s].a[i];
      }
      __syncthreads();
      issue_order();
      load_x<BM, BN, MX, WM, WN, KG>(st[s], X, M, K, m0, kofs(j + NS), t);
      issue_order();
      float sc[TN];
#pragma unroll
      for (int jn = 0; jn < TN; jn++) sc[jn] = MX ? shifted_scale(st[s].e[jn], s0[jn]) : 0.0f;
      // the operands of kk + 1 (X from LDS, weights converted) are fetched before the MFMAs of kk; kk
      // counts the group's MFMAs (the step's MFMA g*KKG + kk)
      auto operands = [&](half8 (&af)[TM], half8 (&bf)[TN], int kk) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TM; i++) {
          const int row = wm * (BM / WM) + i * 16 + r16;
          const int ch = KG == 1 ? xchunk<MX>(q, kk) : xchunk<MX>(q, g * KKG + kk);
          af[i] = __builtin_bit_cast(half8, buf[row * CH + (ch ^ (row & 15))]);
        }
#pragma unroll
        for (int jn = 0; jn < TN; jn++) {
          if constexpr (MX) {
            bf[jn] = fp4x8_to_half8(st[s].b[jn][0][kk], sc[jn]);
          } else {
            const u32x4 v = st[s].b[jn][kk >> 1];  // KG = 2: the group's half, loaded alone
            bf[jn] = i8x8_to_half8(v[(kk & 1) * 2], v[(kk & 1) * 2 + 1]);
          }
        }
      };
      half8 af[2][TM], bf[2][TN];
      operands(af[0], bf[0], 0);
#pragma unroll
      for (int kk = 0; kk < KKG; kk++) {
        if (kk + 1 < KKG) operands(af[(kk + 1) & 1], bf[(kk + 1) & 1], kk + 1);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int jn = 0; jn < TN; jn++)
            acc[i][jn] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[kk & 1][i], bf[kk & 1][jn], acc[i][jn], 0, 0, 0);
      }
      issue_order();
      load_w<BM, BN, MX, WM, WN, KG>(st[s], W, E, K, kofs(j + NS), brow, q, g);
      issue_order();
    }
  }
  if constexpr (KG == 2) {
    // group 1's accumulators to group 0 through the X buffers (every wave is done with them after
    // the barrier), summed in group 0, which writes the tile
    floatx4 *red = (floatx4 *)lds;
    __syncthreads();
    if (g == 1) {
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) red[((wl * TM + i) * TN + j) * 64 + lane] = acc[i][j];
    }
    __syncthreads();
    if (g == 0) {
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] += red[((wl * TM + i) * TN + j) * 64 + lane];
    }
    __syncthreads();  // group 0 is done with the sums' buffers, which its stores reuse
    if (g == 1) return;
  }
  if (staged(Y, N, mode)) {
    // a wave's block in region wl of the X buffers (rows padded where that fits)
    constexpr int CW = TN * 16, PAD = WM * WN * TM * 16 * (CW + 4) <= 2 * BM * CH * 4 ? CW + 4 : CW;
    using G = StageRows<TM, TN, PAD>;
    static_assert(WM * WN * G::FLOATS <= 2 * BM * CH * 4, "the staged blocks fit the X buffers");
    if constexpr (KG == 1) __syncthreads();  // every wave is done with the X buffers
    store_tile_staged<BM, WM, TM, TN, MX, PAD>(acc, s0, S, Y, M, N, m0, nw, wm, lane, mode,
                                               (float *)lds + wl * G::FLOATS);
    return;
  }
  store_tile<BM, WM, TM, TN, MX>(acc, s0, S, Y, M, N, m0, nw, wm, r16, q, mode);
}


// ---- The paired form (K a multiple of 64): two workgroups a CU ----
//
// K goes 64 at a time through a ring of three LDS stages, X and the weights straight from memory into LDS
// (global_load_lds: lane i of an instruction writes 16 bytes at the instruction's LDS base + 16 i), two
// steps ahead, waited for by an explicit count (the wait counter is in order, and a wave issues the same
// number of loads every step: past the last step they reread in-range data into a stage nobody reads).
// A step is one barrier, the operand reads and the MFMAs; nothing is carried in registers but the
// accumulators, so that a wave fits 128 registers and a CU holds two workgroups: while one waits at its
// barrier, scans or stores its tile (the SwiGLU's float64 exp), the other's MFMAs run.
// A lane's operands of a step are the 16 values q*16 .. +15 of a row's 64, in every tile and for both kinds of
// weights: tiles agree bit for bit given the same segments of K (the code object's kernels, in one tile shape, add
// the segments that the library's tile has as k groups).
// The swizzles are applied on the source side (which 16-byte chunk a lane fetches), so that the lanes of an LDS read
// that are served at once land in distinct banks. A 16-byte read does not serve 16 neighbouring lanes, but four rows
// of each quarter of the 16, out of two neighbouring lane groups q, q ^ 1 (what the conflict counter tells: swizzles
// by row >> 1 and column >> 2, right for 16 neighbours, cost every read twice its cycles). So bit 0 of row >> 1 moves
// the chunk's bit 1, the one that q ^ 1 flips, and the quarters the other two; int8 columns: the bit that it does not.
//   X   slot p: row p / 8, chunk (p % 8) ^ x_swizzle(row)                  (128-byte rows)
//   W   int8   slot p: column p / 4, chunk (p % 4) ^ ((column >> 2) & 2)   (64-byte columns)
//       MXFP4  slot p: column p / 2, chunk (p % 2) ^ ((column >> 3) & 1)   (32-byte columns)
//   E   (MXFP4) dword p: column p, the step's two scale bytes
// int8 512 x 6144 x 2048: 2,015,232 -> 49,152 conflict cycles a launch (the rest the store's), 17.06 -> 16.88 us a call; the
// MXFP4 weights' reads, two 8-byte ones in an instruction, still count four cycles each.
__device__ __forceinline__ uint32_t x_swizzle(uint32_t row) { return ((row >> 2) & 1) | (row & 2) | ((row >> 1) & 4); }

// A tile of the paired form: BM x BN, WM x WN waves a k group, KG k groups, RS ring stages, the workgroups of
// it that a CU holds (res), and the picoseconds of a CU that the tile takes a value of K (ps).
struct PairTile {
  uint16_t bm, bn, wm, wn, kg, rs, res, ps;
};
#define HWK_PAIR_MX(F)                                                                                       \
  F(128, 256, 2, 4, 1, 3, 2, 14261) F(128, 192, 2, 4, 1, 3, 2, 11273) F(128, 128, 2, 2, 2, 3, 1, 8300)       \
  F(128, 64, 4, 2, 2, 3, 1, 5439) F(96, 64, 2, 2, 2, 3, 1, 4141) F(64, 64, 2, 2, 2, 3, 2, 3048)              \
  F(32, 64, 2, 2, 4, 4, 1, 2404) F(32, 32, 2, 1, 4, 4, 1, 1350) F(16, 32, 1, 2, 8, 4, 1, 1070)
#define HWK_PAIR_I8(F)                                                                                       \
  F(128, 128, 2, 4, 1, 3, 2, 8075) F(128, 128, 2, 4, 2, 3, 1, 8000) F(128, 96, 2, 3, 2, 3, 1, 6578)          \
  F(128, 64, 4, 2, 2, 3, 1, 5461) F(64, 64, 2, 2, 2, 3, 2, 2854) F(32, 64, 2, 2, 4, 3, 1, 2128)              \
  F(32, 32, 2, 2, 4, 4, 1, 1391) F(16, 32, 1, 2, 8, 4, 1, 769)

// The tile of least cost for Y (m, n) over k, an index into HWK_PAIR_MX or HWK_PAIR_I8. The cost is that of
// the busiest of the 256 CUs: ps * k for each of its tiles, and 3.9 us (prologue, the first loads' latency,
// the groups' sums and the stores) for each round of res tiles. Both constants are fitted to the tiles' measured
// times. Every tile on 224 shapes, m 9..8192, n 512..16384, k 512..8192: the tile picked takes on average 1.011
// (MXFP4) and 1.005 (int8) of the time of the table's best, 1.22 and 1.26 at most, and 0.58 and 0.60 (most 0.97 and
// 1.01) of the one-workgroup-a-CU tiles of 64..128 rows that stood here before. (int8 128 x 128 in two k groups is set
// just below the one-group tile: with one tile a CU it takes 0.94-0.97 of its time from k = 2,048 on, 1.06 at 512.)
// Integer arithmetic, so that the host and a kernel agree.
__host__ __device__ __forceinline__ int pick_pair(bool mx, uint32_t m, uint32_t n, uint32_t k) {
#define HWK_TILE(...) {__VA_ARGS__},
  constexpr PairTile kMx[] = {HWK_PAIR_MX(HWK_TILE)}, kI8[] = {HWK_PAIR_I8(HWK_TILE)};
#undef HWK_TILE
  constexpr int kNMx = sizeof kMx / sizeof kMx[0], kNI8 = sizeof kI8 / sizeof kI8[0];
  int best = 0;
  uint64_t best_cost = ~0ull;
  for (int i = 0; i < (mx ? kNMx : kNI8); i++) {
    const PairTile t = mx ? kMx[i] : kI8[i];
    const uint64_t tiles = (uint64_t)((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn);
    const uint64_t most = (tiles + 255) / 256;  // tiles of the busiest CU
    const uint64_t cost = most * t.ps * k + (most + t.res - 1) / t.res * 3900000ull;
    if (cost < best_cost) {
      best_cost = cost;
      best = i;
    }
  }
  return best;
}
// The k groups of the tile picked.
__host__ __device__ __forceinline__ uint32_t pair_groups(bool mx, uint32_t m, uint32_t n, uint32_t k) {
  const int i = pick_pair(mx, m, n, k);
#define HWK_KG(bm, bn, wm, wn, kg, rs, res, ps) kg,
  constexpr uint8_t kMx[] = {HWK_PAIR_MX(HWK_KG)}, kI8[] = {HWK_PAIR_I8(HWK_KG)};
#undef HWK_KG
  return mx ? kMx[i] : kI8[i];
}
// Whether the paired form takes a product: whole steps of 64 values, scale bytes readable two at a time, and
// its loads' 32-bit byte offsets.
__host__ __device__ __forceinline__ bool pair_takes(bool mx, uint32_t m, uint32_t n, uint32_t k, const void *e) {
  return k % 64 == 0 && (!mx || ((uintptr_t)e & 1) == 0) && (uint64_t)m * k * 2 < (1ull << 32) &&
         (uint64_t)n * (mx ? k / 2 : k) < (1ull << 32);
}

template <int BM, int BN, bool MX, int WM, int WN, int KG, int RS>
struct PairCfg {
  static constexpr int NW = WM * WN, NT = 64 * NW * KG;  // waves a group; threads
  static constexpr int TM = BM / WM / 16, TN = BN / WN / 16;
  static constexpr int WCH = MX ? 2 : 4;                   // 16-byte weight chunks a column a step
  static constexpr int XI = BM * 8 / 64, WI = BN * WCH / 64, EI = MX ? (BN + 63) / 64 : 0;  // load instructions a step
  static constexpr int XB = BM * 8, WB = BN * WCH, EB = EI * 16;  // 16-byte slots a stage
  static constexpr int AX = (XI + NW - 1) / NW, AW = (WI + NW - 1) / NW, AE = (EI + NW - 1) / NW;
  static constexpr int LMIN = XI / NW + WI / NW + EI / NW;  // the fewest loads a wave issues a step
  static constexpr int SLOTS = XB + WB + EB;               // a stage
  static constexpr int STRIP = 16 * (TN * 16 + 4);         // floats of a wave's store strip
  static constexpr int SUMS = KG > 1 ? KG * BM * BN : 0;   // floats of the groups' tiles
  static_assert(TM * WM * 16 == BM && TN * WN * 16 == BN && BM % 8 == 0 && BN * WCH % 64 == 0, "tile shape");
  static constexpr int ENDS = ((SUMS > NW * KG * STRIP ? SUMS : NW * KG * STRIP) + 3) / 4;  // 16-byte slots after the loop
  static constexpr int LDS = KG * RS * SLOTS > ENDS ? KG * RS * SLOTS : ENDS;
  static_assert(LMIN * (RS - 2) + 3 * (RS - 2) <= 63, "loads in flight past the wait counter");
};

// Workgroup id -> tile. Ids x, x+8, x+16, ... share an XCD: each XCD takes a contiguous run of the order
// below, in which the tiles that run at the same time form a block of kGroupN weight panels by some M tiles,
// so that each step's X rows and weights are fetched into the XCD's L2 once for all of them. False: no
// tile (the grid is rounded up to 8).
constexpr uint32_t kGroupN = 8;
__host__ __device__ __forceinline__ uint32_t pair_grid(uint32_t tiles) { return (tiles + 7) / 8 * 8; }
__device__ __forceinline__ bool pair_tile(uint32_t id, uint32_t mt, uint32_t nt, uint32_t &tm, uint32_t &tn) {
  const uint32_t total = mt * nt, per = (total + 7) / 8;
  const uint32_t lin = (id % 8) * per + id / 8;
  if (lin >= total) return false;
  const uint32_t gr = lin / (kGroupN * mt), r = lin - gr * kGroupN * mt;
  const uint32_t gn = min(kGroupN, nt - gr * kGroupN);  // panels of the last group
  tm = r / gn;
  tn = gr * kGroupN + r % gn;
  return true;
}

// rings: PairCfg::LDS 16-byte slots of LDS. SEG (one k group, a grid of exactly the tiles, in tile_of's order): the
// sums of nseg segments of K (seg_first) are added in order, as another tile's k groups' are. (The segment's end is
// found once a segment: seg_first divides.)
template <int BM, int BN, bool MX, int WM, int WN, int KG, int RS, bool SEG = false>
__device__ __forceinline__ void gemm_pair_wg(uint32_t bx, const u32x4 *__restrict__ X, const uint8_t *__restrict__ W,
                                             const uint8_t *__restrict__ E, const uint16_t *__restrict__ S,
                                             void *__restrict__ Y, uint32_t M, uint32_t N, uint32_t K, int mode,
                                             bool equads, u32x4 *rings, uint32_t nseg = 1) {
  using C = PairCfg<BM, BN, MX, WM, WN, KG, RS>;
  constexpr int TM = C::TM, TN = C::TN, NT = C::NT, NW = C::NW, SLOTS = C::SLOTS;
  static_assert(!SEG || KG == 1, "segments in one k group");
  __shared__ uint32_t flags[NW * KG];
  const int t = threadIdx.x, lane = t & 63, wg = __builtin_amdgcn_readfirstlane(t >> 6);
  const int g = wg / NW, wave = wg % NW;  // k group, wave in the group
  u32x4 *ring = rings + g * RS * SLOTS;
  const int wm = wave / WN, wn = wave % WN;
  const int r16 = lane & 15, q = lane >> 4;
  uint32_t tm, tn;
  if constexpr (SEG) tile_of(bx, (M + BM - 1) / BM, (N + BN - 1) / BN, tm, tn);
  else if (!pair_tile(bx, (M + BM - 1) / BM, (N + BN - 1) / BN, tm, tn)) return;
  const uint32_t m0 = tm * BM, n0 = tn * BN;
  const uint32_t nw = n0 + wn * (BN / WN);  // the wave's first column
  // the group's steps of 64 are h0 .. h1-1; all groups run n_steps of them together (a step past a group's
  // segment loads in-range data that nothing reads)
  const uint32_t steps = K / 64, S128 = (steps + 1) / 2;
  const uint32_t h0 = KG == 1 ? 0 : 2 * seg_first(S128, KG, g);
  const uint32_t h1 = KG == 1 ? steps : min(2 * seg_first(S128, KG, g + 1), steps);
  const uint32_t n_steps = KG == 1 ? steps : 2 * ((S128 + KG - 1) / KG);

  // the lane's byte offsets of its loads from the operand's start plus the step's K offset (32-bit: the
  // launcher takes this form for operands under 4 GiB); rows and columns past the end read the last
  uint32_t xo[C::AX], wo[C::AW], eo[C::AE > 0 ? C::AE : 1];
#pragma unroll
  for (int a = 0; a < C::AX; a++) {
    const int p = (a * NW + wave) * 64 + lane, row = p / 8, ch = (p % 8) ^ x_swizzle(row);
    xo[a] = (min(m0 + row, M - 1) * K + ch * 8) * 2;
  }
#pragma unroll
  for (int a = 0; a < C::AW; a++) {
    const int p = (a * NW + wave) * 64 + lane, col = p / C::WCH;
    const int c = (p % C::WCH) ^ (MX ? (col >> 3) & 1 : (col >> 2) & 2);
    wo[a] = min(n0 + col, N - 1) * (MX ? K / 2 : K) + c * 16;
  }
#pragma unroll
  for (int a = 0; a < C::AE; a++) eo[a] = min(n0 + (uint32_t)((a * NW + wave) * 64 + lane), N - 1) * (K / 32);
  auto load = [&](uint32_t j, int s) __attribute__((always_inline)) {
    const uint32_t k0 = min(h0 + j, steps - 1) * 64;
    u32x4 *xb = ring + s * SLOTS, *wb = xb + C::XB;
    uint32_t *eb = (uint32_t *)(wb + C::WB);
#pragma unroll
    for (int a = 0; a < C::AX; a++)
      if (C::XI % NW == 0 || a * NW + wave < C::XI)
        to_lds16((const char *)X + k0 * 2, xo[a], lds_at(xb + (a * NW + wave) * 64));
#pragma unroll
    for (int a = 0; a < C::AW; a++)
      if (C::WI % NW == 0 || a * NW + wave < C::WI)
        to_lds16((const char *)W + (MX ? k0 / 2 : k0), wo[a], lds_at(wb + (a * NW + wave) * 64));
#pragma unroll
    for (int a = 0; a < C::AE; a++)
      if (C::EI % NW == 0 || a * NW + wave < C::EI)
        to_lds2((const char *)E + k0 / 32, eo[a], lds_at(eb + (a * NW + wave) * 64));
  };
  // this wave's loads of all steps but the last RS - 2 issued done
  const int extra = (wave < C::XI % NW) + (wave < C::WI % NW) + (wave < C::EI % NW);
  auto wait_step = [&]() __attribute__((always_inline)) {
    if (extra == 0) wait_loads<C::LMIN * (RS - 2)>();
    else if (extra == 1) wait_loads<(C::LMIN + 1) * (RS - 2)>();
    else if (extra == 2) wait_loads<(C::LMIN + 2) * (RS - 2)>();
    else wait_loads<(C::LMIN + 3) * (RS - 2)>();
  };

  floatx4 acc[TM][TN], total[SEG ? TM : 1][SEG ? TN : 1];
  int s0[TN];
  uint32_t lo = 103, hi = 140;  // the least scale byte less one (a zero one, which needs no shift, wraps), the largest
#pragma unroll
  for (int j = 0; j < TN; j++) s0[j] = 0;
  // the lane's operands in a stage: X rows of 16 apart, weight columns of 16 apart
  const uint32_t xa = (wm * (BM / WM) + r16) * 128, wa = (wn * (BN / WN) + r16) * (C::WCH * 16);
  const uint32_t xsw = x_swizzle(r16);
  const uint32_t wsl = MX ? (((q >> 1) ^ ((r16 >> 3) & 1)) * 16 + (q & 1) * 8) : (q ^ ((r16 >> 2) & 2)) * 16;
  const uint32_t ea = (wn * (BN / WN) + r16) * 4 + (q >> 1);
  auto main_loop = [&](auto shifted) __attribute__((always_inline)) {
    constexpr bool SHIFT = decltype(shifted)::value;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++) acc[i][j] = (floatx4){0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t seg = 0, seg_end = 0;  // the segment, the step after its last
    auto seg_ends = [&](uint32_t g) { return min(2 * seg_first(S128, nseg, g + 1), steps); };
    if constexpr (SEG) {
      while ((seg_end = seg_ends(seg)) == 0) seg++;  // (empty ones)
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) total[i][j] = (floatx4){0.0f, 0.0f, 0.0f, 0.0f};
    }
#pragma unroll
    for (int s = 0; s < RS - 1; s++) load(s, s);
    for (uint32_t j0 = 0; j0 < n_steps; j0 += RS) {
#pragma unroll
      for (int s = 0; s < RS; s++) {
        const uint32_t j = j0 + s;
        if (j >= n_steps) break;
        // every wave's loads of step j landed, every wave done with step j-1's stage, which step j+RS-1 takes
        wait_step();
        wait_lds();
        bare_barrier();
        issue_order();
        load(j + RS - 1, (s + RS - 1) % RS);
        issue_order();
        if (KG > 1 && h0 + j >= h1) continue;
        const char *xb = (const char *)(ring + s * SLOTS), *wb = xb + C::XB * 16, *eb = wb + C::WB * 16;
        u32x2 wc[MX ? TN : 1];
        u32x4 wv[MX ? 1 : TN];
        float sc[TN];
#pragma unroll
        for (int jn = 0; jn < TN; jn++) {
          if constexpr (MX) {
            wc[jn] = *(const u32x2 *)(wb + wa + jn * 16 * 32 + wsl);
            const uint32_t e = *(const uint8_t *)(eb + ea + jn * 64);
            sc[jn] = SHIFT ? shifted_scale(e, s0[jn]) : __uint_as_float(e << 23);
            if constexpr (!SHIFT) {
              lo = min(lo, e - 1u);
              hi = max(hi, e);
            }
          } else {
            wv[jn] = *(const u32x4 *)(wb + wa + jn * 16 * 64 + wsl);
          }
        }
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
          half8 af[TM], bf[TN];
#pragma unroll
          for (int i = 0; i < TM; i++)
            af[i] = __builtin_bit_cast(half8, *(const u32x4 *)(xb + xa + i * 16 * 128 + ((2 * q + kk) ^ xsw) * 16));
#pragma unroll
          for (int jn = 0; jn < TN; jn++) {
            if constexpr (MX) bf[jn] = fp4x8_to_half8(wc[jn][kk], sc[jn]);
            else bf[jn] = i8x8_to_half8(wv[jn][kk * 2], wv[jn][kk * 2 + 1]);
          }
#pragma unroll
          for (int i = 0; i < TM; i++)
#pragma unroll
            for (int jn = 0; jn < TN; jn++)
              acc[i][jn] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[i], bf[jn], acc[i][jn], 0, 0, 0);
        }
        if constexpr (SEG) {
          if (j + 1 == seg_end) {
            do seg_end = seg_ends(++seg);
            while (seg < nseg && seg_end == j + 1);  // (empty ones)
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
              for (int jn = 0; jn < TN; jn++) {
                total[i][jn] += acc[i][jn];
                acc[i][jn] = (floatx4){0.0f, 0.0f, 0.0f, 0.0f};
              }
          }
        }
      }
    }
    wait_loads<0>();  // no load into LDS may land in a stage put to another use
    if constexpr (SEG) {
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = total[i][j];
    }
  };
  main_loop(std::false_type{});
  bool shift = false;
  if constexpr (MX) {
    // a scale whose exponent leaves [-23, 13] (or an infinite one): the tile again, its rows shifted
    if (__ballot(lo < 103 || hi > 140)) shift = true;
    if (lane == 0) flags[wg] = shift;
  }
  wait_lds();
  bare_barrier();  // every wave is done with the stages
  if constexpr (MX) {
    shift = false;
#pragma unroll
    for (int w = 0; w < NW * KG; w++) shift |= flags[w] != 0;
    shift = __builtin_amdgcn_readfirstlane(shift);
    if (shift) {
      int *hs = (int *)rings, *ls = hs + BN;
      for (int i = t; i < BN; i += NT) {
        hs[i] = 0;
        ls[i] = 255;
      }
      __syncthreads();
      scan_shifts<BN, NT>(E, n0, N, K / 32, equads, t, hs, ls);
      __syncthreads();
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const uint32_t r = min(nw + j * 16 + r16, N - 1) - n0;
        s0[j] = shift_of(hs[r], ls[r]);
      }
      __syncthreads();
      main_loop(std::true_type{});
      wait_lds();
      bare_barrier();
    }
  }
  if constexpr (KG > 1) {
    // the groups' tiles through LDS: the wave of group g sums rows i = g, g + KG, ... (16 each) of its block,
    // in the order of the segments, and stores them
    floatx4 *sums = (floatx4 *)rings;
#pragma unroll
    for (int i = 0; i < TM; i++) {
      if (i % KG == g) continue;
#pragma unroll
      for (int j = 0; j < TN; j++) sums[(((g * NW + wave) * TM + i) * TN + j) * 64 + lane] = acc[i][j];
    }
    wait_lds();
    bare_barrier();
#pragma unroll
    for (int i = 0; i < TM; i++) {
      if (i % KG != g) continue;
#pragma unroll
      for (int j = 0; j < TN; j++) {
        floatx4 v;
#pragma unroll
        for (int k = 0; k < KG; k++) {
          const floatx4 p = k == g ? acc[i][j] : sums[(((k * NW + wave) * TM + i) * TN + j) * 64 + lane];
          v = k == 0 ? p : v + p;
        }
        acc[i][j] = v;
      }
    }
    wait_lds();
    bare_barrier();  // the sums are read: the store strips take their place
  }
  if (staged(Y, N, mode))
    store_strips<TM, TN, MX, KG>(acc, s0, shift, S, Y, M, N, m0 + wm * (BM / WM), nw, lane, mode,
                                 (float *)rings + wg * C::STRIP, g);
  else
    store_tile<BM, WM, TM, TN, MX, KG>(acc, s0, S, Y, M, N, m0, nw, wm, r16, q, mode, g);
}

}  // namespace hwk_gemm
