// int8 ConvRot linear on tiled operands: the DiT's fast path.
//
// Operand layouts (16-byte chunks; each 64x64 tile image is what one LDS stage holds per
// 64-row block):
//   A (rotated fp16 activations), written by the producing row kernel:
//     At[ceil(M/64)][K/64][8 k-chunks][64 rows][8 halfs]       (8 KB per 64x64 tile)
//   W (int8 ConvRot weights), re-tiled once after upload (ns2_tile_i8_weight), each byte
//   stored biased as u = w + 128:
//     Wt[N/64][K/64][8 k-chunks][64 rows][8 bytes]            (4 KB per 64x64 tile)
//   or W (bf16 weights of the plain linears), re-tiled once as fp16 (ns2_tile_bf16_weight) in
//   the layout of A:
//     Wt[N/64][K/64][8 k-chunks][64 rows][8 halfs]            (8 KB per 64x64 tile)
// Tiles move into LDS as 1 KB blocks with direct global->LDS copies (no registers, no LDS
// stores) into a ring of LDS stages, and the MFMA fragment reads are conflict-free: the 32
// lanes of a half-wave read 32 consecutive 16-byte (A) or 8-byte (W) rows. The int8
// weights are decoded to fp16 as they are read from LDS into the MFMA B operand (exact:
// half(0x6400 | u) - 1152 = w for |w| <= 128), and the per-output-row scale is applied in
// the epilogue, in the reference's order (app/gpu/gemm.js:159-164).
#pragma once
#include <type_traits>

#include "ns2_common.h"

namespace ns2tiled {

using namespace ns2dev;

struct TGemmArgs {
  const half_t* At;   // tiled, or the rows of kI8Rows (lda halfs apart)
  const uint8_t* Wt;  // tiled, or the int8 rows of kI8Rows
  const float* scale;
  const float* bias;
  float* C;
  uint16_t* Y;  // GLU epilogue: rotated fp16 output in the tiled layout, N/2 columns
  const float* gate;
  long long cOff, gOff;
  int M, N, K, ldc;
  int mblocks, nblocks;  // 64-row blocks of A (rounded up) and W
  int tiles_m, tiles_n;  // block tiles
  float alpha;
  int act, resid;
  // LoRA side path: lt fp32 [M][lr] (the down-projected input), lb fp16 [N][lr] (up-projections,
  // original row order, strengths folded), lr % 32 == 0; lr = 0 without LoRA
  const float* lt;
  const half_t* lb;
  int lr;
  // split-K (plain epilogue only): block (tile, z) sums k-tiles [z * ksplit, (z + 1) * ksplit)
  // into part[z] ([M, N] fp32, no epilogue); tiled_splitk_reduce_kernel adds the splits in z
  // order and applies the epilogue. part = nullptr: no split.
  float* part;
  int ksplit;
  // column bands of the tile order (block_tile): 1 keeps the row-group order
  int bands;
  // Packed attention values (plain store only): output columns [vcol0, vcol0 + heads * vD) are
  // written as fp16 into vpk in the flash kernel's value layout, [head][key tile][8 key chunks]
  // [vD][8] with vtiles 64-key tiles per head (key r = output row r), instead of into C.
  // vpk = nullptr: off. vcol0 and vD are multiples of 32 and M of 16.
  half_t* vpk;
  int vcol0, vD, vtiles;
  int lda;
};

// A launch's operands: tiled fp16 rows with int8 or fp16 weight tiles, or fp16 rows and int8 weight rows as
// they lie (K contiguous).
enum Ops { kI8, kF16, kI8Rows };

// 8 biased bytes (two dwords) -> 8 halfs: byte u -> half(0x6400 | u) - 1152 = u - 128 = w.
// v_perm picks bytes of {x, 0x64646464}: selector bytes 4..7 are x's bytes, 0 is 0x64.
__device__ __forceinline__ half8_t u8x8_to_h8(uint2 w) {
  const half2_t off = {(half_t)1152.0f, (half_t)1152.0f};
  half8_t r;
  const uint32_t ws[2] = {w.x, w.y};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint32_t lo = __builtin_amdgcn_perm(ws[i], 0x64646464u, 0x00050004u);
    const uint32_t hi = __builtin_amdgcn_perm(ws[i], 0x64646464u, 0x00070006u);
    const half2_t l = __builtin_bit_cast(half2_t, lo) - off;
    const half2_t h = __builtin_bit_cast(half2_t, hi) - off;
    r[4 * i + 0] = l[0];
    r[4 * i + 1] = l[1];
    r[4 * i + 2] = h[0];
    r[4 * i + 3] = h[1];
  }
  return r;
}

// One output: (acc * alpha) * rs + bi, activation, then store or add into the residual `old`
// (gated by gt) in the reference's order (app/gpu/gemm.js:159-164).
template <int ACT>
__device__ __forceinline__ float act_t(float x) {
  if (ACT == NS2_ACT_SILU) return silu(x);
  if (ACT == NS2_ACT_GELU_TANH) return gelu_tanh(x);
  return x;
}

// The GLU epilogue's gate activation. SiLU's quotient as the reciprocal's, corrected once by its residual
// (5 instructions; the division's scaling steps for quotients out of range make it 10, which were a
// third of the epilogue's vector instructions; 3952 x 8192 x 1536: 102.6 -> 101.0 us, the uncorrected
// product 100.2). Compared with the division for all 2^32 inputs: the same bits for every result above
// 1e-35, at most 1e-36 off below.
template <int ACT>
__device__ __forceinline__ float glu_act(float x) {
  if (ACT == NS2_ACT_SILU) {
    const float d = 1.0f + __expf(-x), r = __builtin_amdgcn_rcpf(d), q = x * r;
    return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-d, q, x), r, q), d, x);
  }
  return act_t<ACT>(x);
}

// XCD-aware tile order: consecutive block ids go to different XCDs (round-robin dispatch);
// block i is given tile start(x) + i/8 of XCD x = i % 8, where XCD x owns the contiguous range
// of T/8 (+1 for the first T%8 XCDs) tiles of a linear tile order, so neighbouring tiles
// (sharing A rows and W columns) run on the same XCD and meet in its L2. The linear order:
//  * bands > 1: column bands of ceil(tiles_n / bands) tiles, band by band, rows within a band,
//    N fastest. An XCD's range is then a 2-D block of one band, whose weight slice (sized on
//    the host to about half an L2) stays resident while its rows stream through once;
//  * bands = 1: N fastest inside groups of 4 row-tiles (A reuse in L2), for weights that fit.
__device__ __forceinline__ void block_tile(const TGemmArgs& p, int& tm, int& tn) {
  const int tiles = p.tiles_m * p.tiles_n;
  const int x = blockIdx.x % 8, local = blockIdx.x / 8;
  const int q = tiles / 8, rmd = tiles % 8;
  const int tile = x * q + (x < rmd ? x : rmd) + local;
  if (p.bands > 1) {
    const int bw = (p.tiles_n + p.bands - 1) / p.bands;
    const int band = tile / (bw * p.tiles_m), rem = tile % (bw * p.tiles_m);
    const int w = p.tiles_n - band * bw < bw ? p.tiles_n - band * bw : bw;  // the last band may be narrower
    tm = rem / w;
    tn = band * bw + rem % w;
    return;
  }
  const int group = 4;
  const int gsize = group * p.tiles_n;
  const int g = tile / gsize, rem = tile % gsize;
  const int rows_in_g = (p.tiles_m - g * group) < group ? (p.tiles_m - g * group) : group;
  tm = g * group + rem % rows_in_g;
  tn = rem / rows_in_g;
}

// The epilogues below work on a wave's sums acc[i][j][r] = C[mw + 32i + 8(r/4) + 4hi + r%4][nw + 32j + lq]
// (mw, nw the wave's first row and column, both uniform; lq = lane % 32, hi = lane / 32). Rows are
// addressed as a uniform pointer plus a lane offset of 64 bits (4 ldc may exceed 32). Every value loaded for an epilogue is
// waited for once, before the first store (pin): the stores then issue back to back. With the
// wait inside a per-row branch the compiler drained every earlier store before each one, and the
// stores of a wave ran one memory round trip after another.
__device__ __forceinline__ void pin(float& x) { asm volatile("" : "+v"(x)); }

// Old outputs of tile (i, j); rows past M read the last one (their results are dropped).
__device__ __forceinline__ void load_old(const TGemmArgs& p, float (&old)[16], int mw, int nw, int lq, int hi) {
  const float* base = p.C + p.cOff + (long long)mw * p.ldc + nw;
  const int rows = p.M - mw;
  if (rows >= 32) {
    const long long lane_off = 4LL * hi * p.ldc + lq;
#pragma unroll
    for (int r = 0; r < 16; ++r) old[r] = (base + (long long)(8 * (r >> 2) + (r & 3)) * p.ldc)[lane_off];
    return;
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    int dm = 8 * (r >> 2) + 4 * hi + (r & 3);
    dm = dm < rows ? dm : (rows > 0 ? rows - 1 : 0);
    old[r] = base[(long long)dm * p.ldc + lq];
  }
}

// Plain epilogue of one wave (EPI 0). Per column: scale, bias and gate; per element the
// arithmetic of gemm.js:159-164, with the row check only in tiles that cross M. RM 0 stores, RM 1
// adds (gate times) the result (no gate: times 1, the same sum); old outputs come from cold when
// PRE_C, else they are loaded here one tile ahead of the tile being stored.
// LORA: the low-rank term of each tile (lora_tile) is added after the bias.
template <int TM, int TN, int ACT, int RM, bool PRE_C, bool LORA, int CI, int CJ>
__device__ __forceinline__ void store_plain(const TGemmArgs& p, const float16_t (&acc)[TM][TN],
                                            const float (&cold)[CI][CJ][16], int mw, int nw, bool full, int lq, int hi) {
  if (mw >= p.M) return;
  float rs[TN], bi[TN], gt[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const bool in = nw + 32 * j < p.N;  // N is a multiple of 64: uniform per column tile
    const int n = in ? nw + 32 * j + lq : 0;
    rs[j] = p.scale ? p.scale[n] : 1.0f;  // no per-row scale on fp16 weights
    bi[j] = p.bias ? p.bias[n] : 0.0f;
    gt[j] = RM && p.gate ? p.gate[p.gOff + n] : 1.0f;
  }
  constexpr bool LOAD_OLD = RM && !PRE_C;
  float old[2][LOAD_OLD ? 16 : 1];
  if constexpr (LOAD_OLD) load_old(p, old[0], mw, nw < p.N ? nw : 0, lq, hi);
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    pin(rs[j]);
    pin(bi[j]);
    if (RM) pin(gt[j]);
  }
  float* base = p.C + p.cOff + (long long)mw * p.ldc + nw;
  const long long lane_off = 4LL * hi * p.ldc + lq;
#pragma unroll
  for (int t = 0; t < TM * TN; ++t) {
    const int j = t / TM, i = t % TM;
    if constexpr (LOAD_OLD) {
      if (t + 1 < TM * TN) {
        const int j1 = (t + 1) / TM, i1 = (t + 1) % TM;
        const int mi = mw + 32 * i1 < p.M ? mw + 32 * i1 : mw, nj = nw + 32 * j1 < p.N ? nw + 32 * j1 : 0;
        load_old(p, old[(t + 1) & 1], mi, nj, lq, hi);
      }
    }
    if (nw + 32 * j >= p.N) continue;
    float16_t d;
    if constexpr (LORA) {
      const int m = mw + 32 * i + lq;
      d = lora_tile(p.lt, p.lb, p.lr, m < p.M ? m : p.M - 1, nw + 32 * j + lq, hi);
    }
    float v[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float x = acc[i][j][r] * p.alpha;
      x *= rs[j];
      x += bi[j];
      if constexpr (LORA) x += d[r];
      x = act_t<ACT>(x);
      if (RM) x = (PRE_C ? cold[PRE_C ? i : 0][PRE_C ? j : 0][r] : old[t & 1][LOAD_OLD ? r : 0]) + gt[j] * x;
      v[r] = x;
      if (LORA || RM) pin(v[r]);
    }
    if (full) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        (base + (long long)(32 * i + 8 * (r >> 2) + (r & 3)) * p.ldc + 32 * j)[lane_off] = v[r];
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int dm = 32 * i + 8 * (r >> 2) + (r & 3);
        if (mw + dm + 4 * hi < p.M) (base + (long long)dm * p.ldc + 32 * j)[lane_off] = v[r];
      }
    }
  }
}

// Plain store of one wave whose 32-column tiles lie in the packed-value window (RM 0): the
// values of the same epilogue, rounded to fp16 once, into the flash kernel's value layout. The
// 16 accumulator rows of a lane are keys {4hi..4hi+3, 8+4hi..8+4hi+3} of two 16-key groups,
// which the layout stores as one 16-byte chunk each (chunk 2g + hi of the group's 32 keys in
// a 64-key tile holds keys 16g + 4hi + {0..3} then 16g + 8 + 4hi + {0..3}).
template <int TM, int TN, int ACT, bool LORA>
__device__ __forceinline__ void store_vpack(const TGemmArgs& p, const float16_t (&acc)[TM][TN], int mw, int nw, int lq,
                                            int hi) {
  float rs[TN], bi[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = nw + 32 * j + lq;
    rs[j] = p.scale ? p.scale[n] : 1.0f;
    bi[j] = p.bias ? p.bias[n] : 0.0f;
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    pin(rs[j]);
    pin(bi[j]);
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = nw + 32 * j + lq;
    const int c = n - p.vcol0, h = c / p.vD, dd = c % p.vD;
    half_t* const dst0 = p.vpk + ((long long)h * p.vtiles * 64 * p.vD + (long long)dd * 8);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      float16_t d;
      if constexpr (LORA) {
        const int m = mw + 32 * i + lq;
        d = lora_tile(p.lt, p.lb, p.lr, m < p.M ? m : p.M - 1, n, hi);
      }
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float x = acc[i][j][8 * g + e] * p.alpha;
          x *= rs[j];
          x += bi[j];
          if constexpr (LORA) x += d[8 * g + e];
          v[e] = act_t<ACT>(x);
          // the fp32 value first, as the plain store writes it: the conversion must not fuse
          // with the multiply-add into one rounding to fp16 (v_fma_mix)
          pin(v[e]);
        }
        const int key16 = mw + 32 * i + 16 * g;
        if (key16 >= p.M) continue;
        const int kt = key16 >> 6, kc = 2 * ((key16 & 63) >> 4) + hi;
        uint4 q;
        q.x = pack_half2(v[0], v[1]);
        q.y = pack_half2(v[2], v[3]);
        q.z = pack_half2(v[4], v[5]);
        q.w = pack_half2(v[6], v[7]);
        *reinterpret_cast<uint4*>(dst0 + ((long long)kt * 8 + kc) * p.vD * 8) = q;
      }
    }
  }
}

// What a wave does with its sums (plain epilogues): the raw partial products of a split, the
// packed values of the attention, or store_plain.
template <int TM, int TN, int ACT, int RM, bool PRE_C, bool LORA, int CI, int CJ>
__device__ __forceinline__ void finish(const TGemmArgs& p, const float16_t (&acc)[TM][TN], const float (&cold)[CI][CJ][16],
                                       int mw, int nw, bool full, int lq, int hi) {
  if (p.part) {
    // split-K: the raw partial products of split blockIdx.y
    float* base = p.part + ((long long)blockIdx.y * p.M + mw) * p.N + nw;
    const long long lane_off = 4LL * hi * p.N + lq;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if (nw + 32 * j >= p.N) continue;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int dm = 32 * i + 8 * (r >> 2) + (r & 3);
          if (full || mw + dm + 4 * hi < p.M) (base + (long long)dm * p.N + 32 * j)[lane_off] = acc[i][j][r];
        }
    }
    return;
  }
  // a wave whose columns straddle vcol0 goes column tile by column tile
  if (RM == 0 && p.vpk && nw + 32 * TN > p.vcol0) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      float16_t col[TM][1];
#pragma unroll
      for (int i = 0; i < TM; ++i) col[i][0] = acc[i][j];
      const int n = nw + 32 * j;
      if (n >= p.N) continue;
      if (n >= p.vcol0) store_vpack<TM, 1, ACT, LORA>(p, col, mw, n, lq, hi);
      else store_plain<TM, 1, ACT, RM, false, LORA>(p, col, cold, mw, n, full, lq, hi);
    }
    return;
  }
  store_plain<TM, TN, ACT, RM, PRE_C, LORA>(p, acc, cold, mw, nw, full, lq, hi);
}

// Block tile BM x BN (multiples of 64), k-tiles of 64 KT. WAVES_M x WAVES_N waves per k group, each
// computing (BM/WAVES_M) x (BN/WAVES_N) with v_mfma_f32_32x32x16_f16 tiles; KG k groups of waves
// share a block's tile and take alternate k16 steps (their sums are added through LDS at the end),
// which puts two waves on every SIMD where the grid leaves one tile per CU. STAGES LDS stages.
//
// What bounds it: the matrix cores, at the clock the chip's power allows (1.5-1.75 GHz with all CUs
// multiplying), and what a wave issues beside its products. Of a whole launch's active cycles they are
// busy 43 % with the 192x384 tile (3952 x 4608 x 1536), 48 % with the GLU's 128x512 (3952 x 8192 x 1536),
// 41 % with 256x256 (2432 x 6144 x 1536), 35 and 32 % with 128x192 in one and two k groups and 30 % with
// 64x128 (SQ_VALU_MFMA_BUSY_CYCLES against GRBM_GUI_ACTIVE); the prologue (2 us) and the stores, when they
// idle, are in those cycles. Three things keep the k loop's products together:
//  * fragments are read one k16 step ahead, across the k-tile's barrier too: the barrier comes
//    before the last step of a tile (whose fragments are in registers by then), so no wave waits
//    for LDS behind it;
//  * the weight fragment of the next column is decoded behind the current column's products;
//  * the copies of a k-tile go out in SPREAD steps between products, since a wave that issues them
//    all at once issues no products meanwhile (64 bytes per clock and CU).
// A raised wave priority around the products measured no faster; a third stage pays where a tile has
// its CU to itself.
// EPI 0: C = act(A W^T * alpha * scale + bias) (RM 0) or C += (gate *) that (RM 1), the order of
// gemm.js:159-164. EPI 1 (GLU): W's rows are interleaved in 32-row blocks
// (ns2_tile_i8_weight_glu), so 64 columns of a wave hold 32 columns of each GLU half; the
// block's 512 columns give 256 consecutive outputs act(h1) * h2, one rotation group, which is
// rotated and written to Y as the tiled fp16 operand of the next int8 linear.
// OPS kF16: fp16 weight tiles (the plain bf16 linears, re-tiled as fp16; no per-row scale unless
// given): 8 KB per 64x64 weight tile, read straight into the MFMA B operand.
// OPS kI8Rows: nothing is re-tiled. A copy of 1 KB takes 8 rows x 128 bytes of A or 16 rows x 64 bytes of W
// (whole lines), and each lane fetches the 16-byte piece whose index is XORed with its row's (row % 8
// for A, row / 4 % 4 for W), so that the fragment reads of consecutive rows fall in different banks as
// those of the tiled layout do. The sums have the order of the tiled launch.
// WPE: waves per SIMD the registers must leave room for.
template <int BM, int BN, int WAVES_M, int WAVES_N, int KG, int KT, int STAGES, int SPREAD, int EPI, int ACT, int RM, bool LORA, Ops OPS, int WPE>
__global__ __launch_bounds__(WAVES_M * WAVES_N * KG * 64) __attribute__((amdgpu_waves_per_eu(WPE)))
void gemm_tiled_kernel(TGemmArgs p) {
  constexpr bool WF16 = OPS == kF16, ROWS = OPS == kI8Rows;
  constexpr int NW = WAVES_M * WAVES_N * KG;
  constexpr int WTM = BM / WAVES_M, WTN = BN / WAVES_N;
  constexpr int TM = WTM / 32, TN = WTN / 32;
  constexpr int NS = 4 * KT / KG;    // k16 steps of a k-tile (64 KT wide) per wave
  constexpr int WCH = WF16 ? 8 : 4;  // 1 KB blocks per 64 weight rows of a k-tile
  constexpr int WB = WF16 ? 2 : 1;   // bytes per weight element
  constexpr int A_BLOCKS = BM / 64 * 8 * KT, W_BLOCKS = BN / 64 * WCH * KT;  // 1 KB blocks per stage
  constexpr int BLOCKS = A_BLOCKS + W_BLOCKS;
  constexpr int PER_WAVE = BLOCKS / NW;  // copies per wave and k-tile
  constexpr int A_BYTES = BM * 64 * KT * 2, W_BYTES = BN * 64 * KT * WB;
  static_assert(BM % 64 == 0 && BN % 64 == 0 && WTM % 32 == 0 && WTN % 32 == 0, "tile shape");
  static_assert(BLOCKS % NW == 0, "copies must split evenly over the waves");
  static_assert(NS % 2 == 0, "an even number of steps per k-tile");
  static_assert(STAGES == 2 || (STAGES == 3 && SPREAD == 1), "two or three LDS stages");
  static_assert(OPS == kI8 || EPI == 0, "the GLU epilogue takes int8 weight tiles");
  __shared__ __attribute__((aligned(16))) char smem[STAGES * (A_BYTES + W_BYTES)];
  char* const as = smem;
  char* const ws = smem + STAGES * A_BYTES;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = KG > 1 ? wave / (WAVES_M * WAVES_N) : 0, wi = KG > 1 ? wave % (WAVES_M * WAVES_N) : wave;
  const int wm = wi / WAVES_N, wn = wi % WAVES_N;
  const int lq = lane & 31, hi = lane >> 5;

  int tm, tn;
  block_tile(p, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;

  // k-tiles of this block: all of K, or split z = blockIdx.y's range
  const int kt0 = p.part ? (int)blockIdx.y * p.ksplit : 0;
  const int kblocks = (p.part ? (p.K / 64 - kt0 < p.ksplit ? p.K / 64 - kt0 : p.ksplit) : p.K / 64) / KT;
  const int kall = p.K / 64;
  // Stage image: A blocks (8 k-chunks of 1 KB per 64-row block), then W blocks (WCH per 64-row
  // block). Block ids past the last real 64-row block re-read the last one (their rows are
  // dropped). The per-wave sources and destinations are fixed up front; a k-tile adds its offset.
  const char* g_src[PER_WAVE];
  uint32_t l_dst[PER_WAVE];
  int g_step[PER_WAVE], l_step[PER_WAVE];
  {
    const uint32_t as_base = lds_addr(as), ws_base = lds_addr(ws);
#pragma unroll
    for (int i = 0; i < PER_WAVE; ++i) {
      const int j = wave + i * NW;
      if (ROWS && j < A_BLOCKS) {
        // block (64 rows, k-tile, 8 rows); rows past M re-read the last one
        const int c = j % (8 * KT);
        const int mr = m0 + 64 * (j / (8 * KT)) + 8 * (c % 8) + (lane >> 3), m = mr < p.M ? mr : p.M - 1;
        g_src[i] = reinterpret_cast<const char*>(p.At + (long long)m * p.lda + 64 * (kt0 + c / 8)) +
                   ((lane & 7) ^ (lane >> 3)) * 16;
        l_dst[i] = as_base + j * 1024;
        g_step[i] = 128 * KT;
        l_step[i] = A_BYTES;
      } else if (ROWS) {
        // block (64 weight rows, k-tile, 16 rows)
        const int jw = j - A_BLOCKS, c = jw % (4 * KT);
        int nb = n0 / 64 + jw / (4 * KT);
        nb = nb < p.nblocks ? nb : p.nblocks - 1;
        g_src[i] = reinterpret_cast<const char*>(p.Wt) + (long long)(64 * nb + 16 * (c % 4) + (lane >> 2)) * p.K +
                   64 * (kt0 + c / 4) + ((lane & 3) ^ (lane >> 4)) * 16;
        l_dst[i] = ws_base + jw * 1024;
        g_step[i] = 64 * KT;
        l_step[i] = W_BYTES;
      } else if (j < A_BLOCKS) {
        const int mbi = j / (8 * KT), c = j % (8 * KT);
        int mb = m0 / 64 + mbi;
        mb = mb < p.mblocks ? mb : p.mblocks - 1;
        g_src[i] = reinterpret_cast<const char*>(p.At) + ((long long)mb * kall * 8 + (long long)kt0 * 8 + c) * 1024 + lane * 16;
        l_dst[i] = as_base + j * 1024;
        g_step[i] = 8 * KT * 1024;
        l_step[i] = A_BYTES;
      } else {
        const int jw = j - A_BLOCKS;
        const int nbi = jw / (WCH * KT), c = jw % (WCH * KT);
        int nb = n0 / 64 + nbi;
        nb = nb < p.nblocks ? nb : p.nblocks - 1;
        g_src[i] = reinterpret_cast<const char*>(p.Wt) + ((long long)nb * kall * WCH + (long long)kt0 * WCH + c) * 1024 + lane * 16;
        l_dst[i] = ws_base + jw * 1024;
        g_step[i] = WCH * KT * 1024;
        l_step[i] = W_BYTES;
      }
    }
  }
  auto dma_one = [&](int i, int kt, int st) {
    dma16(g_src[i] + (long long)kt * g_step[i], __builtin_amdgcn_readfirstlane(l_dst[i] + st * l_step[i]));
  };

  float16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  // Residual launches of small wave tiles load their old outputs before the k loop, where the
  // latency hides behind it, instead of in the epilogue.
  constexpr bool PRE_C = EPI == 0 && RM != 0 && KG == 1 && TM * TN * 16 <= 32;
  float cold[PRE_C ? TM : 1][PRE_C ? TN : 1][16];
  if constexpr (PRE_C) {
    if (!p.part) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int mi = m0 + wm * WTM + 32 * i, nj = n0 + wn * WTN + 32 * j;
          load_old(p, cold[i][j], mi < p.M ? mi : 0, nj < p.N ? nj : 0, lq, hi);
        }
    }
  }

  // fragments of k-step s (16 k) of a stage: A rows wm*WTM + 32i + lq, k 16s + 8hi .. +7 (chunk
  // 2s + hi); W columns wn*WTN + 32j + lq, the same k (8-byte chunk 2s + hi, or 16-byte chunk for
  // fp16 weights, read as the B operand itself)
  using WRaw = std::conditional_t<WF16, half8_t, uint2>;
  auto read_frags = [&](int st, int s, half8_t (&a)[TM], WRaw (&w)[TN]) {
    const int ks = s * KG + kg, kc = 2 * ks + hi;
    if constexpr (ROWS) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int col = wn * WTN + 32 * j;
        w[j] = *reinterpret_cast<const WRaw*>(ws + st * W_BYTES + (col / 64 * KT + ks / 4) * 4096 + (col % 64 + lq) * 64 +
                                              (((ks % 4) ^ (lq >> 2 & 3)) * 16 + hi * 8));
      }
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int row = wm * WTM + 32 * i;
        a[i] = *reinterpret_cast<const half8_t*>(as + st * A_BYTES + (row / 64 * KT + ks / 4) * 8192 + (row % 64 + lq) * 128 +
                                                 ((kc % 8) ^ (lq & 7)) * 16);
      }
      return;
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = wn * WTN + 32 * j;
      w[j] = *reinterpret_cast<const WRaw*>(ws + st * W_BYTES + ((col / 64 * 8 * KT + kc) * 64 + col % 64 + lq) * 8 * WB);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int row = wm * WTM + 32 * i;
      a[i] = *reinterpret_cast<const half8_t*>(as + st * A_BYTES + ((row / 64 * 8 * KT + kc) * 64 + row % 64 + lq) * 16);
    }
  };
  auto decode = [&](const WRaw& w) {
    if constexpr (WF16) return w;
    else if constexpr (ROWS) return u8x8_to_h8(make_uint2(w.x ^ 0x80808080u, w.y ^ 0x80808080u));
    else return u8x8_to_h8(w);
  };

  // The copies of a k-tile are issued in SPREAD steps, between the products: the first part in the
  // last step of tile kt, once every wave has read its last fragment of it (tile kt + STAGES takes
  // its stage), the rest in the first steps of tile kt + 1. copy_part issues those of slot `slot`.
  constexpr int SLOTS = SPREAD * TN;
  auto copy_part = [&](int slot, int kt, int st) {
#pragma unroll
    for (int i = 0; i < PER_WAVE; ++i)
      if (i * SLOTS / PER_WAVE == slot) dma_one(i, kt, st);
  };
#pragma unroll
  for (int t = 0; t < STAGES; ++t)
    if (t < kblocks) {
#pragma unroll
      for (int i = 0; i < PER_WAVE; ++i)
        if (t + 1 < STAGES || i * SLOTS / PER_WAVE < TN) dma_one(i, t, t);
    }
  // tile 0 has landed; the copies of later tiles may be in flight
  constexpr int FIRST = [] { int n = 0; for (int i = 0; i < PER_WAVE; ++i) n += i * SLOTS / PER_WAVE < TN; return n; }();
  if (kblocks >= STAGES) vm_wait<(STAGES - 2) * PER_WAVE + FIRST>();
  else vm_wait<0>();
  __syncthreads();
  half8_t a[2][TM];
  WRaw w[2][TN];
  read_frags(0, 0, a[0], w[0]);
  half8_t b = decode(w[0][0]);
  int st = 0;
  auto ktile = [&](int kt, auto last_c) {
    constexpr bool LAST = decltype(last_c)::value;
    const int nst = st + 1 == STAGES ? 0 : st + 1;
    const int pst = st == 0 ? STAGES - 1 : st - 1;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      if (s + 1 < NS) {
        read_frags(st, s + 1, a[(s + 1) & 1], w[(s + 1) & 1]);
      } else if (!LAST) {
        // this wave's copies of tile kt+1 have landed once at most the later tiles' remain in
        // flight; the barrier then covers every wave's copies, and every wave's reads of tile
        // kt (waited for here), whose stage the next copies overwrite
        if (STAGES == 3 && kt + 2 < kblocks) vm_wait<PER_WAVE>();
        else vm_wait<0>();
        __syncthreads();
        read_frags(nst, 0, a[0], w[0]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[s & 1][i], b, acc[i][j], 0, 0, 0);
        if (j + 1 < TN) b = decode(w[s & 1][j + 1]);
        else if (s + 1 < NS || !LAST) b = decode(w[(s + 1) & 1][0]);
        if (!LAST) {
          if (s == NS - 1) {
            if (kt + STAGES < kblocks) copy_part(j, kt + STAGES, st);
          } else if (s + 1 < SPREAD) {
            if (kt + STAGES - 1 < kblocks) copy_part((s + 1) * TN + j, kt + STAGES - 1, pst);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    st = nst;
  };
  for (int kt = 0; kt + 1 < kblocks; ++kt) ktile(kt, std::integral_constant<bool, false>{});
  ktile(kblocks - 1, std::integral_constant<bool, true>{});

  if constexpr (EPI == 1) {
    // ---- GLU + rotation epilogue (BN = 512: 256 outputs, one rotation group; a wave's columns are
    // pairs of 32 gate and 32 value columns), 64 rows at a time
    static_assert(KG == 1 && BN == 512 && TN % 2 == 0, "GLU epilogue tile");
    static_assert(sizeof(smem) >= 64 * 256 * 4, "one 64 x 256 fp32 chunk in the stages");
    constexpr int JP = TN / 2;
    const int I = p.N / 2;
    const int gb = n0 / 2;  // first output (GLU) column of the block
    float* T = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int ch = 0; ch < BM / 64; ++ch) {
      __syncthreads();  // every wave is done with the LDS stages (or the previous chunk)
#pragma unroll
      for (int jj = 0; jj < JP; ++jj) {
        const int gc = 32 * (wn * JP + jj) + lq;  // this lane's output column within the block
        const int G = gb + gc;
        const float s1 = p.scale[G], s2 = p.scale[I + G];
        const float b1 = p.bias ? p.bias[G] : 0.0f, b2 = p.bias ? p.bias[I + G] : 0.0f;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          if ((wm * WTM + 32 * i) / 64 != ch) continue;
          const int rb = (wm * WTM + 32 * i) % 64 + 4 * hi;
          if constexpr (LORA) {
            // the low-rank terms of the two halves' tiles (weight rows G and I + G), one tile at a
            // time: act(h1) goes through T, then h2 multiplies it in place
            int m = m0 + wm * WTM + 32 * i + lq;
            m = m < p.M ? m : p.M - 1;
            const float16_t d1 = lora_tile(p.lt, p.lb, p.lr, m, G, hi);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const int row = rb + 8 * (r >> 2) + (r & 3);
              float h1 = acc[i][2 * jj][r] * p.alpha;
              h1 *= s1;
              h1 += b1;
              T[row * 256 + gc] = glu_act<ACT>(h1 + d1[r]);
            }
            const float16_t d2 = lora_tile(p.lt, p.lb, p.lr, m, I + G, hi);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const int row = rb + 8 * (r >> 2) + (r & 3);
              float h2 = acc[i][2 * jj + 1][r] * p.alpha;
              h2 *= s2;
              h2 += b2;
              T[row * 256 + gc] *= h2 + d2[r];
            }
          } else {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const int row = rb + 8 * (r >> 2) + (r & 3);
              // the linear's epilogue order (no activation there), then the GLU
              float h1 = acc[i][2 * jj][r] * p.alpha;
              h1 *= s1;
              h1 += b1;
              float h2 = acc[i][2 * jj + 1][r] * p.alpha;
              h2 *= s2;
              h2 += b2;
              T[row * 256 + gc] = glu_act<ACT>(h1) * h2;
            }
          }
        }
      }
      __syncthreads();
      // rotation: wave w rotates its 64 / NW rows on the matrix cores, the fp16 result in place in
      // the first 512 bytes of the row, its 16-byte chunk c stored at chunk c ^ (row & 7): the
      // copy-out below reads one chunk of 64 rows 1 KB apart per wave, and the swizzle puts 8
      // consecutive rows in 8 different bank groups (unswizzled, all 64 lanes hit the same four
      // banks)
#pragma unroll
      for (int rr = 0; rr < 64 / NW; ++rr) {
        // the matrix-core FWHT: lane l holds columns lo .. lo+3, lo = 16(l%16) + 4(l/16)
        const half4v_t hf = fwht_h16_fragment();
        const int lo = fwht_mfma_offset();
        const int row = (64 / NW) * wave + rr;
        const float4 in = *reinterpret_cast<const float4*>(T + row * 256 + lo);
        float v[4] = {in.x, in.y, in.z, in.w};
        fwht256_mfma(v, hf);
        uint2 o;
        o.x = pack_half2(v[0], v[1]);
        o.y = pack_half2(v[2], v[3]);
        char* rb = reinterpret_cast<char*>(T + row * 256);
        *reinterpret_cast<uint2*>(rb + ((lo >> 3) ^ (row & 7)) * 16 + ((lo >> 2) & 1) * 8) = o;
      }
      __syncthreads();
      // 32 chunks of 8 columns x 64 rows: 1 KB contiguous each in the tiled layout; the row blocks
      // past the last one of Y (BM > 64) are dropped
      if (BM > 64 && m0 + 64 * ch >= p.mblocks * 64) break;
      for (int q = tid; q < 32 * 64; q += NW * 64) {
        const int row = q % 64, c = q / 64;
        const char* rb = reinterpret_cast<const char*>(T + row * 256);
        const uint4 v = *reinterpret_cast<const uint4*>(rb + (c ^ (row & 7)) * 16);
        *reinterpret_cast<uint4*>(p.Y + tiled_off(m0 + 64 * ch + row, gb + c * 8, I)) = v;
      }
    }
    return;
  }
  if constexpr (KG == 1) {
    finish<TM, TN, ACT, RM, PRE_C, LORA>(p, acc, cold, m0 + wm * WTM, n0 + wn * WTN, m0 + BM <= p.M, lq, hi);
  } else {
    // the two k groups' sums: group g keeps row tiles [g TM/2, (g+1) TM/2) and hands the others
    // over through LDS, one column tile at a time (16 values per lane as four float4 planes)
    static_assert(KG == 2 && TM % 2 == 0, "row tiles split between two k groups");
    constexpr int H = TM / 2;
    static_assert(sizeof(smem) >= (size_t)NW * H * 4096, "exchange buffer");
    constexpr bool PRE = RM && H * TN * 16 <= 48;
    float kold[PRE ? H : 1][PRE ? TN : 1][16];
    if constexpr (PRE) {
      // the kept tiles' old outputs, in flight behind the exchange
      if (!p.part) {
#pragma unroll
        for (int i = 0; i < H; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            const int mi = m0 + wm * WTM + (kg * H + i) * 32, nj = n0 + wn * WTN + 32 * j;
            load_old(p, kold[i][j], mi < p.M ? mi : 0, nj < p.N ? nj : 0, lq, hi);
          }
      }
    }
    float16_t keep[H][TN];
    float4* X = reinterpret_cast<float4*>(smem);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      __syncthreads();
#pragma unroll
      for (int i = 0; i < H; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float16_t& g = kg ? acc[i][j] : acc[H + i][j];
          X[((wave * H + i) * 4 + q) * 64 + lane] = make_float4(g[4 * q], g[4 * q + 1], g[4 * q + 2], g[4 * q + 3]);
        }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < H; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float4 o = X[(((wave ^ (NW / 2)) * H + i) * 4 + q) * 64 + lane];
          const float16_t& k = kg ? acc[H + i][j] : acc[i][j];
          keep[i][j][4 * q + 0] = k[4 * q + 0] + o.x;
          keep[i][j][4 * q + 1] = k[4 * q + 1] + o.y;
          keep[i][j][4 * q + 2] = k[4 * q + 2] + o.z;
          keep[i][j][4 * q + 3] = k[4 * q + 3] + o.w;
        }
    }
    finish<H, TN, ACT, RM, PRE, LORA>(p, keep, kold, m0 + wm * WTM + kg * H * 32, n0 + wn * WTN,
                                        m0 + BM <= p.M, lq, hi);
  }
}

// Adds the splits of a split-K launch in z order and applies the plain epilogue.
int launch_splitk_reduce(const TGemmArgs& p, int splits);

// Weight bytes per column band of the tile order: half of an XCD's 4 MB L2.
constexpr long long kBandBytes = 2ll << 20;

// What a block tile has kernels for, beside plain launches: old outputs (C +=), the LoRA term, both, and the
// activations (one kernel each) of those.
enum Forms : unsigned { kPlain = 0, kResid = 1, kLora = 2, kResidLora = 4, kAct = 8 };

template <int BM, int BN, int WM, int WN, int KG, int KT, int STAGES, int SPREAD, int WPE, Ops OPS, unsigned FORMS, int EPI = 0>
int launch_tiled(TGemmArgs p, int splits = 1, bool reduce = true) {
  p.tiles_m = (p.M + BM - 1) / BM;
  p.tiles_n = (p.N + BN - 1) / BN;
  // column bands (1, 2, 4 or 8) by an estimate of the bytes the XCDs' L2s miss: with b bands
  // each of the 8 XCDs reads its rows of A (A b / 8 in all) and a 1/b slice of W, re-read about
  // twice when the slice exceeds kBandBytes and three times when it exceeds an L2 (the factors
  // fit FETCH_SIZE at the DiT shapes: 3952 rows x {4608, 1536, 8192} x {1536, 4096}). Launches
  // with a few row tiles read each weight tile about once whatever the order.
  p.bands = 1;
  if (p.tiles_m >= 8) {
    const double a_bytes = (double)p.tiles_m * BM * p.K * 2, w_bytes = (double)p.N * p.K * (OPS == kF16 ? 2 : 1);
    double best = 0;
    for (int b = 1; b <= 8 && b <= p.tiles_n; b *= 2) {
      const double slice = w_bytes / b;
      const double f = slice <= kBandBytes ? 1.0 : (slice <= 2 * kBandBytes ? 2.0 : 3.0);
      const double est = a_bytes * b + w_bytes * (8.0 / b) * f;
      if (b == 1 || est < best) {
        best = est;
        p.bands = b;
      }
    }
  }
  const dim3 grid(p.tiles_m * p.tiles_n, splits), block(WM * WN * KG * 64);
  hipStream_t s = ns2::stream();
  using std::integral_constant;
  // a form without a kernel is not picked (linear_tiled)
  bool ran = false;
  auto run = [&](auto act_c, auto rm_c) {
    constexpr int A = decltype(act_c)::value, R = decltype(rm_c)::value;
    if constexpr ((FORMS & (R ? kResidLora : kLora)) != 0) {
      if (p.lr) {
        gemm_tiled_kernel<BM, BN, WM, WN, KG, KT, STAGES, SPREAD, EPI, A, R, true, OPS, WPE><<<grid, block, 0, s>>>(p);
        ran = true;
      }
    }
    if constexpr (!R || (FORMS & kResid)) {
      if (!p.lr) {
        gemm_tiled_kernel<BM, BN, WM, WN, KG, KT, STAGES, SPREAD, EPI, A, R, false, OPS, WPE><<<grid, block, 0, s>>>(p);
        ran = true;
      }
    }
  };
  auto run_act = [&](auto act_c) {
    if constexpr (EPI == 0 && (FORMS & kResid)) {
      if (p.resid) return run(act_c, integral_constant<int, 1>{});
    }
    if (!p.resid) run(act_c, integral_constant<int, 0>{});
  };
  if (p.act == NS2_ACT_NONE) {
    run_act(integral_constant<int, NS2_ACT_NONE>{});
  } else if constexpr (EPI == 1 || (FORMS & kAct)) {
    if (p.act == NS2_ACT_SILU) run_act(integral_constant<int, NS2_ACT_SILU>{});
    else run_act(integral_constant<int, NS2_ACT_GELU_TANH>{});
  }
  if (!ran) return ns2::set_error(NS2_ERR_INVALID, "gemm_tiled: a block tile without a kernel for the call");
  NS2_LAUNCHED("gemm_tiled");
  if (p.part && reduce) return launch_splitk_reduce(p, splits);
  return NS2_OK;
}

// The block tiles of the plain launches (ns2_gemm_tiled.hip has their time model), and the launch of tile t:
// one instantiation per operand kind, each compiled in a file of its own.
enum Tile { T64x64, T64x128K2, T64x128K2S3, T64x128, T128x128, T128x192, T128x192K2, T192x384, T256x256, kTiles };

// The forms of each tile. Each activation has its own kernels, although none of the models' tiled linears
// has one: chosen at run time it cost small launches 2 us (33 x 64 x 1536 with SiLU: 7.2 -> 9.3) and spilled on the
// largest tiles. 192x384 gains over the other tiles by 4 % at most with old outputs or a LoRA,
// so it is plain only; 128x128 has no registers for old outputs beside the LoRA term at three blocks
// per CU; fp16 weights have the six tiles that any launch gains from.
constexpr unsigned kNotBuilt = ~0u;
template <Ops OPS>
constexpr unsigned tile_forms(Tile t) {
  if (OPS == kF16 && (t == T64x128K2 || t == T128x192K2 || t == T192x384)) return kNotBuilt;
  return t == T192x384 ? kPlain : t == T128x128 ? kResid | kLora | kAct : kResid | kLora | kResidLora | kAct;
}

// The tiles with a kernel for the call, bit t for tile t.
template <Ops OPS>
inline unsigned allowed_tiles(int act, int resid, int lora_r) {
  unsigned m = 0;
  for (int t = 0; t < kTiles; ++t) {
    const unsigned f = tile_forms<OPS>((Tile)t);
    if (f == kNotBuilt) continue;
    const unsigned need = (act != NS2_ACT_NONE ? kAct : 0u) | (resid ? kResid : 0u) | (lora_r ? kLora : 0u) |
                          (resid && lora_r ? kResidLora : 0u);
    if ((f & need) == need) m |= 1u << t;
  }
  return m;
}

template <Ops OPS>
int launch_tile(Tile t, const TGemmArgs& p, int splits) {
  if constexpr (OPS == kF16) {
    switch (t) {
      case T64x64: return launch_tiled<64, 64, 1, 2, 2, 1, 3, 1, 2, OPS, tile_forms<OPS>(T64x64)>(p, splits);
      case T64x128K2S3: return launch_tiled<64, 128, 1, 4, 2, 1, 3, 1, 2, OPS, tile_forms<OPS>(T64x128K2S3)>(p);
      case T64x128: return launch_tiled<64, 128, 1, 4, 1, 1, 2, 1, 3, OPS, tile_forms<OPS>(T64x128)>(p);
      case T128x128: return launch_tiled<128, 128, 2, 2, 1, 1, 2, 1, 2, OPS, tile_forms<OPS>(T128x128)>(p);
      case T128x192: return launch_tiled<128, 192, 2, 2, 1, 1, 2, 2, 2, OPS, tile_forms<OPS>(T128x192)>(p);
      default: return launch_tiled<256, 256, 2, 4, 1, 1, 2, 2, 2, OPS, tile_forms<OPS>(T256x256)>(p);
    }
  } else {
    switch (t) {
      case T64x64: return launch_tiled<64, 64, 1, 2, 2, 2, 3, 1, 2, OPS, tile_forms<OPS>(T64x64)>(p, splits);
      case T64x128K2: return launch_tiled<64, 128, 1, 4, 2, 2, 2, 1, 4, OPS, tile_forms<OPS>(T64x128K2)>(p);
      case T64x128K2S3: return launch_tiled<64, 128, 1, 4, 2, 2, 3, 1, 2, OPS, tile_forms<OPS>(T64x128K2S3)>(p);
      case T64x128: return launch_tiled<64, 128, 1, 4, 1, 1, 2, 1, 4, OPS, tile_forms<OPS>(T64x128)>(p);
      case T128x128: return launch_tiled<128, 128, 2, 2, 1, 1, 2, 1, 3, OPS, tile_forms<OPS>(T128x128)>(p);
      case T128x192: return launch_tiled<128, 192, 2, 2, 1, 1, 2, 2, 2, OPS, tile_forms<OPS>(T128x192)>(p);
      case T128x192K2: return launch_tiled<128, 192, 2, 2, 2, 2, 2, 2, 2, OPS, tile_forms<OPS>(T128x192K2)>(p);
      case T192x384: return launch_tiled<192, 384, 2, 4, 1, 1, 2, 2, 2, OPS, tile_forms<OPS>(T192x384)>(p);
      default: return launch_tiled<256, 256, 2, 4, 1, 1, 2, 2, 2, OPS, tile_forms<OPS>(T256x256)>(p);
    }
  }
}

extern template int launch_tile<kI8>(Tile, const TGemmArgs&, int);
extern template int launch_tile<kF16>(Tile, const TGemmArgs&, int);
extern template int launch_tile<kI8Rows>(Tile, const TGemmArgs&, int);

}  // namespace ns2tiled
