// The tiled linears' entry points, the choice of the block tile, the split-K reduce and the weight re-tiling.
// The kernel is in ns2_gemm_tiled.h; ns2_gemm_tiled_i8.hip, _f16.hip and _rows.hip compile it per operand kind.
#include "ns2_gemm_tiled.h"

using namespace ns2dev;
using namespace ns2tiled;

namespace {

// The splits of a split-K launch summed in z order (deterministic), then the plain epilogue of
// store_plain (scale, bias, activation, store / += / += gate times).
__global__ __launch_bounds__(256) void tiled_splitk_reduce_kernel(TGemmArgs p, int splits) {
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long mn = (long long)p.M * p.N;
  if (idx >= mn) return;
  float acc = 0.f;
  for (int z = 0; z < splits; ++z) acc += p.part[z * mn + idx];
  const int m = (int)(idx / p.N), n = (int)(idx % p.N);
  float v = acc * p.alpha;
  if (p.scale) v *= p.scale[n];
  v += p.bias ? p.bias[n] : 0.0f;
  if (p.act == NS2_ACT_SILU) v = silu(v);
  else if (p.act == NS2_ACT_GELU_TANH) v = gelu_tanh(v);
  float* c = p.C + p.cOff + (long long)m * p.ldc + n;
  if (!p.resid) *c = v;
  else if (!p.gate) *c = *c + v;
  else *c = *c + p.gate[p.gOff + n] * v;
}

// W [N, K] row-major int8 -> Wt tiles [N/64][K/64][8 k-chunks of 8][64 rows][8 bytes] of biased
// bytes (w + 128); one thread per 8-byte chunk.
__global__ __launch_bounds__(256) void tile_w_kernel(const int8_t* __restrict__ W, uint8_t* __restrict__ Wt,
                                                      int N, int K, int glu) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;  // output chunk index
  const long long chunks = (long long)N * K / 8;
  if (i >= chunks) return;
  // chunk order: [nb][kb][c 0..7][row 0..63]
  const int row = (int)(i % 64);
  const int c = (int)((i / 64) % 8);
  const long long rest = i / 512;  // nb * (K/64) + kb
  const int kb = (int)(rest % (K / 64));
  const int nb = (int)(rest / (K / 64));
  int n = nb * 64 + row;
  // GLU interleave: tiled row 64q + t holds row 32q + t of the first half (t < 32) or row
  // N/2 + 32q + t - 32 of the second half
  if (glu) n = row < 32 ? 32 * nb + row : N / 2 + 32 * nb + row - 32;
  uint2 v = *reinterpret_cast<const uint2*>(W + (long long)n * K + kb * 64 + c * 8);
  v.x ^= 0x80808080u;
  v.y ^= 0x80808080u;
  *reinterpret_cast<uint2*>(Wt + i * 8) = v;
}

// W [N, K] row-major bf16 -> Wt tiles [N/64][K/64][8 k-chunks of 8][64 rows][8 halfs] of fp16
// (round to nearest even, as the row-major kernel's loader converts them); one thread per
// 16-byte chunk.
__global__ __launch_bounds__(256) void tile_w16_kernel(const uint16_t* __restrict__ W, uint16_t* __restrict__ Wt,
                                                        int N, int K) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;  // output chunk index
  const long long chunks = (long long)N * K / 8;
  if (i >= chunks) return;
  const int row = (int)(i % 64);
  const int c = (int)((i / 64) % 8);
  const long long rest = i / 512;  // nb * (K/64) + kb
  const int kb = (int)(rest % (K / 64));
  const int nb = (int)(rest / (K / 64));
  const uint4 v = *reinterpret_cast<const uint4*>(W + (long long)(nb * 64 + row) * K + kb * 64 + c * 8);
  const uint32_t in[4] = {v.x, v.y, v.z, v.w};
  uint32_t out[4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    out[j] = pack_half2(__builtin_bit_cast(float, in[j] << 16), __builtin_bit_cast(float, in[j] & 0xffff0000u));
  *reinterpret_cast<uint4*>(Wt + i * 8) = make_uint4(out[0], out[1], out[2], out[3]);
}

}  // namespace

int ns2tiled::launch_splitk_reduce(const TGemmArgs& p, int splits) {
  const long long mn = (long long)p.M * p.N;
  tiled_splitk_reduce_kernel<<<(unsigned)((mn + 255) / 256), 256, 0, ns2::stream()>>>(p, splits);
  NS2_LAUNCHED("gemm_tiled_splitk_reduce");
  return NS2_OK;
}

namespace {

// Block tiles and their time model: a launch gives every CU `per` = ceil(tiles / 256) tiles, run as
// rounds of up to `occ` co-resident blocks; a round of n blocks per CU takes e[n-1] + c[n-1] us per
// 64-wide k-tile, and a launch L us more. These are weights for ranking the tiles against each other, not
// times: int8 rows were fitted to launches of 64-3952 rows x 1536-27648 x 1536-6144 with weights cycled through 8
// copies (three stages: through 600 MB), fp16 rows to the tiles near the best of 396 launches of 33-8192 rows x
// 64-16384 x 64-4096 (16 copies); two per CU of int8 128x192, fp16 128x192 and three per CU of fp16 64x64 were
// raised by hand where they were picked too early. They know only the busiest CU and no clock, which
// falls from 2.3 to 1.5 GHz as CUs fill up: one large tile per CU is put up to 26 % too low (3952 x 4608 x 1536:
// 42.6 for 57.5 us; 3328: 39.9 for 49.6), fewer or smaller tiles within about 10 %. What counts is the pick: over 1254
// measured launches of every tile (33-8192 rows, 19 shapes N x K; plain, C += and with a LoRA) it is 0.9 % off the
// best on average and 60 % at most (8192 x 1024 x 256).
//   64x64, 4 waves (2 k groups)   few tiles: each block's k chain halved, three 128-wide stages
//   64x128, 8 waves (2 k groups)  two tiles per CU (1900 x 1536 x 1536 +=: 17.9 us)
//   the same, three stages        one tile per CU: with the block alone on its CU, one k-tile ahead does not
//                                 cover a weight's way from memory (weights cycled through 600 MB, two ->
//                                 three stages: 1024 x 1536 x 1536 +=: 14.3 -> 11.8 us, x 4096 29.8 -> 22.5, x 6144
//                                 42.1 -> 32.4, 250 x 4608 x 1536 13.6 -> 11.3; six stages of the 64x64 tile
//                                 or five of 128x192 gained nothing more)
//   64x128, 4 waves               3 or 4 tiles per CU
//   128x128, 4 waves              3 tiles per CU (1792 x 4608 x 1536: 35.4 -> 30.1 us)
//   128x192, 4 waves              2 tiles per CU (2432 x 4608 x 1536: 47.2 -> 39.1 us)
//   128x192, 8 waves (2 k groups) one tile per CU, long K (3952 x 1536 x 4096 +=: 62.2 -> 54.7 us)
//   192x384, 8 waves              one tile per CU (3952 x 4608 x 1536: 70.3 -> 57.5 us)
//   256x256, 8 waves              one tile per CU (3328 x 4608 x 1536: 51.9 -> 49.6 us)
struct TileCfg {
  const char* name;
  int bm, bn, occ;
  float L, e[4], c[4];
};
constexpr TileCfg kCfgs[kTiles] = {
    {"64x64", 64, 64, 2, 1.8f, {1.86f, 2.65f}, {0.210f, 0.322f}},
    {"64x128K2", 64, 128, 2, 1.5f, {2.56f, 4.34f}, {0.398f, 0.474f}},
    {"64x128K2S3", 64, 128, 1, 1.5f, {3.20f}, {0.263f}},
    {"64x128", 64, 128, 4, 3.8f, {0.f, 1.49f, 3.17f, 0.f}, {0.413f, 0.510f, 0.731f, 1.147f}},
    {"128x128", 128, 128, 3, 2.9f, {2.49f, 5.20f, 0.f}, {0.513f, 0.790f, 1.550f}},
    {"128x192", 128, 192, 2, 0.9f, {5.77f, 5.00f}, {0.696f, 1.289f}},
    {"128x192K2", 128, 192, 1, 0.f, {8.83f}, {0.520f}},
    {"192x384", 192, 384, 1, 0.f, {13.86f}, {1.199f}},
    {"256x256", 256, 256, 1, 0.f, {12.80f}, {1.130f}},
};
constexpr TileCfg kCfgsF16[kTiles] = {
    {"64x64", 64, 64, 3, 2.88f, {0.61f, 1.42f, 2.88f}, {0.245f, 0.384f, 0.520f}},
    {},
    {"64x128K2S3", 64, 128, 1, 2.63f, {1.68f}, {0.314f}},
    {"64x128", 64, 128, 3, 3.33f, {0.55f, 1.94f, 3.85f}, {0.504f, 0.653f, 0.894f}},
    {"128x128", 128, 128, 2, 1.05f, {4.13f, 6.69f}, {0.644f, 0.949f}},
    {"128x192", 128, 192, 2, 1.44f, {5.86f, 10.11f}, {0.920f, 1.205f}},
    {},
    {},
    {"256x256", 256, 256, 1, 0.f, {12.05f}, {1.605f}},
};
constexpr int kCUs = 256;

// The reduce launch of a split-K linear and its traffic (33 x 64 x 1536 in 3: 2.0 us, 33 x 1536 x 1536 in 3: 2.9, 120 x 1536 x 6144
// in 3: 3.8, 256 x 1536 x 4096 in 2: 4.5).
float reduce_time(int M, int N, int splits) { return 2.0f + 3e-6f * (float)M * (float)N * (float)splits; }

// Modelled time of `tiles` block tiles of configuration t over kt k-tiles each.
float tile_time(const TileCfg& t, long long tiles, int kt) {
  const long long per = (tiles + kCUs - 1) / kCUs, full = per / t.occ;
  const int rem = (int)(per % t.occ);
  float us = t.L + full * (t.e[t.occ - 1] + kt * t.c[t.occ - 1]);
  if (rem) us += t.e[rem - 1] + kt * t.c[rem - 1];
  return us;
}

long long tile_count(const TileCfg& t, int M, int N) {
  return (long long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
}

// The tile of the least modelled time, and for 64x64 tiles how many ways K is split (over
// blockIdx.y, reduced in a second launch; at least 8 k-tiles per split). `allowed`: bit t for tile t. Only a
// grid of up to kSplitTiles is split, over at least 16 k-tiles: the launches that take the scratch for it.
constexpr long long kSplitTiles = 213;
Tile pick_tile(const TileCfg* cfgs, int M, int N, int K, unsigned allowed, bool can_split, int* splits) {
  const int kt = K / 64;
  Tile best = T64x64;
  float best_us = 0;
  *splits = 0;
  for (int i = 0; i < kTiles; ++i) {
    if (!(allowed >> i & 1)) continue;
    const long long tiles = tile_count(cfgs[i], M, N);
    const int most = i == T64x64 && can_split && tiles <= kSplitTiles ? (kt / 8 < 8 ? kt / 8 : 8) : 1;
    for (int s = 1; s <= (most > 1 ? most : 1); ++s) {
      const float us = tile_time(cfgs[i], tiles * s, (kt + s - 1) / s) + (s > 1 ? reduce_time(M, N, s) : 0.f);
      if (!*splits || us < best_us) {
        best = (Tile)i;
        best_us = us;
        *splits = s;
      }
    }
  }
  return best;
}

// The block tile of a linear, and its K splits: whole 128-wide stages of int8 tiles; none with a LoRA,
// whose term the reduce would have to add (256 x 1536 x 4096, rank 32: 51.5 us split, 27.6 unsplit), none where the
// values are packed, none for row-major operands, which use no scratch.
Tile plan_tile(Ops ops, int M, int N, int K, int act, int resid, int lora_r, bool packed, int* splits, int* ksplit) {
  const unsigned allowed = ops == kF16 ? allowed_tiles<kF16>(act, resid, lora_r) : allowed_tiles<kI8>(act, resid, lora_r);
  const Tile t = pick_tile(ops == kF16 ? kCfgsF16 : kCfgs, M, N, K, allowed, ops != kI8Rows && !packed && !lora_r, splits);
  *ksplit = 0;
  if (*splits > 1) {
    const int kt = K / 64;
    *ksplit = (kt + *splits - 1) / *splits;
    if (ops != kF16) *ksplit += *ksplit & 1;
    *splits = (kt + *ksplit - 1) / *ksplit;
  }
  return t;
}

inline bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// ops kF16: Wt holds fp16 weight tiles (ns2_tile_bf16_weight) and scale may be null; otherwise int8 ConvRot
// weights with their per-row scales (K a whole number of rotation groups). lda: row stride of kI8Rows.
int linear_tiled(const char* fn, Ops ops, const uint16_t* At, int lda, const void* Wt, const float* scale, const float* bias,
                 float* C, int M, int N, int K, int ldc, long long cOff, float alpha, int act, int resid,
                 const float* gate, long long gOff, const uint16_t* lora_a, const uint16_t* lora_b, int lora_r,
                 uint16_t* vpk = nullptr, int vcol0 = 0, int vD = 0, int vtiles = 0) {
  NS2_READY();
  if (M == 0) return NS2_OK;
  NS2_REQUIRE(At && Wt && (scale || ops == kF16) && C, "%s: null At, Wt, scale or C", fn);
  const int kmul = ops == kF16 ? 64 : 256;
  NS2_REQUIRE(M > 0 && N > 0 && N % 64 == 0 && K > 0 && K % kmul == 0,
              "%s: M=%d N=%d K=%d (N %% 64 == 0, K %% %d == 0 required)", fn, M, N, K, kmul);
  NS2_REQUIRE(ldc >= N && cOff >= 0 && gOff >= 0, "%s: bad ldc/offsets", fn);
  NS2_REQUIRE(aligned16(At) && aligned16(Wt), "%s: operands must be 16-byte aligned", fn);
  NS2_REQUIRE(act >= NS2_ACT_NONE && act <= NS2_ACT_GELU_TANH, "%s: unknown act %d", fn, act);
  TGemmArgs p{reinterpret_cast<const half_t*>(At), static_cast<const uint8_t*>(Wt), scale, bias, C, nullptr, gate,
              cOff, gOff, M, N, K, ldc, (M + 63) / 64, N / 64, 0, 0, alpha, act, resid};
  p.vpk = reinterpret_cast<half_t*>(vpk);
  p.vcol0 = vcol0;
  p.vD = vD;
  p.vtiles = vtiles;
  p.lda = lda;
  if (lora_r) {
    int rc = ns2::lora_prepare(&p.lt, lora_a, lora_b, lora_r, At, ops == kI8Rows ? 1 : 2, ops == kI8Rows ? lda : K, M, K, fn);
    if (rc) return rc;
    p.lb = reinterpret_cast<const half_t*>(lora_b);
    p.lr = lora_r;
  }
  ns2::ProfScope prof_(ops == kF16 ? "gemm_f16_tiled" : ops == kI8 ? "gemm_i8_tiled" : "linear_i8");
  int splits;
  const Tile tile = plan_tile(ops, M, N, K, act, resid, lora_r, vpk != nullptr, &splits, &p.ksplit);
  if (splits > 1) {
    p.part = static_cast<float*>(ns2::workspace(5, (size_t)splits * M * N * sizeof(float)));
    if (!p.part) return ns2::set_error(NS2_ERR_OOM, "%s: split-K workspace allocation failed", fn);
  }
  if (ops == kF16) return launch_tile<kF16>(tile, p, splits);
  return ops == kI8 ? launch_tile<kI8>(tile, p, splits) : launch_tile<kI8Rows>(tile, p, 1);
}

}  // namespace

int ns2::linear_i8_rows(const uint16_t* x, int ldx, const int8_t* W, const float* scale, const float* bias, float* C, int M,
                        int N, int K, int ldc, long long cOff, float alpha, int act, int resid, const float* gate,
                        long long gOff, const uint16_t* lora_a, const uint16_t* lora_b, int lora_r) {
  return linear_tiled("ns2_linear_i8", kI8Rows, x, ldx, W, scale, bias, C, M, N, K, ldc, cOff, alpha, act, resid, gate, gOff,
                      lora_a, lora_b, lora_r);
}

int ns2::linear_f16w_tiled_raw(const char* fn, const uint16_t* At, const uint16_t* Wt, int M, int N, int K,
                               float** part, int* splits) {
  NS2_REQUIRE(At && Wt && M > 0 && N > 0 && N % 64 == 0 && K > 0 && K % 64 == 0 && aligned16(At) && aligned16(Wt),
              "%s: At, Wt, M=%d, N=%d (N %% 64 == 0), K=%d (K %% 64 == 0) or alignment", fn, M, N, K);
  TGemmArgs p{reinterpret_cast<const half_t*>(At), reinterpret_cast<const uint8_t*>(Wt), nullptr, nullptr, nullptr,
              nullptr, nullptr, 0, 0, M, N, K, N, (M + 63) / 64, N / 64, 0, 0, 1.0f, NS2_ACT_NONE, 0};
  // 64x64 tiles (the few-row launches this serves); K split until about one block per CU, at
  // least 4 k-tiles per split
  const long long tiles = (long long)((M + 63) / 64) * (N / 64);
  const int kt = K / 64;
  int s = (int)(kCUs / tiles);
  if (s > kt / 4) s = kt / 4;
  if (s > 8) s = 8;
  if (s < 1) s = 1;
  p.ksplit = (kt + s - 1) / s;
  s = (kt + p.ksplit - 1) / p.ksplit;
  p.part = static_cast<float*>(ns2::workspace(5, (size_t)s * M * N * sizeof(float)));
  if (!p.part) return ns2::set_error(NS2_ERR_OOM, "%s: split-K workspace allocation failed", fn);
  *part = p.part;
  *splits = s;
  ns2::ProfScope prof_("gemm_f16_tiled");
  return launch_tiled<64, 64, 2, 2, 1, 1, 3, 1, 2, kF16, kPlain>(p, s, false);
}

extern "C" {

// For tests, not part of the C ABI: the block tile and the K splits that a linear would be launched with
// (ops: 0 int8 tiles, 1 fp16 tiles, 2 row-major operands). Host only.
const char* ns2_internal_tile(int ops, int M, int N, int K, int act, int resid, int lora_r, int packed, int* splits) {
  int ksplit;
  const Tile t = plan_tile((Ops)ops, M, N, K, act, resid, lora_r, packed, splits, &ksplit);
  return kCfgs[t].name;
}

int ns2_tile_i8_weight(const int8_t* W, int8_t* Wt, int N, int K) {
  NS2_READY();
  NS2_REQUIRE(W && Wt && aligned16(W) && aligned16(Wt), "ns2_tile_i8_weight: null or unaligned buffer");
  NS2_REQUIRE(N > 0 && K > 0 && N % 64 == 0 && K % 64 == 0,
              "ns2_tile_i8_weight: N=%d and K=%d must be multiples of 64", N, K);
  const long long chunks = (long long)N * K / 8;
  ns2::ProfScope prof_("tile_i8_weight");
  tile_w_kernel<<<(unsigned)((chunks + 255) / 256), 256, 0, ns2::stream()>>>(W, reinterpret_cast<uint8_t*>(Wt), N, K, 0);
  NS2_LAUNCHED("tile_i8_weight");
  return NS2_OK;
}

int ns2_tile_i8_weight_glu(const int8_t* W, int8_t* Wt, int N, int K) {
  NS2_READY();
  NS2_REQUIRE(W && Wt && aligned16(W) && aligned16(Wt), "ns2_tile_i8_weight_glu: null or unaligned buffer");
  NS2_REQUIRE(N > 0 && K > 0 && N % 64 == 0 && K % 64 == 0,
              "ns2_tile_i8_weight_glu: N=%d and K=%d must be multiples of 64", N, K);
  const long long chunks = (long long)N * K / 8;
  ns2::ProfScope prof_("tile_i8_weight");
  tile_w_kernel<<<(unsigned)((chunks + 255) / 256), 256, 0, ns2::stream()>>>(W, reinterpret_cast<uint8_t*>(Wt), N, K, 1);
  NS2_LAUNCHED("tile_i8_weight_glu");
  return NS2_OK;
}

int ns2_linear_i8_glu_rot_tiled(const uint16_t* At, const int8_t* Wt, const float* scale, const float* bias,
                                uint16_t* Y, int M, int N, int K, float alpha, int act) {
  return ns2_linear_i8_glu_rot_tiled_lora(At, Wt, scale, bias, Y, M, N, K, alpha, act, nullptr, nullptr, 0);
}

int ns2_linear_i8_glu_rot_tiled_lora(const uint16_t* At, const int8_t* Wt, const float* scale, const float* bias,
                                     uint16_t* Y, int M, int N, int K, float alpha, int act, const uint16_t* lora_a,
                                     const uint16_t* lora_b, int lora_r) {
  NS2_READY();
  if (M == 0) return NS2_OK;
  NS2_REQUIRE(At && Wt && scale && Y, "ns2_linear_i8_glu_rot_tiled: null At, Wt, scale or Y");
  NS2_REQUIRE(M > 0 && N > 0 && N % 512 == 0 && K > 0 && K % 256 == 0,
              "ns2_linear_i8_glu_rot_tiled: M=%d N=%d K=%d (N %% 512 == 0, K %% 256 == 0 required)", M, N, K);
  NS2_REQUIRE(aligned16(At) && aligned16(Wt) && aligned16(Y), "ns2_linear_i8_glu_rot_tiled: operands must be 16-byte aligned");
  NS2_REQUIRE(act >= NS2_ACT_NONE && act <= NS2_ACT_GELU_TANH, "ns2_linear_i8_glu_rot_tiled: unknown act %d", act);
  TGemmArgs p{reinterpret_cast<const half_t*>(At), reinterpret_cast<const uint8_t*>(Wt), scale, bias, nullptr, Y,
              nullptr, 0, 0, M, N, K, N, (M + 63) / 64, N / 64, 0, 0, alpha, act, 0};
  if (lora_r) {
    int rc = ns2::lora_prepare(&p.lt, lora_a, lora_b, lora_r, At, 2, K, M, K, "ns2_linear_i8_glu_rot_tiled_lora");
    if (rc) return rc;
    p.lb = reinterpret_cast<const half_t*>(lora_b);
    p.lr = lora_r;
  }
  ns2::ProfScope prof_("gemm_i8_glu_rot");
  // 64-row tiles fit a CU twice and run in pairs, one block's epilogue behind the other's products;
  // a 128-row tile does the work of a pair with 24 % fewer LDS bytes (104 instead of 136 per clock
  // of the matrix cores, where the LDS moves 128) but with its epilogue in the open. Where the
  // busiest CU gets an even number of 64-row tiles, that many halves as 128-row tiles are faster
  // (x 8192 x 1536, us 64 -> 128: 1100 rows 44.1 -> 38.7, 2048 53.0 -> 49.8, 3328 94.3 -> 88.9, 3952 101.6 ->
  // 96.8, 5200 143.3 -> 134.8); where it gets an odd number, a last pair's half would be padding
  // (1024 29.0 -> 39.1, 2304 70.5 -> 83.5, 6200 166.9 -> 175.6). A 64-row tile alone on its CU takes a third
  // stage for a long K, whose weights come from memory too late otherwise (x 16384 x 4096, 33-512 rows: 77 ->
  // 58-60 us; x 8192 x 1536: 23.4 -> 24.1).
  const long long per = ((long long)p.mblocks * (N / 512) + kCUs - 1) / kCUs;
  if (per == 1 && K > 2048) return launch_tiled<64, 512, 1, 8, 1, 1, 3, 1, 2, kI8, kLora, 1>(p);
  if (per % 2 == 0) return launch_tiled<128, 512, 1, 8, 1, 1, 2, 2, 2, kI8, kLora, 1>(p);
  return launch_tiled<64, 512, 1, 8, 1, 1, 2, 1, 4, kI8, kLora, 1>(p);
}

int ns2_linear_i8_tiled(const uint16_t* At, const int8_t* Wt, const float* scale, const float* bias,
                        float* C, int M, int N, int K, int ldc, long long cOff, float alpha, int act,
                        int resid, const float* gate, long long gOff) {
  return linear_tiled("ns2_linear_i8_tiled", kI8, At, 0, Wt, scale, bias, C, M, N, K, ldc, cOff, alpha, act, resid, gate,
                         gOff, nullptr, nullptr, 0);
}

int ns2_linear_i8_tiled_lora(const uint16_t* At, const int8_t* Wt, const float* scale, const float* bias,
                             float* C, int M, int N, int K, int ldc, long long cOff, float alpha, int act,
                             int resid, const float* gate, long long gOff, const uint16_t* lora_a,
                             const uint16_t* lora_b, int lora_r) {
  return linear_tiled("ns2_linear_i8_tiled_lora", kI8, At, 0, Wt, scale, bias, C, M, N, K, ldc, cOff, alpha, act, resid,
                         gate, gOff, lora_a, lora_b, lora_r);
}

int ns2_tile_bf16_weight(const uint16_t* W, uint16_t* Wt, int N, int K) {
  NS2_READY();
  NS2_REQUIRE(W && Wt && aligned16(W) && aligned16(Wt), "ns2_tile_bf16_weight: null or unaligned buffer");
  NS2_REQUIRE(N > 0 && K > 0 && N % 64 == 0 && K % 64 == 0,
              "ns2_tile_bf16_weight: N=%d and K=%d must be multiples of 64", N, K);
  const long long chunks = (long long)N * K / 8;
  ns2::ProfScope prof_("tile_bf16_weight");
  tile_w16_kernel<<<(unsigned)((chunks + 255) / 256), 256, 0, ns2::stream()>>>(W, Wt, N, K);
  NS2_LAUNCHED("tile_bf16_weight");
  return NS2_OK;
}

int ns2_linear_f16w_tiled(const uint16_t* At, const uint16_t* Wt, const float* bias, float* C, int M, int N, int K,
                          int ldc, long long cOff, float alpha, int act, int resid, const float* gate, long long gOff) {
  return linear_tiled("ns2_linear_f16w_tiled", kF16, At, 0, Wt, nullptr, bias, C, M, N, K, ldc, cOff, alpha, act, resid,
                      gate, gOff, nullptr, nullptr, 0);
}

int ns2_linear_f16w_tiled_lora(const uint16_t* At, const uint16_t* Wt, const float* bias, float* C, int M, int N,
                               int K, int ldc, long long cOff, float alpha, int act, int resid, const float* gate,
                               long long gOff, const uint16_t* lora_a, const uint16_t* lora_b, int lora_r) {
  return linear_tiled("ns2_linear_f16w_tiled_lora", kF16, At, 0, Wt, nullptr, bias, C, M, N, K, ldc, cOff, alpha, act,
                      resid, gate, gOff, lora_a, lora_b, lora_r);
}

int ns2_linear_i8_tiled_vpack(const uint16_t* At, const int8_t* Wt, const float* scale, const float* bias,
                              float* C, int M, int N, int K, int ldc, long long cOff, float alpha, int act,
                              const uint16_t* lora_a, const uint16_t* lora_b, int lora_r, uint16_t* vpk,
                              int vcol0, int H, int D, int Lk) {
  NS2_READY();
  if (M == 0) return NS2_OK;
  NS2_REQUIRE(vpk && ((uintptr_t)vpk & 15) == 0, "ns2_linear_i8_tiled_vpack: null or unaligned vpk");
  NS2_REQUIRE(H > 0 && D > 0 && D % 32 == 0 && vcol0 >= 0 && vcol0 % 64 == 0 && vcol0 + (long long)H * D == N,
              "ns2_linear_i8_tiled_vpack: the value columns [vcol0, vcol0 + H*D) must end the output "
              "(vcol0=%d H=%d D=%d N=%d; vcol0 %% 64 == 0, D %% 32 == 0)", vcol0, H, D, N);
  NS2_REQUIRE(M % 16 == 0 && M <= Lk, "ns2_linear_i8_tiled_vpack: M=%d must be a multiple of 16 and at most Lk=%d",
              M, Lk);
  return linear_tiled("ns2_linear_i8_tiled_vpack", kI8, At, 0, Wt, scale, bias, C, M, N, K, ldc, cOff, alpha, act, 0,
                         nullptr, 0, lora_a, lora_b, lora_r, vpk, vcol0, D, (Lk + 63) / 64);
}

}  // extern "C"
