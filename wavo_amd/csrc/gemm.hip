// The quantized GEMM of Pass::gemm (src/gpu/mod.rs:1394-1426) on gfx950 matrix cores:
//   c[m][j] = epi(Σ_k h(a[m][k]) · h(W[j][k]) + bias[j]),  h = round to f16 (RNE), f32 accumulate,
// as gemm.wgsl:170-242 and the CPU backend (src/cpu/gemm.rs:126-177) define it.  The GGUF's rows
// (src/gguf.rs:14-38; Q8_0 34-byte blocks (f16 scale + 32 int8), Q4_0 18-byte blocks (f16 scale + 16 bytes of
// nibbles), F16 or F32) are laid out, for the matrix-core kernels here, in tiles of 32 rows × 64 k in the order
// their lanes load them (WTile, weight_tiles_kernel), once, when the layer is created.
//
// Main kernel (gemm_lds_kernel; k % 64 == 0, W in Q8_0 / Q4_0 / F16, `a` in f16): a ring of LDS stages
// fed by the LDS DMA of gfx950 — per 64- or 128-wide k step, the a tile and W's tiles, all in 16-byte
// global_load_lds_dwordx4 of whole lines — so the next steps' bytes land while the MFMAs work on the
// current one.  (W's rows as the GGUF stores them, 68 or 36 bytes of a row per step from 4-byte aligned
// addresses, cost the loads' address path about twice the cycles and each lane 8 LDS reads of 8 bytes
// instead of 2 of 16: 750×4096×1024 13.3 -> 12.0 µs, 11616×4096×1024 125.2 -> 115.6 µs, the 60 s Parakeet
// call 3.94 -> 3.69 ms, 16 windows 23.8 -> 22.5 ms.)  Each lane dequantizes its 8 weights of a substep into
// the f16 operand of v_mfma_f32_32x32x16_f16: exact conversions of q (int8 by sub-dword conversions, a
// nibble n as the f16 1024 + n less 1032), then one packed f16 multiply by the block scale rounds q·d once
// to nearest even — f16(q·d), the reference's exact rounding (products q·d have at most 19 significant
// bits, so f32 and the f16 multiply round the same value).  The epilogues of Epilogue::params
// (src/gpu/mod.rs:445-455; gemm.wgsl:72-94) and the dual outputs are fused into the store, in f32
// or, for a consumer that rounds its input to f16 anyway (another GEMM), in f16.  Shapes with too
// few output tiles for the 256 CUs and a long k split it 4 ways into f32 partial sums that a second kernel
// adds in a fixed order before the epilogue.
//
// Few tiles (gemm_kw_kernel): the wavefronts of a workgroup split k and read W's tiles straight into
// registers.
//
// Fallback kernel (gemm_reg_kernel; any k % 32 == 0, F32 weights and layers without tiles): a
// double-buffered a tile in LDS and W's blocks as stored loaded straight into registers.
#include <algorithm>
#include <cstdio>
#include <mutex>
#include <type_traits>
#include <utility>

#include "internal.h"
#include "gemm_impl.h"

// Shapes of about one 128×128 tile per CU or more: whole k, and the tile shape whose rounds over the CUs take
// the least time.  Such a GEMM is bound by its last, partly filled round as much as by the tiles' own rate, so
// no single tile is best over a range of rows (µs, Q8_0): 3600×4096×1024 is 61.0 as 96×128 tiles in two k
// groups (4 rounds and three quarters of one) and 40.3 as 256×256 ones; 3000×4096×1024 51.0 (4 rounds) and 34.5 as
// 192×128 ones (one round, two workgroups per CU); 2500×3840×1280 53.6 -> 37.0; 11616×1280×5120 198.6 -> 166.6.
// Over 312 random shapes of 600 to 60000 rows, 256 to 5120 columns and k of 64 to 5120 in the three weight types
// the choice below is within 3% of the best of these tiles in the mean, 1.18 times as fast as one tile per range
// of tile counts.  Below k = 1024 a round costs what its launch, its ring's fill and its stores cost, much the
// same for one or two workgroups per CU and most for 256×256 tiles: from the line above 1024 carried down, those
// seemed the cheapest for a short k (10236×2432×384 43.4 as 256×256 ones, 31.7 as 128×128 ones).
struct TileRounds {
  GemmPlan plan;
  int per_cu, per_cu_f16;  // workgroups that share a CU (LDS), with quantized and with F16 weights
  float t[3][3];  // a round with 1 .. per_cu workgroups per CU, µs: as k goes to 0, at k = 1024, per 1024 of k from there
};
constexpr TileRounds TILE_ROUNDS[] = {
    {{96, 128, 1, 4, 3, 1, 0, 2}, 1, 1, {{7.0f, 13.5f, 6.5f}}},
    {{96, 128, 1, 4, 3, 1}, 2, 1, {{9.0f, 14.0f, 8.0f}, {16.0f, 21.5f, 13.2f}}},
    {{128, 128, 2, 4, 3, 1}, 2, 1, {{7.0f, 15.2f, 8.2f}, {7.3f, 25.7f, 18.2f}}},
    {{128, 128, 2, 2, 2, 1}, 3, 2, {{7.5f, 16.8f, 9.0f}, {7.7f, 25.7f, 17.7f}, {16.5f, 35.5f, 26.8f}}},
    {{192, 128, 2, 4, 2, 1}, 2, 2, {{7.0f, 20.0f, 11.5f}, {8.5f, 31.5f, 27.5f}}},
    {{256, 128, 2, 4, 3, 1}, 1, 1, {{10.0f, 25.8f, 16.6f}}},
    {{192, 256, 2, 4, 2, 1}, 1, 1, {{8.5f, 32.5f, 25.8f}}},
    {{256, 256, 2, 4, 2, 1}, 1, 1, {{26.0f, 40.0f, 31.6f}}},
};

GemmPlan least_rounds(int cus, int m, int cols, int k, bool f16) {
  GemmPlan best = TILE_ROUNDS[0].plan;
  float least = 0.0f;
  for (const TileRounds &r : TILE_ROUNDS) {
    const GemmPlan &p = r.plan;
    const int per_cu = f16 ? r.per_cu_f16 : r.per_cu;
    if (k % (64 * p.wk)) continue;
    const long tiles = (long)((cols + p.bn - 1) / p.bn) * ((m + p.bm - 1) / p.bm), slots = (long)cus * per_cu;
    auto round = [&](long wgs) {
      const float *c = r.t[(wgs - 1) / cus], x = (float)k / 1024.0f;
      return x < 1.0f ? c[0] + (c[1] - c[0]) * x : c[1] + c[2] * (x - 1.0f);
    };
    const float t = (float)(tiles / slots) * round(slots) + (tiles % slots ? round(tiles % slots) : 0.0f);
    if (least == 0.0f || t < least) least = t, best = p;
  }
  return best;
}

// Chosen per GEMM shape from measurements on MI355X (random operands, inside the encoder step, or
// replayed back to back for m ≥ 1024): many output tiles → the tile shape with the cheapest rounds; fewer
// → 96×128, 96×64 or 64×64 tiles in two k groups, wavefronts that split k, or, a long k over few tiles, k split
// 4 ways.  Ring slots of 64-wide k steps (a slot is refilled NS steps ahead, so NS − 1 steps hide the DMA's latency).
GemmPlan gemm_plan_for(const wh_ctx *ctx, int m, int cols, int k, int type) {
  const bool f16 = type == WH_F16;
  const int cus = ctx->cus > 0 ? ctx->cus : 256;
  const long t128 = (long)((cols + 127) / 128) * ((m + 127) / 128), t64 = (long)((cols + 63) / 64) * ((m + 63) / 64);
  const long t9664 = (long)((cols + 63) / 64) * ((m + 95) / 96);
  GemmPlan p{64, 64, 2, 2, 3, 1};
  if (t128 * 4 >= 3L * cus || (m >= 1024 && t128 * 2 > cus && k >= 512) || (f16 && t64 >= 2L * cus && k >= 256))
    // Three quarters of a 128×128 tile per CU or more (the FFN's first projection at 750 frames: 96×128 tiles
    // in two k groups, 256 of them), of many rows half a tile (1100×2048×1024 14.9 -> 12.0 µs, 2500×1024×1024
    // 15.7 -> 13.8 as 96×128 tiles), over a long enough k (4633×480×512 10.1 -> 8.5, but 5163×512×192 7.3 on 64×64
    // tiles, 8.0 on those); with fewer rows 64×64 tiles stay ahead (the 750-frame qkv projection, 144 of 128×128:
    // the 60 s step 4.32 ms, 4.51 as 96×128 ones), up to two per CU with F16 weights, whose tiles they then fetch
    // in step from a part of the memory's channels (500×4096×512 10.5 -> 8.4, 491×4544×256 9.6 -> 6.9).
    p = least_rounds(cus, m, cols, k, f16);
  else if (t128 * 4 <= cus && k % (4 * 64) == 0 && k / (4 * 64) >= 16)
    // Long k over few tiles (the FFN's down projection, 750 × 1024 × 4096): k split 4 ways over
    // 96×64 tiles of 2 wavefronts (96×32 per wavefront: each dequantized W fragment feeds three
    // MFMAs) in two slots: 512 workgroups, two per CU, whose barriers do not align (measured in
    // the encoder step, 60 s: 4.64 ms, against 4.68 for 128×64 tiles of 4 wavefronts, 4.75 for
    // 128×128 tiles of 8 wavefronts, 4.92 for 128×64 tiles in three slots, one per CU); in two k
    // groups where they divide every split (14.3 against 15.0 µs in the step, the groups' sums in
    // LDS planes of their own).
    p = {96, 64, 1, 2, 2, 4, 0, k % (4 * 128) == 0 ? 2 : 1};
  else if (f16 && t64 > cus && t128 * 4 <= 2L * cus && k % (4 * 64) == 0 && k / (4 * 64) >= 16)
    // F16 weights, whose ring of two k groups holds two slots only: k split (865×1472×4480, which cannot
    // split, is 30.8 µs on 64×64 tiles below, 33.9 in the two groups).
    p = {128, 128, 2, 2, 2, 4};
  else if (!f16 && t9664 > cus && t128 * 4 <= 2L * cus && k % 128 == 0 && k / (4 * 64) >= 16)
    // The same over up to half a 128×128 tile per CU (Whisper's fc2, 1500 × 1280 × 5120): the whole k in
    // two k groups over 96×128 tiles, 160 of them; no partial sums (four layers and their window 638 µs,
    // against 645 for 128×128 tiles with k split 4 ways, 640 for 96×64 tiles, 676 split 2 ways).  Not where the
    // 64×64 or 96×64 tiles below run at once, more of them than these (166×2752×4224, 44 of these: 26.9 µs, 20.0 as
    // 64×64 ones; 670×1664×4224 28.5 and, as 96×64 ones, 23.4; 300×4288×4224, 268 of those, 30.2 and 29.6).
    p = {96, 128, 1, 4, 3, 1, 0, 2};
  else if (t64 <= cus) {
    // Two k groups of 4 wavefronts over a 4-slot ring (one workgroup per CU; the 750-frame
    // 1024 × 1024 projections 9.5 against 10.0 µs in the step; deeper rings alone are slower there:
    // 10.8 for 5 slots, 11.4 for 8).  No split of k here: its partial sums and their finish cost more than the
    // extra workgroups win (409×1856×4992 24.5 in two splits, 21.1 whole; 549×1664×4736 F16 23.8 and 19.1; 750
    // frames of GigaAM, whose 768 × 3072 projections split in two and finished with the norm: 2 567 µs per call,
    // whole 2 423).
    if (k % 128 == 0) p = {64, 64, 2, 2, 4, 1, 0, 2};
  } else if (t64 < 2L * cus && k % 128 == 0 && !(f16 && t9664 > cus && k <= 1024))
    // One to two 64×64 tiles per CU (the 750-frame pointwise projection, 750 × 2048 × 1024): 96×64
    // tiles of one row of 2 wavefronts in two k groups, one workgroup per CU (11.7 against 12.7 µs
    // in the step for 64×64 tiles; 12.2 with 4 slots).  64×64 tiles stay where there are no two groups, an odd
    // number of steps (1393×1344×2880 Q4_0 24.2 against 34.0, 918×1472×1984 F16 15.7 against 20.4), and with F16
    // weights over more than a 96×64 tile per CU of a short k (937×1728×1024 11.6 against 12.9; 623×2688×1536 15.4
    // and 16.0, 571×3520×1920 20.7 and 19.5).
    p = {96, 64, 1, 2, 2, 1, 0, 2};
  // Few tiles: wavefronts that split k (gemm_kw_kernel), the smallest of its tiles that still run at once
  // (one workgroup per CU), whose chain of steps is then the shortest.  µs per encoder call with that one
  // layer on the LDS-DMA kernel and here: 60 Parakeet frames 2 289 against 2 073 for the 1024 × 1024
  // projections (32×32 tiles), 2 298 for 4096 × 1024 (32×64), 2 807 for all of them; 275 GigaAM frames
  // 1 790 against 1 682 for the 768 × 768 ones, 1 854 for 768 × 3072.  Not over one or two steps of k, whose sums
  // cost more than the split saves (recorded, one after the other: 260×1408×64 3.9 on the LDS-DMA kernel, 4.3
  // here, 2020×160×128 4.2 and 4.4 on 32×64 tiles, but 103×96×128 4.2 and 3.7).  With 64×64 tiles the LDS-DMA
  // kernel's two k groups are the faster ones while the tiles run at once (750 frames' 1024 × 1024: 3 584
  // against 3 626; 275 frames' 3072 × 1024: 2 846 against 2 886), and so are its 96×64 ones above
  // (750×2048×1024 10.7 there, 12.5 here; 458×2752×1920 Q4_0 13.3 and 16.0); this kernel for one to two tiles per
  // CU of few rows whose 96×64 tiles are too many or walk an odd number of steps (500×3072×1024 12.4 and 12.2,
  // 392×3520×1728 22.5 and 16.4), with Q8_0 and Q4_0: with F16 weights it holds over 256 registers, one
  // workgroup per CU (595×2368×896 11.7 on 96×64 tiles, 10.4 on 64×64 ones, 14.5 here).
  {
    const long t32 = (long)((cols + 31) / 32) * ((m + 31) / 32), t3264 = (long)((cols + 63) / 64) * ((m + 31) / 32);
    if ((size_t)m * k < ((size_t)1 << 30)) {  // 32-bit byte offsets into a
      if (t32 <= cus && k >= 128) p = {32, 32, 1, 1, 2, 1, PIPE_KW, 8};
      else if (t32 > cus && t3264 <= cus && k >= 192) p = {32, 64, 1, 1, 2, 1, PIPE_KW, 8};
      else if (!f16 && m < 1024 && k <= 2048 && t64 > cus && t64 <= 2L * cus && (t9664 > cus || k % 128))
        p = {64, 64, 1, 1, 2, 1, PIPE_KW, 4};
    }
  }
  if (ctx->gemm_plan[0]) {  // tuning override (wh_tune "gemm_plan"): bm, bn, wm, wn, stages, split, pipeline, kgroups
    const int *o = ctx->gemm_plan;
    p = {o[0], o[1], o[2], o[3], o[4], o[5], o[6], std::max(1, o[7])};
  }
  for (const auto &o : ctx->gemm_shape_plans)  // tuning override for one shape (wh_tune "gemm_shape_plans")
    if (o[0] == m && o[1] == cols && o[2] == k) p = {o[3], o[4], o[5], o[6], o[7], o[8], o[9], std::max(1, o[10])};
  if (p.pipe == PIPE_KW) {  // (any k steps: a wavefront may have one less than another, or none)
    p.split = 1;
    return p;
  }
  // Whole k steps per split and k group.
  if (k % (64 * p.wk)) p.wk = 1;
  if (k % (64 * p.wk * p.split)) p.split = 1;
  return p;
}

namespace {

// a (f32) rounded to f16 (RNE; h of the reference), for the GEMMs whose producer wrote f32.
__global__ __launch_bounds__(256) void to_half_kernel(const float4 *__restrict__ x, half4 *__restrict__ y, size_t n4) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (size_t)gridDim.x * 256) {
    const float4 v = x[i];
    y[i] = half4{(_Float16)v.x, (_Float16)v.y, (_Float16)v.z, (_Float16)v.w};
  }
}

// The main kernel's conditions: weight tiles (64-wide k steps over Q8_0 / Q4_0 / F16 weights), and an output
// whose rows start on 16 bytes (its epilogue stores 8 columns at a time).
bool lds_path(const wh_linear *l, const void *c, int ldc) {
  return l->wt && ldc % 8 == 0 && (uintptr_t)c % 16 == 0;
}


// The weight tiles from the GGUF bytes (see WTile): a lane of a tile per thread.
template <int WT>
__global__ __launch_bounds__(256) void weight_tiles_kernel(const uint8_t *__restrict__ w, uint8_t *__restrict__ wt, int rows,
                                                           int nkt, size_t row_bytes, size_t lanes) {
  constexpr int BLK = WT == WH_Q8_0 ? 34 : 18;
  for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < lanes; e += (size_t)gridDim.x * 256) {
    const size_t tile = e / 64;
    const int lane = e % 64, g = lane / 32, row = (int)(tile / nkt) * 32 + lane % 32, kt = (int)(tile % nkt);
    uint8_t *dst = wt + tile * WTile<WT>::BYTES;
    const uint8_t *src = w + (size_t)row * row_bytes;
    u32x4 q[WTile<WT>::LOADS] = {};
    uint32_t sc = 0;
    if (row < rows) {
      if constexpr (WT == WH_F16) {
        // (rows of k % 64 == 0 halves: 16-byte aligned)
#pragma unroll
        for (int s = 0; s < 4; s++) q[s] = *(const u32x4 *)(src + 128 * (size_t)kt + 32 * s + 16 * g);
      } else {
        const uint16_t *b = (const uint16_t *)(src + (size_t)kt * 2 * BLK);  // the step's block pair
        sc = b[0] | (uint32_t)b[BLK / 2] << 16;
        if constexpr (WT == WH_Q8_0) {
#pragma unroll
          for (int s = 0; s < 4; s++) {  // substep s: bytes 16·(s % 2) + 8g .. of block s / 2
            const uint16_t *d = b + (s / 2) * (BLK / 2) + 1 + 8 * (s & 1) + 4 * g;
            q[s / 2][2 * (s & 1)] = d[0] | (uint32_t)d[1] << 16, q[s / 2][2 * (s & 1) + 1] = d[2] | (uint32_t)d[3] << 16;
          }
        } else {
#pragma unroll
          for (int s = 0; s < 4; s++) {  // element 16·(s % 2) + 8g + i of block s / 2: a nibble of byte 8g + i
            const uint8_t *d = (const uint8_t *)b + (s / 2) * BLK + 2 + 8 * g;
            uint32_t x = 0;
#pragma unroll
            for (int i = 0; i < 8; i++) x |= (uint32_t)(s & 1 ? d[i] >> 4 : d[i] & 15) << (4 * (i / 2) + 16 * (i & 1));
            q[0][s] = x;
          }
        }
      }
    }
#pragma unroll
    for (int i = 0; i < WTile<WT>::LOADS; i++) *(u32x4 *)(dst + 1024 * i + 16 * lane) = q[i];
    if (WT != WH_F16 && g == 0) *(uint32_t *)(dst + WTile<WT>::DATA + 4 * lane) = sc;
  }
}

// Scratch bytes for the split-k partial sums of an m-row GEMM (0 when it does not split).
size_t split_bytes(const wh_ctx *ctx, const wh_linear *l, int m) {
  const GemmPlan p = gemm_plan_for(ctx, m, l->cols, l->k, l->type);
  return p.split > 1 ? (size_t)p.split * m * l->cols * 4 : 0;
}

// a16: f16 rows; part: scratch for split-k partial sums (or NULL: no split).  With `splits`, a split
// GEMM stops after writing its partial sums (the caller finishes them) and *splits is the count
// (1: c was written whole).
int launch_lds(wh_ctx *ctx, const _Float16 *a, const wh_linear *l, void *c, int m, int ldc, int epi, float alpha,
               bool out16, float *part, int *splits = nullptr, const HeadsOut *ho = nullptr, int nho = 0) {
  switch (l->type) {
    case WH_Q8_0: return gemm_lds_q8_0(ctx, a, l, c, m, ldc, epi, alpha, out16, part, splits, ho, nho);
    case WH_Q4_0: return gemm_lds_q4_0(ctx, a, l, c, m, ldc, epi, alpha, out16, part, splits, ho, nho);
    default: return gemm_lds_f16(ctx, a, l, c, m, ldc, epi, alpha, out16, part, splits, ho, nho);
  }
}

template <int WT, bool ALIGNED, bool A16, bool OUT16>
int launch_t(wh_ctx *ctx, const void *a, const wh_linear *l, void *c, int m, int ldc, int epi, float alpha) {
  // Tile: the largest whose grid still gives every CU a workgroup, else the smallest.
  const int cus = ctx->cus > 0 ? ctx->cus : 256;
  auto tiles = [&](int bm, int bn) { return (long)((l->cols + bn - 1) / bn) * ((m + bm - 1) / bm); };
  int bm = 64, bn = 64;
  if (tiles(128, 128) >= cus) bm = 128, bn = 128;
  else if (tiles(64, 128) >= cus) bm = 64, bn = 128;
  dim3 grid((l->cols + bn - 1) / bn, (m + bm - 1) / bm);
  // Algorithmic work: 2·m·rows·k flops over the real rows; bytes of W as stored, a, c (and c read
  // back by the residual epilogues).
  static const char *tn = WT == WH_F32 ? "f32" : WT == WH_F16 ? "f16" : WT == WH_Q8_0 ? "q8_0" : "q4_0";
  char name[64];
  snprintf(name, sizeof name, "gemm_reg_%s%s_%dx%d", tn, A16 ? "_a16" : "", bm, bn);
  double width = l->cols + l->dual;
  double bytes = (double)l->rows * l->row_bytes + (A16 ? 2.0 : 4.0) * m * l->k +
                 (OUT16 ? 2.0 : 4.0) * m * width * (epi == WH_RESIDUAL || epi == WH_GELU_RESIDUAL ? 2 : 1);
  ProfScope prof(ctx, name, 2.0 * m * l->rows * l->k, bytes);
  if (bm == 128)
    wh_launch(ctx, gemm_reg_kernel<WT, 128, 128, ALIGNED, A16, OUT16>, grid, 256, 0, a, l->w, l->bias, c, m, l->rows, l->cols, l->k, l->dual, ldc, epi, alpha, l->row_bytes);
  else if (bn == 128)
    wh_launch(ctx, gemm_reg_kernel<WT, 64, 128, ALIGNED, A16, OUT16>, grid, 256, 0, a, l->w, l->bias, c, m, l->rows, l->cols, l->k, l->dual, ldc, epi, alpha, l->row_bytes);
  else
    wh_launch(ctx, gemm_reg_kernel<WT, 64, 64, ALIGNED, A16, OUT16>, grid, 256, 0, a, l->w, l->bias, c, m, l->rows, l->cols, l->k, l->dual, ldc, epi, alpha, l->row_bytes);
  return wh_launched(ctx, "gemm");
}

template <bool A16, bool OUT16>
int launch_typed(wh_ctx *ctx, const void *a, const wh_linear *l, void *c, int m, int ldc, int epi, float alpha) {
  const bool aligned = l->k % 64 == 0;
  if (!l->w) return wh_fail(ctx, WH_EARG, "gemm: only weight tiles are held, and the output is not 16-byte aligned");
  switch (l->type) {
    case WH_F32: return launch_t<WH_F32, true, A16, OUT16>(ctx, a, l, c, m, ldc, epi, alpha);
    case WH_F16: return launch_t<WH_F16, true, A16, OUT16>(ctx, a, l, c, m, ldc, epi, alpha);
    case WH_Q8_0:
      return aligned ? launch_t<WH_Q8_0, true, A16, OUT16>(ctx, a, l, c, m, ldc, epi, alpha)
                     : launch_t<WH_Q8_0, false, A16, OUT16>(ctx, a, l, c, m, ldc, epi, alpha);
    case WH_Q4_0:
      return aligned ? launch_t<WH_Q4_0, true, A16, OUT16>(ctx, a, l, c, m, ldc, epi, alpha)
                     : launch_t<WH_Q4_0, false, A16, OUT16>(ctx, a, l, c, m, ldc, epi, alpha);
  }
  return wh_fail(ctx, WH_EARG, "gemm: weight type %d", l->type);
}

}  // namespace

size_t weight_tile_bytes(int type, int rows, int k) {
  if (k % 64) return 0;
  const size_t tiles = (size_t)((rows + 31) / 32) * (k / 64);
  switch (type) {
    case WH_Q8_0: return tiles * WTile<WH_Q8_0>::BYTES;
    case WH_Q4_0: return tiles * WTile<WH_Q4_0>::BYTES;
    case WH_F16: return tiles * WTile<WH_F16>::BYTES;
  }
  return 0;
}

int launch_weight_tiles(wh_ctx *ctx, const wh_linear *l, const uint8_t *rows) {
  const size_t lanes = (size_t)((l->rows + 31) / 32) * (l->k / 64) * 64;
  const int blocks = (int)std::min<size_t>((lanes + 255) / 256, 16384);
  auto go = [&](auto kernel) { wh_launch(ctx, kernel, blocks, 256, 0, rows, l->wt, l->rows, l->k / 64, l->row_bytes, lanes); };
  switch (l->type) {
    case WH_Q8_0: go(weight_tiles_kernel<WH_Q8_0>); break;
    case WH_Q4_0: go(weight_tiles_kernel<WH_Q4_0>); break;
    case WH_F16: go(weight_tiles_kernel<WH_F16>); break;
    default: return WH_OK;
  }
  return wh_launched(ctx, "weight tiles");
}

bool gemm_glu_ok(const wh_linear *l, const void *c) {
  return l && !l->dual && l->rows == l->cols && l->cols % 16 == 0 && lds_path(l, c, l->cols / 2);
}

// glu: the caller takes EPI_GLU (launch_gemm_h only; the public entry points take WH_BIAS .. WH_TANH).
static int check(wh_ctx *ctx, const void *a, const wh_linear *l, const void *c, int m, int epi, bool glu = false) {
  if (m < 0 || !l || (m && (!a || !c))) return wh_fail(ctx, WH_EARG, "gemm: bad arguments (m %d)", m);
  if ((epi < WH_BIAS || epi > WH_TANH) && !(glu && epi == EPI_GLU))
    return wh_fail(ctx, WH_EARG, "gemm: epilogue %d", epi);
  if (epi == EPI_GLU && !gemm_glu_ok(l, c)) return wh_fail(ctx, WH_EARG, "gemm: GLU epilogue off its layout");
  if ((uintptr_t)a % 16) return wh_fail(ctx, WH_EARG, "gemm: a must be 16-byte aligned");
  return WH_OK;
}

// Workspace of an f32-input GEMM on the main kernel: the f16 copy of `a`, then the split-k partial sums.
static size_t f32_gemm_abytes(const wh_linear *l, int m) { return ((size_t)m * l->k * 2 + 255) / 256 * 256; }

// The f32-input GEMM on the main kernel with its workspace at ws (f32_gemm_abytes + split_bytes).
static int gemm_f32_ws(wh_ctx *ctx, const float *a, const wh_linear *l, float *c, int m, int ldc, int epi, float alpha,
                       uint8_t *ws) {
  const size_t n = (size_t)m * l->k, abytes = f32_gemm_abytes(l, m);
  _Float16 *a16 = (_Float16 *)ws;
  {
    ProfScope prof(ctx, "to_half", 0.0, 6.0 * n);
    const size_t n4 = n / 4;
    const int blocks = (int)std::min<size_t>((n4 + 255) / 256, 4096);
    wh_launch(ctx, to_half_kernel, blocks, 256, 0, (const float4 *)a, (half4 *)a16, n4);
    if (int rc = wh_launched(ctx, "gemm: rounding a")) return rc;
  }
  return launch_lds(ctx, a16, l, c, m, ldc, epi, alpha, false, (float *)(ws + abytes));
}

int launch_gemm(wh_ctx *ctx, const float *a, const wh_linear *l, float *c, int m, int ldc, int epi, float alpha) {
  if (int rc = check(ctx, a, l, c, m, epi)) return rc;
  if (m == 0) return WH_OK;
  if (!lds_path(l, c, ldc)) return launch_typed<false, false>(ctx, a, l, c, m, ldc, epi, alpha);
  // The main kernel takes a in f16: round it once into scratch (followed by the split partials).
  uint8_t *ws = (uint8_t *)wh_scratch(ctx, f32_gemm_abytes(l, m) + split_bytes(ctx, l, m));
  if (!ws) return WH_EOOM;
  return gemm_f32_ws(ctx, a, l, c, m, ldc, epi, alpha, ws);
}

// ------------------------------------------------------------------ the GEMM that allocates nothing
// wh_gemm_noalloc's workspace (the f16 copy of `a` and the split-k partial sums): a file-scope device
// array, which every device the library runs on holds until the process ends.  In host code its name
// is not a device address: the address comes from hipGetSymbolAddress, once per device with that
// device current (gemm_noalloc_init, from wh_open), and only that address is used.  Every call on a
// device shares the array, so calls that overlap on one device (other streams or contexts) race; a
// call writes all of the workspace it reads (the rounded `a` and every split's partial plane), so
// nothing in it has to start at zero.
constexpr size_t NOALLOC_BYTES = (size_t)32 << 20;
static __device__ __align__(256) uint8_t scratch[NOALLOC_BYTES];

namespace {
constexpr int NOALLOC_DEVICES = 64;
// Per device: the workspace address, the failed lookup's error, and the last call's stream with an
// event recorded after its kernels (created at set-up, with the address).
struct NoallocDevice {
  void *addr = nullptr;
  hipError_t err = hipSuccess;
  hipEvent_t done = nullptr;
  hipStream_t last = nullptr;
};
std::mutex noalloc_mu;
NoallocDevice noalloc_dev[NOALLOC_DEVICES];
}  // namespace

int gemm_noalloc_init(wh_ctx *ctx) {
  std::lock_guard<std::mutex> lock(noalloc_mu);
  ctx->noalloc = nullptr;
  if (ctx->device < 0 || ctx->device >= NOALLOC_DEVICES) return WH_EGPU;
  NoallocDevice &d = noalloc_dev[ctx->device];
  if (!d.addr && d.err == hipSuccess) {
    void *p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e == hipSuccess && p) e = hipEventCreateWithFlags(&d.done, hipEventDisableTiming);
    if (e != hipSuccess || !p) {
      (void)hipGetLastError();
      d.err = e != hipSuccess ? e : hipErrorInvalidSymbol;
    } else {
      d.addr = p;
    }
  }
  ctx->noalloc = d.addr;
  ctx->noalloc_error = ctx->noalloc ? hipSuccess : d.err;
  return ctx->noalloc ? WH_OK : WH_EGPU;
}

size_t wh_gemm_noalloc_limit(void) { return NOALLOC_BYTES; }

int wh_gemm_noalloc(wh_ctx *ctx, const float *a, const wh_linear *l, float *c, int m, int epi, float alpha) {
  if (!ctx || !l) return WH_EARG;
  if (int rc = check(ctx, a, l, c, m, epi)) return rc;
  if (!ctx->noalloc)
    return wh_fail(ctx, WH_EGPU, "wh_gemm_noalloc: no workspace address on device %d (%s)", ctx->device,
                   hipGetErrorString(ctx->noalloc_error));
  if (ctx->prof == 1) return wh_fail(ctx, WH_EARG, "wh_gemm_noalloc: per-launch profiling creates events; turn it off");
  if (m == 0) return WH_OK;
  const int ldc = l->cols + l->dual;
  if (!lds_path(l, c, ldc)) return launch_typed<false, false>(ctx, a, l, c, m, ldc, epi, alpha);  // no workspace
  const size_t need = f32_gemm_abytes(l, m) + split_bytes(ctx, l, m);
  if (need > NOALLOC_BYTES)
    return wh_fail(ctx, WH_EARG, "wh_gemm_noalloc: %d x %d x %d needs %zu bytes of workspace, more than its %zu", m,
                   l->rows, l->k, need, NOALLOC_BYTES);
  // The workspace is shared by every call on the device: a call from another stream while the last
  // call's kernels may still run would corrupt both, so it is refused (calls must be serialized).  A
  // stream under capture is neither checked nor remembered (its kernels run at replay).
  std::lock_guard<std::mutex> lock(noalloc_mu);
  NoallocDevice &d = noalloc_dev[ctx->device];
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(ctx->stream, &cs) != hipSuccess) {
    (void)hipGetLastError();
    cs = hipStreamCaptureStatusNone;
  }
  const bool capturing = cs != hipStreamCaptureStatusNone;
  if (!capturing && d.last && d.last != ctx->stream) {
    const hipError_t q = hipEventQuery(d.done);
    if (q != hipSuccess) {
      (void)hipGetLastError();
      if (q == hipErrorNotReady)
        return wh_fail(ctx, WH_EARG,
                       "wh_gemm_noalloc: the last call on device %d (another stream) may still be running; its "
                       "workspace is shared, so calls on one device must not overlap", ctx->device);
    }
  }
  const int rc = gemm_f32_ws(ctx, a, l, c, m, ldc, epi, alpha, (uint8_t *)ctx->noalloc);
  if (rc == WH_OK && !capturing) {
    if (hipEventRecord(d.done, ctx->stream) == hipSuccess) d.last = ctx->stream;
    else (void)hipGetLastError();
  }
  return rc;
}

int launch_to_half(wh_ctx *ctx, const float *x, void *y, size_t n) {
  if (n % 4 || (uintptr_t)x % 16 || (uintptr_t)y % 8) return wh_fail(ctx, WH_EARG, "to_half: n %% 4 == 0 and aligned buffers");
  if (!n) return WH_OK;
  ProfScope prof(ctx, "to_half", 0.0, 6.0 * n);
  const size_t n4 = n / 4;
  const int blocks = (int)std::min<size_t>((n4 + 255) / 256, 4096);
  wh_launch(ctx, to_half_kernel, blocks, 256, 0, (const float4 *)x, (half4 *)y, n4);
  return wh_launched(ctx, "to_half");
}

int launch_gemm_h(wh_ctx *ctx, const void *a16, const wh_linear *l, void *c, int m, int ldc, int epi, float alpha,
                  int out16) {
  if (int rc = check(ctx, a16, l, c, m, epi, true)) return rc;
  if (out16 && (epi == WH_RESIDUAL || epi == WH_GELU_RESIDUAL))
    return wh_fail(ctx, WH_EARG, "gemm: residual epilogues accumulate into f32 outputs");
  if (epi == EPI_GLU && (out16 || ldc != l->cols / 2))
    return wh_fail(ctx, WH_EARG, "gemm: the GLU epilogue writes f32 rows of cols / 2");
  if (m == 0) return WH_OK;
  // (no split-k partials for the GLU epilogue: the main kernel finishes its own tiles)
  if (epi == EPI_GLU) return launch_lds(ctx, (const _Float16 *)a16, l, c, m, ldc, epi, alpha, false, nullptr);
  if (lds_path(l, c, ldc)) {
    const size_t pb = split_bytes(ctx, l, m);
    float *part = nullptr;
    if (pb && !(part = (float *)wh_scratch(ctx, pb))) return WH_EOOM;
    return launch_lds(ctx, (const _Float16 *)a16, l, c, m, ldc, epi, alpha, out16 != 0, part);
  }
  if (out16) return launch_typed<true, true>(ctx, a16, l, c, m, ldc, epi, alpha);
  return launch_typed<true, false>(ctx, a16, l, c, m, ldc, epi, alpha);
}

int launch_gemm_h_heads(wh_ctx *ctx, const void *a16, const wh_linear *l, void *c, int m, int ldc, int epi,
                        const HeadsOut *outs, int n) {
  if (int rc = check(ctx, a16, l, c, m, epi)) return rc;
  if (epi == WH_RESIDUAL || epi == WH_GELU_RESIDUAL) return wh_fail(ctx, WH_EARG, "gemm: packed output with a residual epilogue");
  if (!lds_path(l, c, ldc) || !outs || n <= 0) return wh_fail(ctx, WH_EARG, "gemm: packed output needs the main kernel");
  for (int i = 0; i < n; i++)
    if (!outs[i].dst || outs[i].hd <= 0) return wh_fail(ctx, WH_EARG, "gemm: packed output %d", i);
  if (m == 0) return WH_OK;
  return launch_lds(ctx, (const _Float16 *)a16, l, c, m, ldc, epi, 0.0f, true, nullptr, nullptr, outs, n);
}

int launch_gemm_h_ln(wh_ctx *ctx, const void *a16, const wh_linear *l, float *x, int m, float alpha, const float *g,
                     const float *b, void *y, int out16, int keep_x, const float *g2, const float *b2, void *y2,
                     int residual) {
  const int epi = residual ? WH_RESIDUAL : WH_BIAS;
  if (int rc = check(ctx, a16, l, x, m, epi)) return rc;
  if (m == 0) return WH_OK;
  if (g2 && (out16 || !b2 || !y2)) return wh_fail(ctx, WH_EARG, "gemm_h_ln: the second norm takes an f32 y");
  const int cols = l->cols;
  // The GEMM adds the residual into x, then one or two LayerNorm launches (one pass for both norms,
  // the fused finish kernel without partial sums, measured slower at 11616 rows: 51 against ~24 µs).
  auto unfused = [&](int rc) {
    if (rc) return rc;
    if ((rc = launch_layer_norm(ctx, x, g, b, y, m, cols, nullptr, nullptr, 0, out16))) return rc;
    return g2 ? launch_layer_norm(ctx, (const float *)y, g2, b2, y2, m, cols, nullptr, nullptr, 0, 1) : WH_OK;
  };
  if (l->dual || !lds_path(l, x, cols)) return unfused(launch_gemm_h(ctx, a16, l, x, m, cols, epi, alpha, 0));
  const size_t pb = split_bytes(ctx, l, m);
  float *part = nullptr;
  if (pb && !(part = (float *)wh_scratch(ctx, pb))) return WH_EOOM;
  int splits = 1;
  if (int rc = launch_lds(ctx, (const _Float16 *)a16, l, x, m, cols, epi, alpha, false, part, &splits)) return rc;
  if (splits > 1)
    return launch_split_residual_ln(ctx, part, splits, l->bias, l->rows, residual ? alpha : 1.0f, x, g, b, y, m, cols,
                                    out16, keep_x, g2, b2, y2, residual);
  return unfused(WH_OK);
}
