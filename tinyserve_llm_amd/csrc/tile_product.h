// One tile of x · W^T in a workgroup, for the products of many rows (gemm_slices.hip, gemm_whole.hip).
//
// Operands go from memory straight into LDS, 64 of K a step, as gemm_glu.hip lays them out (a row's eight 16-byte pieces
// turned by (row / 2) % 8), and like there x has XN = 2 steps in LDS, W three, and a step one barrier, in its middle (three and five
// steps of both: the same within a tenth, but with tiles of 64 x 128, whose steps are short: 300 rows, N 2,048, K 4,096 19.6 and 17.5 µs with the norm).
// The last two steps are written out apart, so that no load is made that nothing reads.
#pragma once
#include "lds_loads.h"

#define COMPUTE_UNITS 256

// Whether tiles of `bm` rows (128, 192 or 256) are 192 columns wide instead of 256: where the chip, which holds one a compute unit, takes as many rounds for them. A step
// costs what its products do and a third of a microsecond, and a tile's sums are the same bits. us by 256 and by 192 columns: whole, 32-bit, over 2,048, 256 rows, 1,000 x
// 11,296 (180 and 236 tiles) 54.0 and 46.2, 2,048 x 10,304 (328 and 432) 103 and 90; 192 rows, 768 x 10,304 (164 and 216) 42.8 and 36.7, 1,792 x 9,280 (370 and 490)
// 85.6 and 73.6; 128 rows, 1,000 x 6,144 (192 and 256) 33.6 and 30.7, but in one round only (1,200 x 8,192, 320 and 430, 55.5 and 56.4). A round more: 1,024 x
// 12,352 (196 and 260) 54.7 and 77.4. In two slices with the norm, 192 rows, 1,514 x 3,072 over 8,192 (192 and 256) 86.6 and
// 84.1, over 3,072 51.5 and 46.4; 256 rows, 2,048 x 3,072 over 8,192 (192 and 256) 106.0 and 101.6. (224 columns in tiles of 256 rows: 54.2 where 256 take 54.0.)
// The plans that choose between tiles, and between these and the library (whole_plan, slices_plan, group_plan of ops/hip.py), cost 256 columns: where tiles go narrow a product
// takes 2 to 15 % less than they count on, so they leave gains there that they do not see. (qkv_rope_whole_plan knows its narrow tile.)
static inline bool tiles_go_narrow(int64_t wide, int64_t narrow, int bm) {
  const int64_t rounds = (wide + COMPUTE_UNITS - 1) / COMPUTE_UNITS;
  return narrow <= rounds * COMPUTE_UNITS && (bm > 128 || rounds == 1);
}

template <int BM, int BN, int WM, int WN, int XN> struct TileProduct {
  static constexpr int WAVES = WM * WN, TM = BM / WM / 16, TN = BN / WN / 16;
  static constexpr int NX = BM / 8 / WAVES, NW = BN / 8 / WAVES;      // kilobytes of a step that a wave fetches
  static constexpr int XS = BM * 128, WS = BN * 128;                  // bytes of a step of x and of W
  static constexpr int LDS = XN * XS + 3 * WS;
  static constexpr int MIN_STEPS = 3;
  static_assert(BM % (8 * WAVES) == 0 && BN % (8 * WAVES) == 0, "whole kilobytes a wave");

  // Where in the tile the row lies that this lane fetches with a wave's load q of x or of W, and the byte of its 16 in a step of that row
  static __device__ __forceinline__ int x_row(int q) { return (wave_index() * NX + q) * 8 + (int)(threadIdx.x % TS_WAVE) / 8; }
  static __device__ __forceinline__ int w_row(int q) { return (wave_index() * NW + q) * 8 + (int)(threadIdx.x % TS_WAVE) / 8; }
  static __device__ __forceinline__ uint32_t piece(int row) { return ((threadIdx.x % 8) ^ ((row >> 1) & 7)) * 16; }

  // acc[j][i]: lane (r, g) gets columns 16 j + 4 g .. + 3 of row 16 i + r of the wave's part of the tile (rows from wm 16 TM,
  // columns from wn 16 TN; wave = wm + WM wn). x and W are fetched from their bases at xoff and woff, 128 bytes further on a step;
  // `steps` at least MIN_STEPS.
  static __device__ __forceinline__ void run(unsigned char* lds, __amdgpu_buffer_rsrc_t rsrc_x, __amdgpu_buffer_rsrc_t rsrc_w, const uint32_t (&xoff)[NX],
                                             const uint32_t (&woff)[NW], int steps, float4_t (&acc)[TN][TM]) {
    const int lane = threadIdx.x % TS_WAVE, r = lane % 16, g = lane / 16;
    const int wave = wave_index(), wm = wave % WM, wn = wave / WM;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)lds;
    const uint32_t xfirst = lds0 + wave * NX * 1024, wfirst = lds0 + XN * XS + wave * NW * 1024;
    auto fetch_x = [&](int step, uint32_t place) {
#pragma unroll
      for (int q = 0; q < NX; ++q) load_to_lds(rsrc_x, xfirst + place + q * 1024, xoff[q], (uint32_t)step * 128);
    };
    auto fetch_w = [&](int step, uint32_t place) {
#pragma unroll
      for (int q = 0; q < NW; ++q) load_to_lds(rsrc_w, wfirst + place + q * 1024, woff[q], (uint32_t)step * 128);
    };
    const uint32_t rd0 = (uint32_t)(r * 128 + (g ^ (r >> 1)) * 16), rd1 = rd0 ^ 64;      // a step's two halves of K
    const unsigned char* rx = lds + wm * TM * 2048;
    const unsigned char* rw = lds + XN * XS + wn * TN * 2048;
    u32x4_t fw[2][TN], fx[2][TM];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[j][i] = (float4_t){0.f, 0.f, 0.f, 0.f};
    fetch_x(0, 0), fetch_w(0, 0), fetch_w(1, WS), fetch_x(1, XS);
    if constexpr (XN == 3) fetch_x(2, 2 * XS);
    wait_for<NW + NX * (XN - 1)>();
    __builtin_amdgcn_s_barrier();
    uint32_t xc = 0, wc = 0, wfree = 2 * WS;      // the places of the step that is multiplied, and of the next one of W to come
#define TS_READ(S, RD)                                                                                         \
  _Pragma("unroll") for (int j = 0; j < TN; ++j) fw[S][j] = *(const u32x4_t*)(rw + (RD + wc) + j * 2048);      \
  _Pragma("unroll") for (int i = 0; i < TM; ++i) fx[S][i] = *(const u32x4_t*)(rx + (RD + xc) + i * 2048);
#define TS_MULTIPLY(S)                                                                                         \
  _Pragma("unroll") for (int i = 0; i < TM; ++i)                                                               \
      _Pragma("unroll") for (int j = 0; j < TN; ++j) acc[j][i] = mfma32v(fw[S][j], fx[S][i], acc[j][i]);
// the order of a half step: TM TN products, among their first two thirds the TM + TN operand reads, among all the loads
#define TS_DEAL(LOADS)                                                                                         \
  _Pragma("unroll") for (int q = 0; q < TM * TN; ++q) {                                                        \
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                                         \
    if ((q + 1) * (TM + TN) * 3 / 2 / (TM * TN) > q * (TM + TN) * 3 / 2 / (TM * TN)) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0); \
    if ((q + 1) * (LOADS) / (TM * TN) > q * (LOADS) / (TM * TN)) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0); \
  }                                                                                                            \
  __builtin_amdgcn_sched_barrier(0);
// A step that another follows, with (where W, X) the loads of W's step after the next one and of x's XN steps on. At its
// barrier every wave has read the last of the step's x and of W (so their places may be filled), and the next step has
// landed once at most LATER loads are under way: W's step after it and x's XN - 2 steps after it.
#define TS_STEP(W, X, LATER)                                                                                   \
  __builtin_amdgcn_sched_barrier(0);                                                                           \
  if constexpr (W) fetch_w(s + 2, wfree);                                                                      \
  TS_READ(1, rd1)                                                                                              \
  TS_MULTIPLY(0)                                                                                               \
  TS_DEAL(W ? NW : 0)                                                                                          \
  const uint32_t xfree = xc;                                                                                   \
  wfree = wc;                                                                                                  \
  xc = xc == (XN - 1) * XS ? 0 : xc + XS;                                                                      \
  wc = wc == 2 * WS ? 0 : wc + WS;                                                                             \
  wait_for<LATER, 0>();                                                                                        \
  __builtin_amdgcn_s_barrier();                                                                                \
  __builtin_amdgcn_sched_barrier(0);                                                                           \
  if constexpr (X) fetch_x(s + XN, xfree);                                                                     \
  TS_READ(0, rd0)                                                                                              \
  TS_MULTIPLY(1)                                                                                               \
  TS_DEAL(X ? NX : 0)
    TS_READ(0, rd0)
    int s = 0;
    for (; s < steps - XN; ++s) { TS_STEP(true, true, NW + NX * (XN - 2)) }
    if constexpr (XN == 3) {
      TS_STEP(true, false, NW + NX)
      ++s;
    }
    { TS_STEP(false, false, 0) }
    TS_READ(1, rd1)
    TS_MULTIPLY(0)
    TS_MULTIPLY(1)
#undef TS_READ
#undef TS_MULTIPLY
#undef TS_DEAL
#undef TS_STEP
  }
};
