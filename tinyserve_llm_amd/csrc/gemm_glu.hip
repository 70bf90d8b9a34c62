// y[M, F] = unit(x · Wg^T, x · Wu^T) for many rows of x in bfloat16: the gate|up product of a gated feed-forward with
// the unit on its way out, from the 32-bit sums in the matrix cores' registers. W holds F gate rows, then F up rows.
//
// What bounds it: the matrix cores, and next to them the memory path of a compute unit. The product alone runs at the
// vendor library's rate (2,048 rows, F 8,192, K 2,048: 1.2 to 1.3 PFLOP/s either way, at the clocks such products hold);
// what is gained is the trip of the product through memory and the launch that read it again. Measured with the weights
// coming from memory, against the library's product followed by the unit's kernel: 2,048 rows 120 µs against 134 (bfloat16
// product) and 171 (32-bit product: 125 with relu, 135 with the sigmoid), 999 rows 63 against 71, 512 rows 36 against 46,
// 160 rows 24 against 31.
//
// The tile is the one whose rounds of one workgroup a compute unit cost least (hip.glu_plan): a round of 256 x 256 is the chip's best
// rate, and other heights fill the last round where that one would not. F 8,192, weights from memory, in tiles of 256, 192 and
// 128 x 256: K 2,048, 700 rows 48.5, 43.7 and 57.5 µs, 1,514 rows 96.0, 81.7 and 87.7, 2,048 rows 104.8, 117.3 and 118.9; K 3,072,
// 1,514 rows 138, 117 and 135.
//
// A workgroup of 8 waves computes BM rows by BN rows of W (BN / 2 columns of the unit), 64 of K at a time. Slices of x
// and W go from memory straight into LDS, a kilobyte (8 rows of 128 bytes) an instruction; a row's eight 16-byte pieces
// are turned by (row / 2) % 8, which frees the operand reads of bank conflicts: a 16-byte read of a wave is served in four
// groups of 16 lanes (0-3, 12-15, 20-27; 4-11, 16-19, 28-31; and those 32 higher), 4 cycles without conflicts, 8 with the
// pieces as they stand or turned by row / 4. x has two steps in LDS and W three (W comes from memory, x from the second
// level cache): while a step is multiplied, the next step of x and the next two of W are under way, and the operands of
// the next half step are read while the matrix instructions of this one run; a step has one barrier, in its middle.
// Loads, reads and products are dealt out evenly in the code (all loads first made both waves of a SIMD wait at the
// memory path together: 1.46 against 1.40 µs a step with every compute unit busy). A workgroup takes several tiles in
// turn and fetches the next tile's first steps before it writes out the present one. The gate rows of a wave's columns
// and their up rows lie side by side in the tile, so that a gate and its up meet in one lane; two lanes exchange halves so
// that every store is 16 bytes (8-byte stores: 45 µs against 24 for the same product with K = 128).
#include "glu_unit.h"
#include "lds_loads.h"

// The unit's forms (glu_unit.h; the hardware's 2^x and reciprocal throughout would take 12 of 135 µs off the sigmoid form).
template <int ACT> static __device__ __forceinline__ float glu_unit(float g, float u, float limit, float slope, float up_shift) {
  if constexpr (ACT == GLU_SILU_ROUNDED) {          // both branches as a bfloat16 product leaves them
    const uint32_t both = pack_bf16(g, u);
    g = __uint_as_float(both << 16);
    return g * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-1.44269504088896340736f * g)) * __uint_as_float(both & 0xffff0000u);
  }
  return glu_capped(ACT, g, u, limit, slope, up_shift);
}

struct GluArgs {
  bf16_t* y;
  const bf16_t *x, *w;
  int M, F, K, row_tiles, col_tiles, per_die;
  int64_t ldx, ldw, ldy;
  float limit, slope, up_shift;
};

template <int BM, int BN, int WM, int WN, int ACT>
__global__ __launch_bounds__(WM * WN * TS_WAVE, 2) void gemm_glu_kernel(const GluArgs a) {
  constexpr int WAVES = WM * WN, TM = BM / WM / 16, TN = BN / WN / 16, TO = TN / 2, HALF = BN / WN / 2;
  constexpr int NX = BM / 8 / WAVES, NW = BN / 8 / WAVES;      // kilobytes of a step that a wave fetches
  constexpr int XS = BM * 128, WS = BN * 128;                  // bytes of a step of x and of W
  static_assert(BM % (8 * WAVES) == 0 && BN % (8 * WAVES) == 0 && TN % 2 == 0, "whole kilobytes a wave, gate and up in one wave");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * XS + 3 * WS];
  const int lane = threadIdx.x % TS_WAVE, r = lane % 16, g = lane / 16;
  const int wave = wave_index(), wm = wave % WM, wn = wave / WM;
  // consecutive workgroups go to different dies: a die takes a contiguous run of tiles, column tile by column tile, so
  // that the tiles sharing a slice of W run on the die whose second-level cache holds it
  const int die = blockIdx.x % 8, first = blockIdx.x / 8, stride = gridDim.x / 8;
  const int turns = min(a.per_die, a.row_tiles * a.col_tiles - die * a.per_die);
  if (first >= turns) return;
  const int steps = a.K / 64;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)lds;

  // ---- the loading side: where the next step of x and of W comes from and goes to ----
  uint32_t xoff[NX], woff[NW];
  __amdgpu_buffer_rsrc_t rsrc_x, rsrc_w;
  auto aim_x = [&](int turn) {
    const int m0 = (die * a.per_die + turn) % a.row_tiles * BM;
    rsrc_x = load_base(a.x + (int64_t)m0 * a.ldx);
#pragma unroll
    for (int q = 0; q < NX; ++q) {
      const int at = (wave * NX + q) * 8 + lane / 8;
      xoff[q] = (uint32_t)(min(at, a.M - 1 - m0) * a.ldx * 2) + ((lane % 8) ^ ((at >> 1) & 7)) * 16;      // (rows past the end: the last one again)
    }
  };
  auto aim_w = [&](int turn) {
    const int c0 = (die * a.per_die + turn) / a.row_tiles * (BN / 2);
    rsrc_w = load_base(a.w + (int64_t)c0 * a.ldw);
#pragma unroll
    for (int q = 0; q < NW; ++q) {
      const int at = (wave * NW + q) * 8 + lane / 8, in = at % (2 * HALF);
      const int row = min(at / (2 * HALF) * HALF + in % HALF, a.F - 1 - c0) + (in >= HALF ? a.F : 0);
      woff[q] = (uint32_t)(row * a.ldw * 2) + ((lane % 8) ^ ((at >> 1) & 7)) * 16;
    }
  };
  int xturn = first, xk = 0, wturn = first, wk = 0;
  const uint32_t xfirst = lds0 + wave * NX * 1024, wfirst = lds0 + 2 * XS + wave * NW * 1024;
  uint32_t xslot = xfirst, wslot = wfirst;
  auto fetch_x = [&]() {
#pragma unroll
    for (int q = 0; q < NX; ++q) load_to_lds(rsrc_x, xslot + q * 1024, xoff[q], (uint32_t)xk * 128);
  };
  auto fetch_w = [&]() {
#pragma unroll
    for (int q = 0; q < NW; ++q) load_to_lds(rsrc_w, wslot + q * 1024, woff[q], (uint32_t)wk * 128);
  };
  // (after a workgroup's last step the last tile's first steps are fetched again: a few loads, in bounds and never read)
  auto next_x = [&]() {
    xslot = xslot == xfirst ? xfirst + XS : xfirst;
    if (++xk == steps) {
      xk = 0;
      if (xturn + stride < turns) aim_x(xturn += stride);
    }
  };
  auto next_w = [&]() {
    wslot = wslot == wfirst + 2 * WS ? wfirst : wslot + WS;
    if (++wk == steps) {
      wk = 0;
      if (wturn + stride < turns) aim_w(wturn += stride);
    }
  };

  // ---- the multiplying side ----
  const uint32_t rd0 = (uint32_t)(r * 128 + (g ^ (r >> 1)) * 16), rd1 = rd0 ^ 64;      // a step's two halves of K
  const unsigned char* rx = lds + wm * TM * 2048;
  const unsigned char* rw = lds + 2 * XS + wn * TN * 2048;
  uint32_t xc = 0, wc = 0;
  u32x4_t fw[2][TN], fx[2][TM];
  float4_t acc[TN][TM];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i) acc[j][i] = (float4_t){0.f, 0.f, 0.f, 0.f};
  aim_x(first);
  aim_w(first);
  fetch_x(), next_x();
  fetch_w(), next_w();
  fetch_w(), next_w();
  fetch_x(), next_x();
  wait_for<NW + NX>();
  __builtin_amdgcn_s_barrier();
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
    if ((q + 1) * LOADS / (TM * TN) > q * LOADS / (TM * TN)) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0); \
  }                                                                                                            \
  __builtin_amdgcn_sched_barrier(0);
  TS_READ(0, rd0)
  for (int turn = first; turn < turns; turn += stride) {
    for (int s = 0; s < steps; ++s) {
      __builtin_amdgcn_sched_barrier(0);
      fetch_w();
      TS_READ(1, rd1)
      TS_MULTIPLY(0)
      TS_DEAL(NW)
      next_w();
      xc = XS - xc;
      wc = wc == 2 * WS ? 0 : wc + WS;
      // every wave has read the last of this step's x and of W (so their places may be filled), and the next step has
      // landed: x was asked for half a step later than W, so all but the newest NW loads are done
      wait_for<NW, 0>();
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      fetch_x();
      TS_READ(0, rd0)
      TS_MULTIPLY(1)
      TS_DEAL(NX)
      next_x();
    }
    const int item = die * a.per_die + turn;
    const int m0 = item % a.row_tiles * BM, c0 = item / a.row_tiles * (BN / 2) + wn * HALF;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = m0 + (wm * TM + i) * 16 + r;
      uint32_t p[TO][2];
#pragma unroll
      for (int j = 0; j < TO; ++j) {
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = glu_unit<ACT>(acc[j][i][e], acc[j + TO][i][e], a.limit, a.slope, a.up_shift);
        p[j][0] = pack_bf16(o[0], o[1]);
        p[j][1] = pack_bf16(o[2], o[3]);
      }
      bf16_t* row = a.y + (int64_t)m * a.ldy;
      // lane (r, g) holds columns 16 j + 4 g .. + 3 of row r: lanes g and g ^ 1 exchange so that each has eight in a row
#pragma unroll
      for (int j = 0; j + 1 < TO; j += 2) {
        const auto lo = __builtin_amdgcn_permlane16_swap(p[j][0], p[j + 1][0], false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap(p[j][1], p[j + 1][1], false, false);
        const int c = c0 + (j + (g & 1)) * 16 + (g >> 1) * 8;
        if (m < a.M && c < a.F) *(u32x4_t*)(row + c) = (u32x4_t){lo[0], hi[0], lo[1], hi[1]};
      }
      if constexpr (TO % 2) {
        const int c = c0 + (TO - 1) * 16 + 4 * g;
        if (m < a.M && c < a.F) *(uint2*)(row + c) = make_uint2(p[TO - 1][0], p[TO - 1][1]);
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[j][i] = (float4_t){0.f, 0.f, 0.f, 0.f};
    }
  }
#undef TS_READ
#undef TS_MULTIPLY
#undef TS_DEAL
  wait_for<0>();      // what was fetched beyond the end lands before the workgroup's LDS is another's
}

template <int BM, int BN, int WM, int WN>
static int launch_glu(GluArgs a, int act, hipStream_t stream) {
  a.row_tiles = (a.M + BM - 1) / BM, a.col_tiles = (a.F + BN / 2 - 1) / (BN / 2);
  a.per_die = (a.row_tiles * a.col_tiles + 7) / 8;
  const dim3 grid(8 * (a.per_die < 32 ? a.per_die : 32));
  switch (act) {
    case GLU_SILU_ROUNDED: gemm_glu_kernel<BM, BN, WM, WN, GLU_SILU_ROUNDED><<<grid, WM * WN * TS_WAVE, 0, stream>>>(a); break;
    case GLU_SIGMOID: gemm_glu_kernel<BM, BN, WM, WN, GLU_SIGMOID><<<grid, WM * WN * TS_WAVE, 0, stream>>>(a); break;
    case GLU_RELU: gemm_glu_kernel<BM, BN, WM, WN, GLU_RELU><<<grid, WM * WN * TS_WAVE, 0, stream>>>(a); break;
    default: gemm_glu_kernel<BM, BN, WM, WN, GLU_GELU><<<grid, WM * WN * TS_WAVE, 0, stream>>>(a);
  }
  return ts_check_launch();
}

// x [M, K], w [2 F, K], y [M, F] bfloat16, 16-byte aligned, rows ldx, ldw, ldy elements apart (multiples of 8); K a
// multiple of 64, F of 8. tile: rows of x by rows of W of a workgroup, 0 256 x 256, 1 192 x 256, 2 128 x 128,
// 3 128 x 256. act: 0 silu(gate) up with both branches rounded to bfloat16 first (limit, slope and up_shift
// unused); 1, 2, 3: the capped unit from the 32-bit sums with the gate through a sigmoid of slope, relu or gelu's tanh form.
extern "C" int ts_gemm_glu_bf16(void* y, const void* x, const void* w, int M, int F, int K, int64_t ldx, int64_t ldw, int64_t ldy,
                                int tile, int act, float limit, float slope, float up_shift, hipStream_t stream) {
  if (M <= 0 || F <= 0) return TS_OK;
  if (K <= 0 || K % 64 || F % 8 || ldx < K || ldw < K || ldy < F || ldx % 8 || ldw % 8 || ldy % 8 || act < 0 || act > 3 || tile < 0 || tile > 3) return TS_BAD_SHAPE;
  if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) & 15) return TS_BAD_SHAPE;
  if (!x || !w || !y || 2 * (int64_t)F * ldw * 2 >= (1ll << 31) || 256 * ldx * 2 >= (1ll << 31)) return TS_TOO_LARGE;   // (byte offsets from a tile's start)
  const GluArgs a = {(bf16_t*)y, (const bf16_t*)x, (const bf16_t*)w, M, F, K, 0, 0, 0, ldx, ldw, ldy, limit, slope, up_shift};
  switch (tile) {
    case 0: return launch_glu<256, 256, 2, 4>(a, act, stream);
    case 1: return launch_glu<192, 256, 2, 4>(a, act, stream);
    case 2: return launch_glu<128, 128, 2, 4>(a, act, stream);
    default: return launch_glu<128, 256, 2, 4>(a, act, stream);
  }
}
