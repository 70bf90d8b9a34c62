// y[M, N] = x[M, K] · W[N, K]^T in bfloat16 for many rows of x and a long reduction, which is cut into slices so that few
// tiles of y still occupy the chip: a workgroup adds up one slice of one tile, in 32 bits, and a second kernel adds the slices'
// parts, the first slice first, and stores them, or takes them through the residual sum and the norm that follow.
//
// What bounds it: W's way from memory and the parts' (slices M N of 32 bits, written once and read once), between a launch
// and a workgroup's first loads; from about 500 rows on the matrix cores and the path from the second level cache into
// LDS, which brings a tile of 128 x 128 its operands in the time its products take. A product of 2,048 columns is 16 to 32 such
// tiles at 160 to 256 rows: with the whole reduction in one workgroup (as the vendor library's kernels have it) most of the chip
// reads nothing. Measured with W coming from memory, N 2,048, K 8,192, against the library's product, without the second
// kernel: 160 rows 14.4 µs (26.8), 256 rows 16.3 (27.5), 512 rows 23.0 (34.0), 1,024 rows 34.5 (51.1), 2,048 rows 61.5
// (75.1); K 2,048: 256 rows 7.6 (12.4), 512 rows 10.4 (13.2).
//
// The tile itself is tile_product.h's. A workgroup computes one and ends. Tiles that share a slice of W run on one die.
#include "tile_product.h"

#define GS_THREADS 256
#define GS_HELD 4               // 8-column pieces of a row that a thread of the norm's kernel keeps

struct SlicesArgs {
  float* parts;                 // [slices][M][N]
  const bf16_t *x, *w;
  int M, N, steps, slices, row_tiles, col_tiles, items, per_die;
  int64_t ldx, ldw;
};

template <int BM, int BN, int WM, int WN, int XN>
__global__ __launch_bounds__(WM * WN * TS_WAVE, 2) void gemm_slices_kernel(const SlicesArgs a) {
  using Tile = TileProduct<BM, BN, WM, WN, XN>;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[Tile::LDS];
  // consecutive workgroups go to different dies: a die takes a run of tiles, those of one slice of W's rows side by side
  const int item = blockIdx.x % 8 * a.per_die + blockIdx.x / 8;
  if (item >= a.items) return;
  const int m0 = item % a.row_tiles * BM, c0 = item / a.row_tiles % a.col_tiles * BN, slice = item / (a.row_tiles * a.col_tiles);
  const int base = a.steps / a.slices, longer = a.steps % a.slices;      // (the first slices take a step more where they are uneven)
  const int64_t k0 = 64 * ((int64_t)slice * base + min(slice, longer));
  uint32_t xoff[Tile::NX], woff[Tile::NW];
#pragma unroll
  for (int q = 0; q < Tile::NX; ++q) {
    const int at = Tile::x_row(q);
    xoff[q] = (uint32_t)(min(at, a.M - 1 - m0) * a.ldx * 2) + Tile::piece(at);      // (rows past the end: the last one again)
  }
#pragma unroll
  for (int q = 0; q < Tile::NW; ++q) {
    const int at = Tile::w_row(q);
    woff[q] = (uint32_t)(min(at, a.N - 1 - c0) * a.ldw * 2) + Tile::piece(at);
  }
  float4_t acc[Tile::TN][Tile::TM];
  Tile::run(lds, load_base(a.x + (int64_t)m0 * a.ldx + k0), load_base(a.w + (int64_t)c0 * a.ldw + k0), xoff, woff, base + (slice < longer ? 1 : 0), acc);
  const int lane = threadIdx.x % TS_WAVE, r = lane % 16, g = lane / 16, wm = wave_index() % WM, wn = wave_index() / WM;
  float* y = a.parts + (int64_t)slice * a.M * a.N;
#pragma unroll
  for (int i = 0; i < Tile::TM; ++i) {
    const int m = m0 + (wm * Tile::TM + i) * 16 + r;
#pragma unroll
    for (int j = 0; j < Tile::TN; ++j) {
      const int c = c0 + (wn * Tile::TN + j) * 16 + 4 * g;
      if (m < a.M && c < a.N) *(float4_t*)(y + (int64_t)m * a.N + c) = acc[j][i];
    }
  }
}

// ---- what finishes it ----

// Four neighbouring sums, the first slice's first; four slices are asked for together.
static __device__ __forceinline__ float4_t slices_sum(const float* __restrict__ parts, int64_t at, int64_t size, int slices) {
  float4_t sum;
  for (int s0 = 0; s0 < slices; s0 += 4) {
    float4_t p[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) p[j] = *(const float4_t*)(parts + min(s0 + j, slices - 1) * size + at);
#pragma unroll
    for (int j = 0; j < 4; ++j) sum = s0 + j == 0 ? p[0] : s0 + j < slices ? sum + p[j] : sum;      // (not 0 + p: a sum of -0 stays -0)
  }
  return sum;
}

template <bool WIDE>
__global__ void __launch_bounds__(GS_THREADS) slices_finish_kernel(void* __restrict__ y, const float* __restrict__ parts, int64_t size, int slices) {
  const int64_t at = 4 * ((int64_t)blockIdx.x * GS_THREADS + threadIdx.x);
  if (at >= size) return;
  const float4_t v = slices_sum(parts, at, size, slices);
  if constexpr (WIDE) *(float4_t*)((float*)y + at) = v;
  else *(uint2*)((bf16_t*)y + at) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
}

// A workgroup a row: t = T(product) + residual, its norm and the sum, rounded as the product stored and `rmsnorm` of it are,
// in the order of that kernel's sums.
__global__ void __launch_bounds__(GS_THREADS)
slices_norm_kernel(bf16_t* __restrict__ out, bf16_t* __restrict__ sum_out, const float* __restrict__ parts, const bf16_t* __restrict__ res,
                   const bf16_t* __restrict__ w, int64_t size, int slices, int width, float eps) {
  __shared__ float partial[GS_THREADS / TS_WAVE];
  const int64_t row = (int64_t)blockIdx.x * width;
  float v[GS_HELD][8];
  uint4 rraw[GS_HELD], wraw[GS_HELD];
#pragma unroll
  for (int c = 0; c < GS_HELD; ++c) {
    const int n = 8 * (threadIdx.x + c * GS_THREADS);
    if (n < width) {
      wraw[c] = *(const uint4*)(w + n);
      rraw[c] = res ? *(const uint4*)(res + row + n) : make_uint4(0, 0, 0, 0);
      const float4_t a = slices_sum(parts, row + n, size, slices), b = slices_sum(parts, row + n + 4, size, slices);
#pragma unroll
      for (int k = 0; k < 4; ++k) v[c][k] = a[k], v[c][4 + k] = b[k];
    }
  }
  float acc = 0.f;
#pragma unroll
  for (int c = 0; c < GS_HELD; ++c)
    if (8 * (threadIdx.x + c * GS_THREADS) < width) {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint32_t word = (&rraw[c].x)[k >> 1];
        v[c][k] = bf2f(f2bf(v[c][k]));
        if (res) v[c][k] += __uint_as_float(k & 1 ? word & 0xffff0000u : word << 16);
        acc = fmaf(v[c][k], v[c][k], acc);
      }
    }
  acc = wave_sum(acc);
  if ((threadIdx.x & (TS_WAVE - 1)) == 0) partial[threadIdx.x / TS_WAVE] = acc;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int i = 0; i < GS_THREADS / TS_WAVE; ++i) total += partial[i];
  const float inv = 1.0f / sqrtf(total / (float)width + eps);
#pragma unroll
  for (int c = 0; c < GS_HELD; ++c) {
    const int n = 8 * (threadIdx.x + c * GS_THREADS);
    if (n < width) {
      uint32_t s[4], o[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float w0 = __uint_as_float((&wraw[c].x)[k] << 16), w1 = __uint_as_float((&wraw[c].x)[k] & 0xffff0000u);
        s[k] = (uint32_t)f2bf(v[c][2 * k]) | ((uint32_t)f2bf(v[c][2 * k + 1]) << 16);
        o[k] = (uint32_t)f2bf(bf2f(f2bf(v[c][2 * k] * inv)) * w0) | ((uint32_t)f2bf(bf2f(f2bf(v[c][2 * k + 1] * inv)) * w1) << 16);
      }
      *(uint4*)(sum_out + row + n) = make_uint4(s[0], s[1], s[2], s[3]);
      *(uint4*)(out + row + n) = make_uint4(o[0], o[1], o[2], o[3]);
    }
  }
}

template <int BM, int BN, int WM, int WN, int XN>
static int launch_slices(SlicesArgs a, hipStream_t stream) {
  a.row_tiles = (a.M + BM - 1) / BM, a.col_tiles = (a.N + BN - 1) / BN;
  const int64_t items = (int64_t)a.row_tiles * a.col_tiles * a.slices;
  if (items > (1 << 24)) return TS_TOO_LARGE;
  a.items = (int)items, a.per_die = (a.items + 7) / 8;
  gemm_slices_kernel<BM, BN, WM, WN, XN><<<8 * a.per_die, WM * WN * TS_WAVE, 0, stream>>>(a);
  return ts_check_launch();
}

// The slices' parts of a product.
static int slices_parts(float* parts, const void* x, const void* w, int M, int N, int K, int64_t ldx, int64_t ldw, int tile, int slices, hipStream_t stream) {
  if (K <= 0 || K % 64 || N % 8 || ldx < K || ldw < K || ldx % 8 || ldw % 8 || tile < 0 || tile > 4 || slices < 1 || slices > 64 || K / 64 / slices < TileProduct<64, 128, 1, 4, 3>::MIN_STEPS) return TS_BAD_SHAPE;
  if (!x || !w || !parts || (((uintptr_t)x | (uintptr_t)w | (uintptr_t)parts) & 15)) return TS_BAD_SHAPE;
  if ((int64_t)M * N >= (1ll << 40) || 256 * ldx * 2 >= (1ll << 31) || 256 * ldw * 2 >= (1ll << 31)) return TS_TOO_LARGE;      // (byte offsets from a tile's start)
  const SlicesArgs a = {parts, (const bf16_t*)x, (const bf16_t*)w, M, N, K / 64, slices, 0, 0, 0, 0, ldx, ldw};
  auto narrow = [&](int bm) {
    const int64_t rows = (int64_t)((M + bm - 1) / bm) * slices;
    return tiles_go_narrow(rows * ((N + 255) / 256), rows * ((N + 191) / 192), bm);
  };
  switch (tile) {
    case 0: return launch_slices<128, 128, 2, 2, 2>(a, stream);
    case 1: return narrow(128) ? launch_slices<128, 192, 4, 2, 2>(a, stream) : launch_slices<128, 256, 2, 4, 2>(a, stream);
    case 2: return narrow(192) ? launch_slices<192, 192, 4, 2, 2>(a, stream) : launch_slices<192, 256, 2, 4, 2>(a, stream);
    case 3: return narrow(256) ? launch_slices<256, 192, 4, 2, 2>(a, stream) : launch_slices<256, 256, 2, 4, 2>(a, stream);
    default: return launch_slices<64, 128, 1, 4, 3>(a, stream);
  }
}

template <bool WIDE> static int slices_finish(void* y, const void* parts, int64_t size, int slices, hipStream_t stream) {
  slices_finish_kernel<WIDE><<<(unsigned)((size / 4 + GS_THREADS - 1) / GS_THREADS), GS_THREADS, 0, stream>>>(y, (const float*)parts, size, slices);
  return ts_check_launch();
}

// x [M, K] and w [N, K] bfloat16, 16-byte aligned, rows ldx and ldw elements apart (multiples of 8); K a multiple of 64 with at
// least 3 steps of 64 a slice, N a multiple of 8. parts: float32 [slices][M][N], scratch that the call fills and reads. tile (rows of x by
// rows of W of a workgroup): 0 128 x 128, 1 128 x 256, 2 192 x 256, 3 256 x 256, 4 64 x 128; 192 columns
// for 256 by `tiles_go_narrow`. y [M, N] contiguous, 32-bit or bfloat16; or, with
// norm_w [N]: y the norm of (the product in bfloat16 plus res [M, N], which may be null), sum [M, N] that sum; N at most 8,192. One slice without
// a norm needs no parts (null): its workgroups store y themselves (gemm_whole.hip).
extern "C" int ts_gemm_slices_bf16(void* y, void* sum, void* parts, const void* x, const void* w, int M, int N, int K, int64_t ldx, int64_t ldw,
                                   int tile, int slices, int out_f32, const void* res, const void* norm_w, float eps, hipStream_t stream) {
  if (M <= 0 || N <= 0) return TS_OK;
  if (slices == 1 && !norm_w) return ts_gemm_whole_bf16(1, &y, &x, &w, &N, M, K, ldx, ldw, tile, 0, out_f32, stream);
  if (!y || ((uintptr_t)y & 15)) return TS_BAD_SHAPE;
  if (norm_w && (out_f32 || !sum || N > 8 * GS_THREADS * GS_HELD || (((uintptr_t)sum | (uintptr_t)res | (uintptr_t)norm_w) & 15))) return TS_BAD_SHAPE;
  const int rc = slices_parts((float*)parts, x, w, M, N, K, ldx, ldw, tile, slices, stream);
  if (rc != TS_OK) return rc;
  const int64_t size = (int64_t)M * N;
  if (out_f32 && !norm_w) return slices_finish<true>(y, parts, size, slices, stream);
  if (!norm_w) return slices_finish<false>(y, parts, size, slices, stream);
  slices_norm_kernel<<<M, GS_THREADS, 0, stream>>>((bf16_t*)y, (bf16_t*)sum, (const float*)parts, (const bf16_t*)res, (const bf16_t*)norm_w, size, slices, N, eps);
  return ts_check_launch();
}

// The parts alone, float32 [slices][M][N], for a kernel that adds them up where it takes the rows (residual_stream.hip).
extern "C" int ts_gemm_slices_parts_bf16(float* parts, const void* x, const void* w, int M, int N, int K, int64_t ldx, int64_t ldw, int tile, int slices,
                                         hipStream_t stream) {
  return M <= 0 || N <= 0 ? TS_OK : slices_parts(parts, x, w, M, N, K, ldx, ldw, tile, slices, stream);
}

// y: the sum of such parts of `size` numbers each (a multiple of 4), as ts_gemm_slices_bf16 stores it in 32 bits
extern "C" int ts_slices_sum(float* y, const float* parts, int64_t size, int slices, hipStream_t stream) {
  if (size <= 0) return TS_OK;
  if (!y || !parts || size % 4 || slices < 1 || (((uintptr_t)y | (uintptr_t)parts) & 15)) return TS_BAD_SHAPE;
  return slices_finish<true>(y, parts, size, slices, stream);
}
