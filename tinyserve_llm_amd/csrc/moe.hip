// A mixture of experts: every token goes through `top` of `experts` small gated feed-forward layers.
//   * `ts_moe_route`: router logits z = W_r h in 32-bit (h as it is stored), scores s = sigmoid(z); the `top`
//     experts with the largest s + correction are chosen (ties: the lower index); their weights are their s,
//     divided by the chosen ones' sum (+ 1e-20) if `normalize`, times `scale`. With `softmax_chosen` the logits
//     themselves are the scores, and the weights are the softmax over the chosen experts' logits alone. With
//     `scoring` 2 the scores are the softmax over all the router's outputs. The router may have `extras` more rows
//     than experts: their logits' sigmoids are left beside the choice (a gate on a shared expert, say). With `groups` the
//     experts form that many equal groups of neighbours, and only those of the `keep` groups whose best choice score is
//     largest can be chosen.
//   * `ts_moe_group`: the step's (token, choice) pairs grouped by expert, and the groups cut into tiles of rows
//     that one workgroup of the product takes: [expert, first index, rows] per tile, rows 0 for the tiles of the
//     launch that the step does not fill (the launch is sized for the worst case, so nothing comes back to the host).
//   * `ts_moe_gemm`: for every tile, rows of the operand (a token's row, or a pair's) times the tile's expert's
//     matrix; with `glu` the matrix holds gate rows, then up rows, and the capped gated unit
//     g = min(gate, L), u = clamp(up, -L, L), y = g sigmoid(slope g) (u + shift) leaves instead of the sums.
//     Without `glu`, `act` 1 squares the sums' positive parts on their way out (experts of the form W_down relu(W_up h)^2).
//     Every row's sums run over k in ascending order whatever the tile it lands in, in one stretch (tiles of 64 and 256 rows) or
//     four that are then added in order (16 rows; 128 where the reduction is 512 or more in multiples of 256): the same bits
//     within either kind, and 2.7e-7 and 1.3e-7 from 64 bits over 2,048.
//   * `ts_moe_combine`: out[token] = sum over its choices, in order, of weight * the pair's row (+ a shared
//     expert's row, times a gate per token if there is one). A choice at or beyond `real` is an identity expert: it
//     has no matrices, `ts_moe_group` leaves its pairs out of every tile, and its row is the token's input itself.
// float32 runs 32-bit multiply-adds; bfloat16 operands go through the matrix cores with 32-bit sums.
#include <type_traits>
#include "lds_loads.h"

#define MOE_THREADS 256
#define MOE_ROUTE_TOKENS 4
#define MOE_MAX_EXPERTS 1024
#define MOE_MAX_TOP 32

#define MOE_ROUTE_CHUNK 2048      // elements of a token's row that lie in LDS at a time
#define MOE_ROUTE_THREADS 1024    // sixteen waves: an expert each at a time, so that a step of few tokens has all its loads in flight at once

// BY4: the router's rows are read in 16-byte pieces (a width that is a multiple of 4, from an aligned start); other widths have a
// kernel of their own, whose loads the pieces' registers would hold up (64 tokens over 2,049, 18 rows: 13.4 µs, 16.7 in one kernel).
template <typename TX, bool BY4>
__global__ void __launch_bounds__(MOE_ROUTE_THREADS)
moe_route_kernel(int32_t* __restrict__ ids_out, float* __restrict__ w_out, const TX* __restrict__ x,
                 const float* __restrict__ router, const float* __restrict__ correction, int num_tokens, int K, int E, int top,
                 float scale, int normalize, int scoring, int extras, float* __restrict__ extra_out, int groups, int keep) {
  const bool softmax_chosen = scoring == 1;
  const int rows = E + extras;                            // rows of the router: the experts, then the extras
  extern __shared__ float lds[];
  float* s_s = lds;                                       // [MOE_ROUTE_TOKENS][rows] logits, then scores
  float* c_s = lds + MOE_ROUTE_TOKENS * rows;             // [MOE_ROUTE_TOKENS][rows] choice scores
  float* x_s = c_s + MOE_ROUTE_TOKENS * rows;                // [MOE_ROUTE_TOKENS][MOE_ROUTE_CHUNK] the tokens' rows, 32-bit
  const int wave = threadIdx.x / TS_WAVE, lane = threadIdx.x & (TS_WAVE - 1);
  const int t0 = blockIdx.x * MOE_ROUTE_TOKENS;
  const int nt = min(MOE_ROUTE_TOKENS, num_tokens - t0);
  for (int i = threadIdx.x; i < MOE_ROUTE_TOKENS * rows; i += MOE_ROUTE_THREADS) s_s[i] = 0.f;
  constexpr int PER = 16 / sizeof(TX);                              // elements of a 16-byte piece of x
  const bool whole = K % PER == 0 && ((uintptr_t)x & 15) == 0;
  // A stretch of the rows into LDS, then every wave takes experts in turn: a lane reads the router's row side by
  // side with its neighbours, all of a stretch's pieces asked for before the first is used. A step of few tokens is bound
  // by the chain of these trips: a wave's first row of the router is on its way while the tokens' rows are, and each
  // further one while the sums of the one before go through the wave (48 tokens over 2,048, 18 rows: 12.0 -> 9.5 µs; 2,048 tokens 22.0 -> 19.2).
  constexpr int PIECES = BY4 ? MOE_ROUTE_CHUNK / (4 * TS_WAVE) : 1;
  float4 w[PIECES];
  for (int k0 = 0; k0 < K; k0 += MOE_ROUTE_CHUNK) {
    const int kn = min(MOE_ROUTE_CHUNK, K - k0);
    const auto ask = [&](int e) {
      if (!BY4 || e >= rows) return;
#pragma unroll
      for (int i = 0; i < PIECES; ++i) {
        const int k = 4 * (lane + TS_WAVE * i);
        w[i] = k < kn ? *(const float4*)(router + (int64_t)e * K + k0 + k) : make_float4(0.f, 0.f, 0.f, 0.f);
      }
    };
    ask(wave);
    __syncthreads();
    if (whole) {
      const int pieces = kn / PER;
      for (int i = threadIdx.x; i < MOE_ROUTE_TOKENS * pieces; i += MOE_ROUTE_THREADS) {
        const int r = i / pieces, k = (i - r * pieces) * PER;
        float* to = x_s + r * MOE_ROUTE_CHUNK + k;
        uint4 v = make_uint4(0, 0, 0, 0);
        if (r < nt) v = *(const uint4*)(x + (int64_t)(t0 + r) * K + k0 + k);
        if constexpr (PER == 4) {
          *(uint4*)to = v;
        } else {
          *(uint4*)to = make_uint4(v.x << 16, v.x & 0xffff0000u, v.y << 16, v.y & 0xffff0000u);
          *(uint4*)(to + 4) = make_uint4(v.z << 16, v.z & 0xffff0000u, v.w << 16, v.w & 0xffff0000u);
        }
      }
    } else {
#pragma unroll 8
      for (int i = threadIdx.x; i < MOE_ROUTE_TOKENS * kn; i += MOE_ROUTE_THREADS) {
        const int r = i / kn, k = i - r * kn;
        x_s[r * MOE_ROUTE_CHUNK + k] = r < nt ? Num<TX>::ld(x + (int64_t)(t0 + r) * K + k0 + k) : 0.f;
      }
    }
    __syncthreads();
    for (int e = wave; e < rows; e += MOE_ROUTE_THREADS / TS_WAVE) {
      float acc[MOE_ROUTE_TOKENS];
#pragma unroll
      for (int r = 0; r < MOE_ROUTE_TOKENS; ++r) acc[r] = 0.f;
      if constexpr (BY4) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
          const int k = 4 * (lane + TS_WAVE * i);
          if (k >= kn) continue;
#pragma unroll
          for (int r = 0; r < MOE_ROUTE_TOKENS; ++r) {
            const float4 xv = *(const float4*)(x_s + r * MOE_ROUTE_CHUNK + k);
            acc[r] = fmaf(w[i].x, xv.x, fmaf(w[i].y, xv.y, fmaf(w[i].z, xv.z, fmaf(w[i].w, xv.w, acc[r]))));
          }
        }
        ask(e + MOE_ROUTE_THREADS / TS_WAVE);
      } else {
        const float* wr = router + (int64_t)e * K + k0;
#pragma unroll 8
        for (int k = lane; k < kn; k += TS_WAVE) {
          const float wk = wr[k];
#pragma unroll
          for (int r = 0; r < MOE_ROUTE_TOKENS; ++r) acc[r] = fmaf(wk, x_s[r * MOE_ROUTE_CHUNK + k], acc[r]);
        }
      }
#pragma unroll
      for (int r = 0; r < MOE_ROUTE_TOKENS; ++r) acc[r] = wave_sum(acc[r]);
#pragma unroll
      for (int r = 0; r < MOE_ROUTE_TOKENS; ++r)
        if (lane == 0) s_s[r * rows + e] += acc[r];             // (an expert is one wave's: no other adds to it)
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < MOE_ROUTE_TOKENS * rows; i += MOE_ROUTE_THREADS) {
    const int e = i % rows;
    const float sc = (softmax_chosen || (scoring == 2 && e < E)) ? s_s[i] : 1.0f / (1.0f + expf(-s_s[i]));
    s_s[i] = sc;
    c_s[i] = sc + ((correction && e < E) ? correction[e] : 0.f);
  }
  __syncthreads();
  if (wave >= nt) return;                                 // a wave per token from here on
  const int r = wave, t = t0 + wave;
  s_s += r * rows;
  c_s += r * rows;
  if (extras && lane < extras) extra_out[(int64_t)t * extras + lane] = s_s[E + lane];
  if (scoring == 2) {                                     // the softmax over all the experts' logits
    float top_logit = -INFINITY;
    for (int e = lane; e < E; e += TS_WAVE) top_logit = fmaxf(top_logit, s_s[e]);
    top_logit = wave_max(top_logit);
    float total = 0.f;
    for (int e = lane; e < E; e += TS_WAVE) total += expf(s_s[e] - top_logit);
    total = wave_sum(total);
    wave_sync();
    for (int e = lane; e < E; e += TS_WAVE) {
      const float sc = expf(s_s[e] - top_logit) / total;
      s_s[e] = sc;
      c_s[e] = sc + (correction ? correction[e] : 0.f);
    }
    wave_sync();
  }
  if (groups > 1 && keep < groups) {
    // lane g scores group g (groups <= 64); a group stays if fewer than `keep` beat it (ties: the lower group)
    const int size = E / groups;
    float best = -INFINITY;
    if (lane < groups)
      for (int e = lane * size; e < (lane + 1) * size; ++e) best = fmaxf(best, c_s[e]);
    int ahead = 0;
    for (int g = 0; g < groups; ++g) {
      const float other = __shfl(best, g, TS_WAVE);
      ahead += other > best || (other == best && g < lane);
    }
    wave_sync();
    if (lane < groups && ahead >= keep)
      for (int e = lane * size; e < (lane + 1) * size; ++e) c_s[e] = -INFINITY;
    wave_sync();
  }
  // lane j keeps the j-th choice (top <= 32 lanes of the 64)
  float my_pick = 0.f;
  int my_choice = 0;
  for (int j = 0; j < top; ++j) {
    float best = -INFINITY;
    int at = 0x7fffffff;
    for (int e = lane; e < E; e += TS_WAVE) {
      const float c = c_s[e];
      if (c > best) { best = c; at = e; }                 // (ascending e: the lower index wins a tie)
    }
#pragma unroll
    for (int off = TS_WAVE / 2; off > 0; off >>= 1) {
      const float ob = __shfl_xor(best, off, TS_WAVE);
      const int oa = __shfl_xor(at, off, TS_WAVE);
      if (ob > best || (ob == best && oa < at)) { best = ob; at = oa; }
    }
    if (at >= E) at = j;                                  // (scores that are no numbers: still valid indices)
    if (lane == j) { my_choice = at; my_pick = s_s[at]; }
    wave_sync();
    if (lane == 0) c_s[at] = -INFINITY;
    wave_sync();
  }
  if (softmax_chosen) {                                   // the chosen logits' softmax: the first choice is the largest
    const float top_logit = __shfl(my_pick, 0, TS_WAVE);
    my_pick = lane < top ? expf(my_pick - top_logit) : 0.f;
  }
  const float total = wave_sum(my_pick);                  // (the lanes beyond `top` hold 0)
  const float mult = (softmax_chosen ? 1.0f / total : normalize ? 1.0f / (total + 1e-20f) : 1.0f) * scale;
  if (lane < top) {
    ids_out[(int64_t)t * top + lane] = my_choice;
    w_out[(int64_t)t * top + lane] = my_pick * mult;
  }
}

extern "C" int ts_moe_route(int32_t* ids_out, float* w_out, const void* x, int x_dtype, const float* router,
                            const float* correction, int num_tokens, int K, int E, int top, float scale, int normalize,
                            int scoring, int extras, float* extra_out, int groups, int keep, hipStream_t stream) {
  if (num_tokens <= 0) return TS_OK;
  if (K <= 0 || E <= 0 || E > MOE_MAX_EXPERTS || top <= 0 || top > MOE_MAX_TOP || top > E || scoring < 0 || scoring > 2 ||
      extras < 0 || extras > TS_WAVE || (extras && !extra_out) || groups < 1 || groups > TS_WAVE || E % groups || keep < 1 ||
      keep > groups || top > keep * (E / groups))
    return TS_BAD_SHAPE;
  const unsigned blocks = (num_tokens + MOE_ROUTE_TOKENS - 1) / MOE_ROUTE_TOKENS;
  const size_t lds = (size_t)MOE_ROUTE_TOKENS * (2 * (E + extras) + MOE_ROUTE_CHUNK) * sizeof(float);
  const bool by4 = K % 4 == 0 && ((uintptr_t)router & 15) == 0;
#define MOE_ROUTE(TX, BY4) \
  moe_route_kernel<TX, BY4><<<blocks, MOE_ROUTE_THREADS, lds, stream>>>(ids_out, w_out, (const TX*)x, router, correction, num_tokens, K, E, top, \
                                                                        scale, normalize, scoring, extras, extra_out, groups, keep)
  if (x_dtype == 0 && by4) MOE_ROUTE(float, true);
  else if (x_dtype == 0) MOE_ROUTE(float, false);
  else if (x_dtype == 1 && by4) MOE_ROUTE(bf16_t, true);
  else if (x_dtype == 1) MOE_ROUTE(bf16_t, false);
  else return TS_BAD_DTYPE;
#undef MOE_ROUTE
  return ts_check_launch();
}

// One workgroup: counts per expert, their running sums, the tiles, then every pair into its expert's stretch.
#define MOE_GROUP_THREADS 1024
__global__ void __launch_bounds__(MOE_GROUP_THREADS)
moe_group_kernel(const int32_t* __restrict__ ids, int32_t* __restrict__ sorted, int32_t* __restrict__ tiles, int P, int E,
                 int tile_rows, int max_tiles) {
  __shared__ int count_s[MOE_MAX_EXPERTS];
  __shared__ int first_s[MOE_MAX_EXPERTS + 1];
  __shared__ int tile_s[MOE_MAX_EXPERTS + 1];
  for (int e = threadIdx.x; e < E; e += MOE_GROUP_THREADS) count_s[e] = 0;
  __syncthreads();
  for (int p = threadIdx.x; p < P; p += MOE_GROUP_THREADS)
    if (ids[p] < E) atomicAdd(&count_s[ids[p]], 1);          // (a choice beyond the experts with matrices: an identity expert, in no tile)
  __syncthreads();
  if (threadIdx.x == 0) {
    int first = 0, tile = 0;
    for (int e = 0; e < E; ++e) {
      first_s[e] = first;
      tile_s[e] = tile;
      first += count_s[e];
      tile += (count_s[e] + tile_rows - 1) / tile_rows;
    }
    first_s[E] = first;
    tile_s[E] = tile;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += MOE_GROUP_THREADS) {
    const int n = count_s[e];
    for (int i = 0, tile = tile_s[e]; i < n && tile < max_tiles; i += tile_rows, ++tile) {
      tiles[3 * tile] = e;
      tiles[3 * tile + 1] = first_s[e] + i;
      tiles[3 * tile + 2] = min(tile_rows, n - i);
    }
  }
  for (int tile = tile_s[E] + threadIdx.x; tile < max_tiles; tile += MOE_GROUP_THREADS) {
    tiles[3 * tile] = 0;
    tiles[3 * tile + 1] = 0;
    tiles[3 * tile + 2] = 0;
  }
  // every pair into its expert's stretch, in the order the threads come by (a row's sums do not depend on its
  // place in a tile, so the order inside an expert changes no result)
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += MOE_GROUP_THREADS) count_s[e] = 0;
  __syncthreads();
  for (int p = threadIdx.x; p < P; p += MOE_GROUP_THREADS) {
    const int e = ids[p];
    if (e < E) sorted[first_s[e] + atomicAdd(&count_s[e], 1)] = p;
  }
}

extern "C" int ts_moe_group(const int32_t* ids, int32_t* sorted, int32_t* tiles, int P, int E, int tile_rows, int max_tiles,
                            hipStream_t stream) {
  if (P <= 0) return TS_OK;
  // (tiles of a step: at most P / tile_rows full ones and one partly filled per expert that has pairs)
  if (E <= 0 || E > MOE_MAX_EXPERTS || tile_rows <= 0 || max_tiles < P / tile_rows + (E < P ? E : P)) return TS_BAD_SHAPE;
  moe_group_kernel<<<1, MOE_GROUP_THREADS, 0, stream>>>(ids, sorted, tiles, P, E, tile_rows, max_tiles);
  return ts_check_launch();
}

#define MOE_BM 16
#define MOE_DIES 8
#define MOE_BN 64
#define MOE_KC 32

// What an ungated expert's sums pass on their way out: 0 nothing, 1 the square of relu.
static __device__ __forceinline__ float moe_act(float s, int act) {
  if (act == 1) { const float r = fmaxf(s, 0.f); return r * r; }
  return s;
}

static __device__ __forceinline__ float moe_unit(float g, float u, float limit, float slope, float shift) {
  if (limit > 0.f) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
  }
  return g / (1.0f + expf(-slope * g)) * (u + shift);
}

// Plain 32-bit multiply-adds: a tile of up to 16 rows by 64 columns a workgroup; thread (column, row quarter).
template <typename TX, typename TO>
__global__ void __launch_bounds__(MOE_THREADS)
moe_gemm_kernel(TO* __restrict__ out, const TX* __restrict__ x, const TX* __restrict__ w, const int32_t* __restrict__ sorted,
                const int32_t* __restrict__ tiles, int src_div, int N, int K, int glu, float limit, float slope, float shift, int act) {
  __shared__ float x_s[MOE_BM][MOE_KC + 1];
  __shared__ float w_s[2][MOE_BN][MOE_KC + 1];
  __shared__ int row_s[MOE_BM];
  const int tile = blockIdx.x;
  const int rows = tiles[3 * tile + 2];
  if (rows == 0) return;
  const int e = tiles[3 * tile], first = tiles[3 * tile + 1];
  const int n0 = blockIdx.y * MOE_BN;
  const int tx = threadIdx.x & (MOE_BN - 1), ty = threadIdx.x / MOE_BN;
  if (threadIdx.x < MOE_BM) row_s[threadIdx.x] = threadIdx.x < rows ? sorted[first + threadIdx.x] : -1;
  __syncthreads();
  const int64_t expert_rows = glu ? 2 * (int64_t)N : N;
  const TX* we = w + (int64_t)e * expert_rows * K;
  float acc[4] = {0.f, 0.f, 0.f, 0.f}, acc2[4] = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < K; k0 += MOE_KC) {
    for (int i = threadIdx.x; i < MOE_BM * MOE_KC; i += MOE_THREADS) {
      const int r = i / MOE_KC, kk = i - r * MOE_KC;
      const int p = row_s[r];
      x_s[r][kk] = (p >= 0 && k0 + kk < K) ? Num<TX>::ld(x + (int64_t)(p / src_div) * K + k0 + kk) : 0.f;
    }
    for (int i = threadIdx.x; i < MOE_BN * MOE_KC; i += MOE_THREADS) {
      const int c = i / MOE_KC, kk = i - c * MOE_KC;
      const bool in = n0 + c < N && k0 + kk < K;
      w_s[0][c][kk] = in ? Num<TX>::ld(we + (int64_t)(n0 + c) * K + k0 + kk) : 0.f;
      if (glu) w_s[1][c][kk] = in ? Num<TX>::ld(we + (int64_t)(N + n0 + c) * K + k0 + kk) : 0.f;
    }
    __syncthreads();
#pragma unroll 8
    for (int kk = 0; kk < MOE_KC; ++kk) {
      const float wv = w_s[0][tx][kk];
      const float wu = glu ? w_s[1][tx][kk] : 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float xv = x_s[ty * 4 + r][kk];
        acc[r] = fmaf(xv, wv, acc[r]);
        acc2[r] = fmaf(xv, wu, acc2[r]);
      }
    }
    __syncthreads();
  }
  if (n0 + tx >= N) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int p = row_s[ty * 4 + r];
    if (p < 0) continue;
    const float y = glu ? moe_unit(acc[r], acc2[r], limit, slope, shift) : moe_act(acc[r], act);
    Num<TO>::st(out + (int64_t)p * N + n0 + tx, y);
  }
}

// bfloat16 on the matrix cores: a workgroup of four waves takes a tile's rows (TM blocks of 16) by 4 x TN x 16
// columns, each wave TN column blocks of all the rows. Operands go from memory straight into the instruction's
// registers: lane (r, g) holds eight consecutive k of row r of a block, 16 bytes, for the rows of x (gathered by
// pair) as for the rows of the expert's matrix. The product is formed as y^T = W x^T, which leaves a lane four
// consecutive columns of one row of y. With GLU a lane holds a gate sum and its up sum side by side and stores
// the unit. K is a multiple of 32; a tile's missing rows and a matrix's missing columns are computed on
// repeated rows and not stored.
typedef uint32_t moe_u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 moe_bf16x8 __attribute__((ext_vector_type(8)));
typedef float moe_f32x4 __attribute__((ext_vector_type(4)));

static __device__ __forceinline__ moe_f32x4 moe_mfma(moe_u32x4 a, moe_u32x4 b, moe_f32x4 acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(moe_bf16x8, a), __builtin_bit_cast(moe_bf16x8, b), acc, 0, 0, 0);
}

// Four adjacent columns of a row, `left` of which exist: one store where all do and the place is whole pieces.
static __device__ __forceinline__ void moe_store4(float* p, const float (&y)[4], int left) {
  if (left >= 4 && ((uintptr_t)p & 15) == 0) { *(float4*)p = make_float4(y[0], y[1], y[2], y[3]); return; }
  for (int c = 0; c < 4 && c < left; ++c) p[c] = y[c];
}
static __device__ __forceinline__ void moe_store4(bf16_t* p, const float (&y)[4], int left) {
  if (left >= 4 && ((uintptr_t)p & 7) == 0) {
    uint2 v;
    v.x = (uint32_t)f2bf(y[0]) | ((uint32_t)f2bf(y[1]) << 16);
    v.y = (uint32_t)f2bf(y[2]) | ((uint32_t)f2bf(y[3]) << 16);
    *(uint2*)p = v;
    return;
  }
  for (int c = 0; c < 4 && c < left; ++c) p[c] = f2bf(y[c]);
}

template <int TM, int TN, bool GLU, typename TO>
__global__ void __launch_bounds__(MOE_THREADS)
moe_gemm_mfma_kernel(TO* __restrict__ out, const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                     const int32_t* __restrict__ sorted, const int32_t* __restrict__ tiles, int parts, int src_div, int N, int K,
                     float limit, float slope, float shift, int act) {
  constexpr int SETS = GLU ? 2 : 1;
  const int tile = blockIdx.x / parts, at = blockIdx.x % parts * TM * 16;     // (wider tiles in parts of so many rows)
  const int rows = min(tiles[3 * tile + 2] - at, TM * 16);
  if (rows <= 0) return;
  const int e = tiles[3 * tile], first = tiles[3 * tile + 1] + at;
  const int wave = threadIdx.x / TS_WAVE, lane = threadIdx.x & (TS_WAVE - 1);
  const int r = lane & 15, g = lane >> 4;
  const int n0 = (blockIdx.y * 4 + wave) * TN * 16;
  if (n0 >= N) return;
  const int64_t expert_rows = GLU ? 2 * (int64_t)N : N;
  const bf16_t* we = w + (int64_t)e * expert_rows * K;
  int pair[TM];
  const bf16_t* xp[TM];
  const bf16_t* wp[SETS][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    pair[i] = sorted[first + min(16 * i + r, rows - 1)];
    xp[i] = x + (int64_t)(pair[i] / src_div) * K + 8 * g;
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int col = min(n0 + 16 * j + r, N - 1);
    wp[0][j] = we + (int64_t)col * K + 8 * g;
    if constexpr (GLU) wp[1][j] = we + (int64_t)(N + col) * K + 8 * g;
  }
  moe_f32x4 acc[SETS][TN][TM];
#pragma unroll
  for (int s = 0; s < SETS; ++s)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[s][j][i] = (moe_f32x4){0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < K; k0 += 32) {
    moe_u32x4 fx[TM], fw[SETS][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) fx[i] = *(const moe_u32x4*)(xp[i] + k0);
#pragma unroll
    for (int s = 0; s < SETS; ++s)
#pragma unroll
      for (int j = 0; j < TN; ++j) fw[s][j] = *(const moe_u32x4*)(wp[s][j] + k0);
#pragma unroll
    for (int s = 0; s < SETS; ++s)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i) acc[s][j][i] = moe_mfma(fw[s][j], fx[i], acc[s][j][i]);
  }
  // lane (r, g) of block (j, i): row 16 i + r of the tile, columns n0 + 16 j + 4 g .. + 3
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    if (16 * i + r >= rows) continue;
    TO* orow = out + (int64_t)pair[i] * N;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + 16 * j + 4 * g;
      float y[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if constexpr (GLU) y[c] = moe_unit(acc[0][j][i][c], acc[1][j][i][c], limit, slope, shift);
        else y[c] = moe_act(acc[0][j][i][c], act);
      }
      moe_store4(orow + col, y, N - col);
    }
  }
}

// Tiles of 16 rows, for steps of few tokens, where the experts' matrices are streamed once and nothing else counts, over reductions that are no multiple of 256 (the
// kernel below takes those; the figures here are from when this one took all):
// a workgroup takes a tile's rows by 16 columns (with GLU: 16 gate and 16 up columns), and its four waves take a
// quarter of K each, eight k-steps' loads in flight at a time, so that a step with one token still has a thousand
// waves asking for memory. A row's loads go out side by side (two take a cache line): the two products of 32 experts of 3,072 and 1,536 over four choices each took
// with four steps and each step's row and columns in turn 106 us with 8 tokens and 377 with 128, and take 96 and 322. ONCE: W goes by the caches, which leaves them to the
// weights of other layers (a decode step with two layers of 16 experts of 2,048 and 1,024 beside two without, 6 tokens 600 and 589 us, 16 669 and 647, 48 850 and 821) but asks for each
// line twice: by themselves the products above take 110 and 398 so. The quarters' sums meet through LDS and are added in the waves' order: a row's result
// depends on K alone, not on the tile or the batch it lands in.
template <bool GLU, typename TO, bool ONCE>
__global__ void __launch_bounds__(MOE_THREADS)
moe_gemm_stream_kernel(TO* __restrict__ out, const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                       const int32_t* __restrict__ sorted, const int32_t* __restrict__ tiles, int src_div, int N, int K,
                       float limit, float slope, float shift, int act) {
  constexpr int SETS = GLU ? 2 : 1;
  constexpr int WAVES = MOE_THREADS / TS_WAVE;
  __shared__ moe_f32x4 part_s[WAVES - 1][SETS][TS_WAVE];
  const int tile = blockIdx.x;
  const int rows = tiles[3 * tile + 2];
  if (rows == 0) return;
  const int e = tiles[3 * tile], first = tiles[3 * tile + 1];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TS_WAVE), lane = threadIdx.x & (TS_WAVE - 1);
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.y * 16;
  const int64_t expert_rows = GLU ? 2 * (int64_t)N : N;
  const bf16_t* we = w + (int64_t)e * expert_rows * K;
  const int pair = sorted[first + min(r, rows - 1)];
  const int col = min(n0 + r, N - 1);
  const int steps = K / 32, s0 = wave * steps / WAVES, s1 = (wave + 1) * steps / WAVES;
  const bf16_t* xp = x + (int64_t)(pair / src_div) * K + 8 * g;
  const bf16_t* wp[SETS];
  wp[0] = we + (int64_t)col * K + 8 * g;
  if constexpr (GLU) wp[1] = we + (int64_t)(N + col) * K + 8 * g;
  moe_f32x4 acc[SETS];
#pragma unroll
  for (int s = 0; s < SETS; ++s) acc[s] = (moe_f32x4){0.f, 0.f, 0.f, 0.f};
  int s = s0;
  auto stretch = [&](auto count) {
    constexpr int DEPTH = decltype(count)::value;
    moe_u32x4 fx[DEPTH], fw[SETS][DEPTH];
#pragma unroll
    for (int t = 0; t < SETS; ++t)
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) fw[t][d] = ONCE ? load_once<moe_u32x4>(wp[t] + 32 * (s + d)) : *(const moe_u32x4*)(wp[t] + 32 * (s + d));
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) fx[d] = *(const moe_u32x4*)(xp + 32 * (s + d));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
#pragma unroll
      for (int t = 0; t < SETS; ++t) acc[t] = moe_mfma(fw[t][d], fx[d], acc[t]);
    s += DEPTH;
  };
  while (s + 8 <= s1) stretch(std::integral_constant<int, 8>{});
  if (s + 4 <= s1) stretch(std::integral_constant<int, 4>{});
  for (; s < s1; ++s) {
    const moe_u32x4 fx = *(const moe_u32x4*)(xp + 32 * s);
#pragma unroll
    for (int t = 0; t < SETS; ++t) acc[t] = moe_mfma(*(const moe_u32x4*)(wp[t] + 32 * s), fx, acc[t]);
  }
  if (wave > 0) {
#pragma unroll
    for (int t = 0; t < SETS; ++t) part_s[wave - 1][t][lane] = acc[t];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int v = 0; v < WAVES - 1; ++v)
#pragma unroll
    for (int t = 0; t < SETS; ++t) acc[t] += part_s[v][t][lane];
  // lane (r, g): row r of the tile, columns n0 + 4 g .. + 3
  if (r >= rows) return;
  TO* orow = out + (int64_t)pair * N;
  const int c0 = n0 + 4 * g;
  float y[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    if constexpr (GLU) y[c] = moe_unit(acc[0][c], acc[1][c], limit, slope, shift);
    else y[c] = moe_act(acc[0][c], act);
  }
  moe_store4(orow + c0, y, N - c0);
}

// The same sums, bit for bit (a quarter's steps in turn, then the quarters), for reductions of whole lines (K a multiple of 256): a load of the kernel above takes 64 bytes of each of 16 rows, half a line,
// and past the caches the other half is a line fetched again. Here 64 of k at a time go from memory straight into LDS, 8 rows of 128 bytes a load, pieces turned
// by (row / 2) % 8 against bank conflicts; a wave has MOE_LINES of them there, its own, and waits for nobody. Without the gate a workgroup takes 32 columns.
// Both products of 16 experts over 2,048, 2 x 1,024 and back over 1,024, past the caches, the kernel above and here: 4 tokens of four choices 36.6 and 20.8 us, 16
// tokens 46.6 and 42.1, 48 tokens 55.2 and 45.5 (W at 4.4 TB/s), 64 tokens, some experts in two tiles, 91 and 61; through the caches 48 tokens 52.7 and 51.1.
#define MOE_LINES 3
template <bool GLU, typename TO, bool ONCE>
__global__ void __launch_bounds__(MOE_THREADS)
moe_gemm_lines_kernel(TO* __restrict__ out, const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, const int32_t* __restrict__ sorted,
                      const int32_t* __restrict__ tiles, int src_div, int N, int K, float limit, float slope, float shift, int act) {
  constexpr int WAVES = MOE_THREADS / TS_WAVE, R = MOE_LINES, STAGE = 3 * 2048;      // a stage: 16 rows of W twice, 16 rows of x, 64 of k
  __shared__ __attribute__((aligned(1024))) unsigned char lds[WAVES * R * STAGE];
  __shared__ moe_f32x4 part_s[WAVES - 1][2][TS_WAVE];
  const int tile = blockIdx.x;
  const int rows = tiles[3 * tile + 2];
  if (rows == 0) return;
  const int e = tiles[3 * tile], first = tiles[3 * tile + 1];
  const int wave = wave_index(), lane = threadIdx.x & (TS_WAVE - 1);
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.y * (GLU ? 16 : 32);
  const int stages = K / 256, k0 = wave * (K / 4);
  const bf16_t* we = w + ((int64_t)e * (GLU ? 2 : 1) * N + n0) * K + k0;
  const __amdgpu_buffer_rsrc_t rsrc[2] = {load_base(we), load_base(GLU ? we + (int64_t)N * K : we)};
  const uint32_t turned[2] = {(uint32_t)((lane % 8) ^ (lane / 16)) * 16, (uint32_t)((lane % 8) ^ (4 + lane / 16)) * 16};      // of rows lane / 8 and 8 + lane / 8
  uint32_t woff[2][2];
  int pair_at[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int at = 8 * q + lane / 8;
    pair_at[q] = sorted[first + min(at, rows - 1)];
#pragma unroll
    for (int t = 0; t < 2; ++t) woff[t][q] = (uint32_t)(min(GLU ? at : 16 * t + at, N - 1 - n0) * (int64_t)K * 2) + turned[q];
  }
  const uint32_t mine = (uint32_t)(uintptr_t)(lds_ptr_t)lds + wave * R * STAGE;
  auto fetch_w = [&](int stage, uint32_t slot) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        if constexpr (ONCE) load_to_lds_once(rsrc[t], mine + slot + (2 * t + q) * 1024, woff[t][q], (uint32_t)stage * 128);
        else load_to_lds(rsrc[t], mine + slot + (2 * t + q) * 1024, woff[t][q], (uint32_t)stage * 128);
      }
  };
  const int ahead = min(R, stages);
  for (int s = 0; s < ahead; ++s) fetch_w(s, s * STAGE);
  __builtin_amdgcn_sched_barrier(0);
  const bf16_t* xp[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) xp[q] = x + (int64_t)(pair_at[q] / src_div) * K + k0 + turned[q] / 2;
  auto fetch_x = [&](int stage, uint32_t slot) {
#pragma unroll
    for (int q = 0; q < 2; ++q) row_to_lds(xp[q] + stage * 64, mine + slot + (4 + q) * 1024);
  };
  for (int s = 0; s < ahead; ++s) fetch_x(s, s * STAGE);
  const int pair = sorted[first + min(r, rows - 1)];
  __builtin_amdgcn_sched_barrier(0);
  moe_f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  const uint32_t rd = (uint32_t)(r * 128 + (g ^ (r >> 1)) * 16);
  uint32_t slot = 0;
  for (int s = 0; s < stages; ++s) {
    // what has been asked for behind this stage: first the stages' rows of x behind their rows of W, and the pair's number, later whole stages
    const int behind = s < R ? 2 * (ahead - 1 - s) + 1 + 6 * min(s, stages - ahead) : 6 * min(R - 1, stages - 1 - s);
    if (behind >= 12) wait_for<12>();
    else if (behind >= 8) wait_for<8>();
    else if (behind >= 6) wait_for<6>();
    else if (behind >= 4) wait_for<4>();
    else if (behind >= 2) wait_for<2>();
    else wait_for<0>();
    __builtin_amdgcn_sched_barrier(0);
    const unsigned char* from = lds + wave * R * STAGE + slot;
    u32x4_t fw[2][2], fx[2];
#pragma unroll
    for (int d = 0; d < 2; ++d) {
#pragma unroll
      for (int t = 0; t < 2; ++t) fw[t][d] = *(const u32x4_t*)(from + t * 2048 + (rd ^ (64 * d)));
      fx[d] = *(const u32x4_t*)(from + 4096 + (rd ^ (64 * d)));
    }
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int t = 0; t < 2; ++t) acc[t] = mfma32v(fw[t][d], fx[d], acc[t]);
    __builtin_amdgcn_sched_barrier(0);      // (its operands have been read: the stage's place may be filled)
    if (s + R < stages) fetch_w(s + R, slot), fetch_x(s + R, slot);
    slot = slot == (R - 1) * STAGE ? 0 : slot + STAGE;
  }
  if (wave > 0) part_s[wave - 1][0][lane] = acc[0], part_s[wave - 1][1][lane] = acc[1];
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int v = 0; v < WAVES - 1; ++v) acc[0] += part_s[v][0][lane], acc[1] += part_s[v][1][lane];
  // lane (r, g): row r of the tile, columns n0 + 4 g .. + 3 (and 16 further on)
  if (r >= rows) return;
  TO* orow = out + (int64_t)pair * N;
  float y[4];
  if constexpr (GLU) {
#pragma unroll
    for (int c = 0; c < 4; ++c) y[c] = moe_unit(acc[0][c], acc[1][c], limit, slope, shift);
    moe_store4(orow + n0 + 4 * g, y, N - n0 - 4 * g);
  } else {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int c = 0; c < 4; ++c) y[c] = moe_act(acc[t][c], act);
      moe_store4(orow + n0 + 16 * t + 4 * g, y, N - n0 - 16 * t - 4 * g);
    }
  }
}

// Steps of 64 of k in a stretch of the tiles of 128 rows (a whole number of stretches).
static __device__ __forceinline__ int moe_stretch(int K) { return K >= 512 && K % 256 == 0 ? K / 256 : K / 64; }

// Tiles of 128 or 256 rows, for steps that give an expert dozens or hundreds of rows: the gated product's scheme (gemm_glu.hip)
// with the rows of x gathered by pair, the matrix the tile's expert's, and the rows of y stored at their pairs' places. A
// workgroup of eight waves takes BM rows by as many rows of W (with GLU half gate, half up rows, whose sums meet in one lane), 64
// of K at a time, K a multiple of 64. What bounds it is the matrix cores and a compute unit's path to memory: operands go from memory
// straight into LDS, two steps of x and three of W, pieces turned by (row / 2) % 8 against bank conflicts, and loads, operand
// reads and products are dealt out evenly. Of the smaller tile two workgroups share a compute unit, one waiting while the other
// multiplies: 128 x 128 is as fast as 128 x 256 at any size and faster where tiles are few. Both products of 16 experts over
// 2,048, 2 x 1,024 and back over 1,024, weights from memory: 64 pairs each 55 µs (128 x 256: 72, tiles of 64 rows without LDS 172), 128 each 81, 256
// each 112 (256 x 256: 99), 512 each 165 (184), 1,024 each 295 (274; where operands passed through registers on their way to LDS 342).
template <int BM, bool GLU, typename TO>
__global__ void __launch_bounds__(512, BM == 128 ? 4 : 2)
moe_gemm_lds_kernel(TO* __restrict__ out, const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                    const int32_t* __restrict__ sorted, const int32_t* __restrict__ tiles, int num_tiles, int col_blocks,
                    int src_div, int N, int K, float limit, float slope, float shift, int act) {
  constexpr int BN = BM, WN = BN / 64, WM = 8 / WN, WAVES = WM * WN, TM = BM / WM / 16, TN = BN / WN / 16, HALF = BN / WN / 2;
  constexpr int NX = BM / 8 / WAVES, NW = BN / 8 / WAVES;      // kilobytes of a step that a wave fetches
  constexpr int XS = BM * 128, WS = BN * 128;                  // bytes of a step of x and of W
  static_assert(HALF % (NW * 8) == 0, "a wave fetches gate rows or up rows");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * XS + 3 * WS];
  // Workgroups go to the chip's eight dies in turn, each die with a cache of its own: die d takes the d-th eighth
  // of the (tile, column block) list, column blocks innermost and tiles in the experts' order, so that the
  // workgroups a die runs at one time share a few tiles' rows and one expert's columns in its cache. The eighths are those
  // of the tiles that hold rows, which lead the table: it is made for the worst case, and eighths of all of it leave two
  // of the eight dies without work (the products above then take 98 and 63 µs with tiles of 128 rows).
  const int lane = threadIdx.x % TS_WAVE, r = lane % 16, g = lane / 16;
  int used = 0;
  for (int t0 = 0; t0 < num_tiles; t0 += TS_WAVE) used += __popcll(__ballot(t0 + lane < num_tiles && tiles[3 * min(t0 + lane, num_tiles - 1) + 2] > 0));
  const int per_die = (used * col_blocks + MOE_DIES - 1) / MOE_DIES, turn = blockIdx.x / MOE_DIES;
  const int item = __builtin_amdgcn_readfirstlane((blockIdx.x % MOE_DIES) * per_die + turn);
  if (turn >= per_die || item >= used * col_blocks) return;
  const int tile = item / col_blocks;
  const int rows = tiles[3 * tile + 2];
  const int e = tiles[3 * tile], first = tiles[3 * tile + 1];
  const int n0 = (item - tile * col_blocks) * (GLU ? BN / 2 : BN);
  const int wave = wave_index(), wm = wave % WM, wn = wave / WM;
  const int steps = K / 64;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)lds;

  // ---- the loading side (a row past the tile's, or a column past the matrix's last: the last one again) ----
  const bf16_t* xp[NX];
  uint32_t woff[NW];
#pragma unroll
  for (int q = 0; q < NX; ++q) {
    const int at = (wave * NX + q) * 8 + lane / 8;
    xp[q] = x + (int64_t)(sorted[first + min(at, rows - 1)] / src_div) * K + ((lane % 8) ^ ((at >> 1) & 7)) * 8;
  }
  const int ups = GLU && wave * NW * 8 / HALF % 2 ? N : 0;     // (the waves whose rows of the tile are up rows)
  const __amdgpu_buffer_rsrc_t rsrc_w = load_base(w + ((int64_t)e * (GLU ? 2 : 1) * N + n0 + ups) * K);
#pragma unroll
  for (int q = 0; q < NW; ++q) {
    const int at = (wave * NW + q) * 8 + lane / 8;
    woff[q] = (uint32_t)(min(GLU ? at / (2 * HALF) * HALF + at % HALF : at, N - 1 - n0) * K * 2) + ((lane % 8) ^ ((at >> 1) & 7)) * 16;
  }
  const uint32_t xfirst = lds0 + wave * NX * 1024, wfirst = lds0 + 2 * XS + wave * NW * 1024;
  uint32_t xslot = xfirst, wslot = wfirst;
  int xk = 0, wk = 0;
  auto fetch_x = [&]() {
#pragma unroll
    for (int q = 0; q < NX; ++q) row_to_lds(xp[q] + xk * 64, xslot + q * 1024);
  };
  auto fetch_w = [&]() {
#pragma unroll
    for (int q = 0; q < NW; ++q) load_to_lds(rsrc_w, wslot + q * 1024, woff[q], (uint32_t)wk * 128);
  };
  // (past the last step its loads are made again: a few, in bounds and never read)
  auto next_x = [&]() { xslot = xslot == xfirst ? xfirst + XS : xfirst, xk = min(xk + 1, steps - 1); };
  auto next_w = [&]() { wslot = wslot == wfirst + 2 * WS ? wfirst : wslot + WS, wk = min(wk + 1, steps - 1); };

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
  // (tiles of 128 rows have the registers for it: four stretches of k, so that the sums are as good as the narrow tiles')
  constexpr bool STRETCHES = BM == 128;
  const int stretch = moe_stretch(K);
  float4_t total[STRETCHES ? TN : 1][STRETCHES ? TM : 1];
  int left = stretch;
  if constexpr (STRETCHES)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) total[j][i] = (float4_t){0.f, 0.f, 0.f, 0.f};
  fetch_x(), next_x();
  fetch_w(), next_w();
  fetch_w(), next_w();
  fetch_x(), next_x();
  wait_for<NW + NX>();
  __builtin_amdgcn_s_barrier();
#define MOE_READ(S, RD)                                                                                        \
  _Pragma("unroll") for (int j = 0; j < TN; ++j) fw[S][j] = *(const u32x4_t*)(rw + (RD + wc) + j * 2048);      \
  _Pragma("unroll") for (int i = 0; i < TM; ++i) fx[S][i] = *(const u32x4_t*)(rx + (RD + xc) + i * 2048);
#define MOE_MULTIPLY(S)                                                                                        \
  _Pragma("unroll") for (int i = 0; i < TM; ++i)                                                               \
      _Pragma("unroll") for (int j = 0; j < TN; ++j) acc[j][i] = mfma32v(fw[S][j], fx[S][i], acc[j][i]);
// the order of a half step: TM TN products, among their first two thirds the TM + TN operand reads, among all the loads
#define MOE_DEAL(LOADS)                                                                                        \
  _Pragma("unroll") for (int q = 0; q < TM * TN; ++q) {                                                        \
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                                         \
    if ((q + 1) * (TM + TN) * 3 / 2 / (TM * TN) > q * (TM + TN) * 3 / 2 / (TM * TN)) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0); \
    if ((q + 1) * LOADS / (TM * TN) > q * LOADS / (TM * TN)) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0); \
  }                                                                                                            \
  __builtin_amdgcn_sched_barrier(0);
  MOE_READ(0, rd0)
  for (int s = 0; s < steps; ++s) {
    __builtin_amdgcn_sched_barrier(0);
    fetch_w();
    MOE_READ(1, rd1)
    MOE_MULTIPLY(0)
    MOE_DEAL(NW)
    next_w();
    xc = XS - xc;
    wc = wc == 2 * WS ? 0 : wc + WS;
    // every wave has read the last of this step's x and of W (so their places may be filled), and the next step has
    // landed: x was asked for half a step later than W, so all but the newest NW loads are done
    wait_for<NW, 0>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    fetch_x();
    MOE_READ(0, rd0)
    MOE_MULTIPLY(1)
    MOE_DEAL(NX)
    next_x();
    if constexpr (STRETCHES)
      if (--left == 0) {
        left = stretch;
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int i = 0; i < TM; ++i) total[j][i] += acc[j][i], acc[j][i] = (float4_t){0.f, 0.f, 0.f, 0.f};
      }
  }
  if constexpr (STRETCHES)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[j][i] = total[j][i];
#undef MOE_READ
#undef MOE_MULTIPLY
#undef MOE_DEAL
  // lane (r, g) of block (j, i): row 16 (wm TM + i) + r of the tile, columns .. + 4 g .. + 3
  int pair[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) pair[i] = sorted[first + min((wm * TM + i) * 16 + r, rows - 1)];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    TO* orow = out + (int64_t)pair[i] * N;
    const bool mine = (wm * TM + i) * 16 + r < rows;
    if constexpr (GLU) {
      const int c0 = n0 + wn * HALF;
      float y[TN / 2][4];
#pragma unroll
      for (int j = 0; j < TN / 2; ++j)
#pragma unroll
        for (int c = 0; c < 4; ++c) y[j][c] = moe_unit(acc[j][i][c], acc[j + TN / 2][i][c], limit, slope, shift);
      if (sizeof(TO) == 2 && N % 8 == 0 && ((uintptr_t)out & 15) == 0) {
        // lanes g and g ^ 1 exchange halves so that each has eight columns in a row
        static_assert(TN == 4, "two blocks of columns a wave");
        const auto lo = __builtin_amdgcn_permlane16_swap(pack_bf16(y[0][0], y[0][1]), pack_bf16(y[1][0], y[1][1]), false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap(pack_bf16(y[0][2], y[0][3]), pack_bf16(y[1][2], y[1][3]), false, false);
        const int c = c0 + (g & 1) * 16 + (g >> 1) * 8;
        if (mine && c < N) *(u32x4_t*)((bf16_t*)orow + c) = (u32x4_t){lo[0], hi[0], lo[1], hi[1]};
      } else if (mine) {
#pragma unroll
        for (int j = 0; j < TN / 2; ++j) moe_store4(orow + c0 + j * 16 + 4 * g, y[j], N - (c0 + j * 16 + 4 * g));
      }
    } else if (mine) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = n0 + (wn * TN + j) * 16 + 4 * g;
        const float y[4] = {moe_act(acc[j][i][0], act), moe_act(acc[j][i][1], act), moe_act(acc[j][i][2], act), moe_act(acc[j][i][3], act)};
        moe_store4(orow + n, y, N - n);
      }
    }
  }
  wait_for<0>();      // what was fetched beyond the end lands before the workgroup's LDS is another's
}

extern "C" int ts_moe_gemm(void* out, int out_dtype, const void* x, int x_dtype, const void* w, const int32_t* sorted,
                           const int32_t* tiles, int max_tiles, int tile_rows, int src_div, int N, int K, int glu, float limit,
                           float slope, float shift, int act, int once, hipStream_t stream) {
  if (max_tiles <= 0) return TS_OK;
  if (act < 0 || act > 1 || (glu && act)) return TS_BAD_SHAPE;
  if (N <= 0 || K <= 0 || src_div <= 0 || (tile_rows != 16 && tile_rows != 64 && tile_rows != 128 && tile_rows != 256)) return TS_BAD_SHAPE;
  const bool mfma = x_dtype == 1 && K % 32 == 0 && (((uintptr_t)x | (uintptr_t)w) & 15) == 0;
  if (tile_rows >= 128 && (!mfma || K % 64)) return TS_BAD_SHAPE;
  if (tile_rows >= 128 && K <= (1 << 22)) {                 // (byte offsets within 256 rows of W; longer reductions by 64-bit addresses below)
    const int per_block = glu ? tile_rows / 2 : tile_rows, col_blocks = (N + per_block - 1) / per_block;
    const int64_t items = (int64_t)max_tiles * col_blocks;
    if (items > 0x3fffffff) return TS_BAD_SHAPE;
    const unsigned grid = (unsigned)((items + MOE_DIES - 1) / MOE_DIES * MOE_DIES);
#define MOE_LDS(BM, GLU, TO) \
    moe_gemm_lds_kernel<BM, GLU, TO><<<grid, 512, 0, stream>>>((TO*)out, (const bf16_t*)x, (const bf16_t*)w, sorted, tiles, max_tiles, \
                                                               col_blocks, src_div, N, K, limit, slope, shift, act)
#define MOE_LDS_ROWS(GLU, TO) \
    if (tile_rows == 256) MOE_LDS(256, GLU, TO); \
    else MOE_LDS(128, GLU, TO)
    if (glu && out_dtype == 1) { MOE_LDS_ROWS(true, bf16_t); }
    else if (!glu && out_dtype == 0) { MOE_LDS_ROWS(false, float); }
    else if (!glu && out_dtype == 1) { MOE_LDS_ROWS(false, bf16_t); }
    else return TS_BAD_DTYPE;
#undef MOE_LDS_ROWS
#undef MOE_LDS
    return ts_check_launch();
  }
  if (mfma) {
    if (tile_rows == 16) {
      dim3 grid(max_tiles, (N + 15) / 16);
      if (grid.y > 65535) return TS_BAD_SHAPE;
      if (K % 256 == 0 && K <= (1 << 22)) {                 // (byte offsets within 32 rows of W)
        if (!glu) grid.y = (N + 31) / 32;
#define MOE_BY_LINES(GLU, TO) \
        (once ? moe_gemm_lines_kernel<GLU, TO, true> : moe_gemm_lines_kernel<GLU, TO, false>)<<<grid, MOE_THREADS, 0, stream>>>( \
            (TO*)out, (const bf16_t*)x, (const bf16_t*)w, sorted, tiles, src_div, N, K, limit, slope, shift, act)
        if (glu && out_dtype == 1) MOE_BY_LINES(true, bf16_t);
        else if (!glu && out_dtype == 0) MOE_BY_LINES(false, float);
        else if (!glu && out_dtype == 1) MOE_BY_LINES(false, bf16_t);
        else return TS_BAD_DTYPE;
#undef MOE_BY_LINES
        return ts_check_launch();
      }
#define MOE_STREAM(GLU, TO) \
      (once ? moe_gemm_stream_kernel<GLU, TO, true> : moe_gemm_stream_kernel<GLU, TO, false>)<<<grid, MOE_THREADS, 0, stream>>>( \
          (TO*)out, (const bf16_t*)x, (const bf16_t*)w, sorted, tiles, src_div, N, K, limit, slope, shift, act)
      if (glu && out_dtype == 1) MOE_STREAM(true, bf16_t);
      else if (!glu && out_dtype == 0) MOE_STREAM(false, float);
      else if (!glu && out_dtype == 1) MOE_STREAM(false, bf16_t);
      else return TS_BAD_DTYPE;
#undef MOE_STREAM
      return ts_check_launch();
    }
    // (a wave takes 32 columns of all the tile's rows; with the gate, 32 gate and 32 up columns)
    const int parts = tile_rows / 64;
    dim3 grid((unsigned)max_tiles * parts, (N + 127) / 128);
    if (grid.y > 65535 || max_tiles > 0x3fffffff / parts) return TS_BAD_SHAPE;
#define MOE_MFMA(TM, GLU, TO) \
    moe_gemm_mfma_kernel<TM, 2, GLU, TO><<<grid, MOE_THREADS, 0, stream>>>((TO*)out, (const bf16_t*)x, (const bf16_t*)w, sorted, \
                                                                           tiles, parts, src_div, N, K, limit, slope, shift, act)
    if (glu && out_dtype == 1) MOE_MFMA(4, true, bf16_t);
    else if (!glu && out_dtype == 0) MOE_MFMA(4, false, float);
    else if (!glu && out_dtype == 1) MOE_MFMA(4, false, bf16_t);
    else return TS_BAD_DTYPE;
#undef MOE_MFMA
    return ts_check_launch();
  }
  if (tile_rows != MOE_BM) return TS_BAD_SHAPE;
  dim3 grid(max_tiles, (N + MOE_BN - 1) / MOE_BN);
  if (grid.y > 65535) return TS_BAD_SHAPE;
#define MOE_LAUNCH(TX, TO) \
  moe_gemm_kernel<TX, TO><<<grid, MOE_THREADS, 0, stream>>>((TO*)out, (const TX*)x, (const TX*)w, sorted, tiles, src_div, N, K, \
                                                            glu, limit, slope, shift, act)
  if (x_dtype == 0 && out_dtype == 0) MOE_LAUNCH(float, float);
  else if (x_dtype == 1 && out_dtype == 1) MOE_LAUNCH(bf16_t, bf16_t);
  else if (x_dtype == 1 && out_dtype == 0) MOE_LAUNCH(bf16_t, float);
  else return TS_BAD_DTYPE;
#undef MOE_LAUNCH
  return ts_check_launch();
}

// A thread per four columns of a token (or per column, where rows are no whole 16-byte pieces): a step of one token
// spreads over the row's width and waits for memory once.
template <int VEC, typename TX>
__global__ void __launch_bounds__(MOE_THREADS)
moe_combine_kernel(float* __restrict__ out, const float* __restrict__ rows, const float* __restrict__ weights,
                   const float* __restrict__ shared, int width, int top, const int32_t* __restrict__ ids, int real,
                   const TX* __restrict__ x, const float* __restrict__ shared_gate) {
  const int64_t t = blockIdx.x;
  const int i = (blockIdx.y * MOE_THREADS + threadIdx.x) * VEC;
  if (i >= width) return;
  float acc[VEC];
#pragma unroll
  for (int c = 0; c < VEC; ++c) acc[c] = 0.f;
  for (int j = 0; j < top; ++j) {
    const float w = weights[t * top + j];
    if (ids && ids[t * top + j] >= real) {                // an identity expert: the token's input itself
#pragma unroll
      for (int c = 0; c < VEC; ++c) acc[c] = fmaf(w, Num<TX>::ld(x + t * width + i + c), acc[c]);
      continue;
    }
    const float* row = rows + (t * top + j) * width + i;
    if constexpr (VEC == 4) {
      const float4 v = *(const float4*)row;
      acc[0] = fmaf(w, v.x, acc[0]); acc[1] = fmaf(w, v.y, acc[1]); acc[2] = fmaf(w, v.z, acc[2]); acc[3] = fmaf(w, v.w, acc[3]);
    } else {
      acc[0] = fmaf(w, row[0], acc[0]);
    }
  }
  const float g = shared_gate ? shared_gate[t] : 1.0f;
  if constexpr (VEC == 4) {
    if (shared) {
      const float4 v = *(const float4*)(shared + t * width + i);
      acc[0] = fmaf(g, v.x, acc[0]); acc[1] = fmaf(g, v.y, acc[1]); acc[2] = fmaf(g, v.z, acc[2]); acc[3] = fmaf(g, v.w, acc[3]);
    }
    *(float4*)(out + t * width + i) = make_float4(acc[0], acc[1], acc[2], acc[3]);
  } else {
    if (shared) acc[0] = fmaf(g, shared[t * width + i], acc[0]);
    out[t * width + i] = acc[0];
  }
}

extern "C" int ts_moe_combine(float* out, const float* rows, const float* weights, const float* shared, int num_tokens,
                              int width, int top, const int32_t* ids, int real, const void* x, int x_dtype,
                              const float* shared_gate, hipStream_t stream) {
  if (num_tokens <= 0) return TS_OK;
  if (width <= 0 || top <= 0 || (ids && !x) || (shared_gate && !shared)) return TS_BAD_SHAPE;
  if (x_dtype != 0 && x_dtype != 1) return TS_BAD_DTYPE;
  const bool by4 = width % 4 == 0 && (((uintptr_t)out | (uintptr_t)rows | (uintptr_t)shared) & 15) == 0;
  const int per_block = MOE_THREADS * (by4 ? 4 : 1);
  dim3 grid(num_tokens, (width + per_block - 1) / per_block);
  if (grid.y > 65535) return TS_BAD_SHAPE;
#define MOE_COMBINE(VEC, TX) \
  moe_combine_kernel<VEC, TX><<<grid, MOE_THREADS, 0, stream>>>(out, rows, weights, shared, width, top, ids, real, (const TX*)x, shared_gate)
  if (by4 && x_dtype == 0) MOE_COMBINE(4, float);
  else if (by4) MOE_COMBINE(4, bf16_t);
  else if (x_dtype == 0) MOE_COMBINE(1, float);
  else MOE_COMBINE(1, bf16_t);
#undef MOE_COMBINE
  return ts_check_launch();
}
