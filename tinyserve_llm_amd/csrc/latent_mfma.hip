// Multi-query attention over cached latent rows on the matrix cores (bfloat16 caches). A token's cached row is
// [c | r] (`rank` + `rot` numbers); the values are the rows' first `rank` numbers, which the cache also keeps once
// more, transposed inside its pages ([rank, page_size]), because the product P.V wants, for one dimension,
// consecutive keys side by side. All heads of a token share the keys, so the heads are the rows of the matrix
// products: a workgroup owns a tile of 32 rows (32 heads of one token, or all heads of several tokens of one request
// where a token has fewer) and walks the tile's keys in 32-key steps. Its four waves split the dimensions, not the
// keys: a cached row is long, and a wave that held whole rows and whole value columns would have registers for
// nothing else. Of every step
//     S^T[key, row] = K[key, :] . Q[row, :]       v_mfma_f32_16x16x32_bf16, keys as rows, Q from shared memory:
//                                                 each wave sums over its quarter of the row's 32-wide pieces, the
//                                                 quarters meet in shared memory and every wave adds them in one order
//     P = 2^(S scale log2 e - m), 32-bit, the same in every wave; into the second product as two bfloat16 terms
//     O^T[dim, row] += V^T[dim, key] . P[row, key]  each wave its quarter of the value columns
// while the next step's keys and values are on their way. Where a step has few tiles (decoded tokens) the keys of a
// tile are cut into stretches, a workgroup each, whose parts (maximum, sum, unnormalised rows) a second kernel adds up.
// Queries arrive 32-bit and are rounded to bfloat16 once, as the keys were. Scores, maxima, weights and sums are
// 32-bit. Causal, with a sliding window or chunks (`ts_first_key`). Optionally a learned sink per head in the softmax's
// denominator and a gate per head (sigmoid) on the result.
#include "lds_loads.h"

#define LM_WAVES 4
#define LM_THREADS (LM_WAVES * TS_WAVE)
#define LM_RT 2                 // 16-row tiles of a workgroup
#define LM_ROWS (16 * LM_RT)
#define LM_MAX_SPLITS 16

// What an unnormalised sum is multiplied by: 1 / (its weights' sum `total`, in units of 2^m, and the head's sink's).
static __device__ __forceinline__ float lm_scale(float m, float total, const float* __restrict__ sinks, int head) {
  if (!sinks) return 1.0f / total;
  const float s = sinks[head] * 1.4426950408889634f, top = fmaxf(m, s);
  return fast_exp2(m - top) / (total * fast_exp2(m - top) + fast_exp2(s - top));
}
static __device__ __forceinline__ float lm_gate(const float* __restrict__ gate, int64_t at) {
  return gate ? 1.0f / (1.0f + expf(-gate[at])) : 1.0f;
}

// CPW: 32-wide pieces of a cached row per wave (row <= 128 CPW); VPW: 16-wide blocks of value columns per wave
// (rank <= 64 VPW). Wave w takes pieces w, w + 4, ... and blocks w, w + 4, ...; those past the actual sizes are loaded
// from a valid address (the row's last piece, the last column) and not multiplied.
template <int CPW, int VPW, typename TO>
__global__ void __launch_bounds__(LM_THREADS)
latent_attention_mfma_kernel(TO* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml,
                             const float* __restrict__ q, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
                             const int32_t* __restrict__ block_tables, const int32_t* __restrict__ seq_of_token,
                             const int32_t* __restrict__ positions, const int32_t* __restrict__ tiles, int num_tiles,
                             int tile_tokens, int heads_block, int nh, int rank, int row, int64_t kp, int64_t ks, int64_t vp,
                             int64_t vd, int max_blocks, float scale_log2, int window, int page_run, int splits,
                             const float* __restrict__ sinks, const float* __restrict__ gate, int64_t gate_token) {
  constexpr int QS = CPW * 128 + 8;                         // a row of the queries in shared memory, skewed
  __shared__ __attribute__((aligned(16))) bf16_t q_s[LM_ROWS][QS];
  __shared__ __attribute__((aligned(16))) float4_t s_part[2][LM_WAVES][LM_RT][2][TS_WAVE];
  // tiles that lie side by side in the step go to one die's second-level cache: they read the same keys
  const int per_die = (num_tiles + 7) / 8;
  const int tile = (blockIdx.x & 7) * per_die + (blockIdx.x >> 3);
  if (tile >= num_tiles) return;
  const int t0 = tiles ? tiles[2 * tile] : tile;
  const int count = tiles ? tiles[2 * tile + 1] : 1;
  const int hb = blockIdx.y, split = blockIdx.z;
  const int heads_here = min(nh - heads_block * hb, heads_block);      // heads of a token in this tile
  const int wave = wave_index(), lane = threadIdx.x & (TS_WAVE - 1);
  const int r = lane & 15, g = lane >> 4;
  const int nks = (row + 31) / 32, nvb = rank / 16;
  // row i of the tile: token t0 + i / heads_here, head heads_block hb + i % heads_here
  const int pos0 = positions[t0];
  int my_pos[LM_RT], my_lo[LM_RT];
#pragma unroll
  for (int rt = 0; rt < LM_RT; ++rt) {
    const int tok = (16 * rt + r) / heads_here;
    const bool valid = tok < count && tok < tile_tokens;
    my_pos[rt] = valid ? pos0 + tok : -1;                   // (a tile's tokens are consecutive positions of one request)
    my_lo[rt] = valid ? ts_first_key(my_pos[rt], window) : 0;
  }
  const int lo_min = ts_first_key(pos0, window), pos_max = pos0 + count - 1;
  const int32_t* table = block_tables + (int64_t)seq_of_token[t0] * max_blocks;

  // the tile's queries, rounded once, zeros where there is no row or no dimension. Every thread's loads go out
  // together, each from an address inside the step's queries (a row without a token reads the tile's first).
  __shared__ int64_t src_s[LM_ROWS];
  if (threadIdx.x < LM_ROWS) {
    const int tok = threadIdx.x / heads_here, head = heads_block * hb + threadIdx.x % heads_here;
    src_s[threadIdx.x] = (tok < count && tok < tile_tokens) ? ((int64_t)(t0 + tok) * nh + head) * row : -1;
  }
  __syncthreads();
  {
    constexpr int F4 = CPW * 32, PER = LM_ROWS * F4 / LM_THREADS;       // 16-byte pieces of a row; of a thread
    const int64_t fallback = ((int64_t)t0 * nh + heads_block * hb) * row;
    float4 got[PER];
#pragma unroll
    for (int it = 0; it < PER; ++it) {
      const int i = threadIdx.x + it * LM_THREADS, rr = i / F4, d = 4 * (i - rr * F4);
      const int64_t src = src_s[rr];
      got[it] = *(const float4*)(q + (src < 0 ? fallback : src) + min(d, row - 4));
    }
#pragma unroll
    for (int it = 0; it < PER; ++it) {
      const int i = threadIdx.x + it * LM_THREADS, rr = i / F4, d = 4 * (i - rr * F4);
      const bool in = src_s[rr] >= 0 && d < row;
      uint2 packed;
      packed.x = in ? pack_bf16(got[it].x, got[it].y) : 0u;
      packed.y = in ? pack_bf16(got[it].z, got[it].w) : 0u;
      *(uint2*)&q_s[rr][d] = packed;
    }
  }
  __syncthreads();

  float4_t acc[LM_RT][VPW];
#pragma unroll
  for (int rt = 0; rt < LM_RT; ++rt)
#pragma unroll
    for (int i = 0; i < VPW; ++i) acc[rt][i] = (float4_t){0.f, 0.f, 0.f, 0.f};
  float m[LM_RT], l[LM_RT];
#pragma unroll
  for (int rt = 0; rt < LM_RT; ++rt) m[rt] = -INFINITY, l[rt] = 0.f;
  // this workgroup's stretch of the tile's 32-key steps
  const int kb0 = lo_min & ~31;
  const int steps = ((pos_max - kb0) >> 5) + 1, per = (steps + splits - 1) / splits;
  const int first = split * per, last = min(steps, first + per) - 1;       // (an empty stretch: last < first)
  auto page_of = [&](int step) -> int64_t {                  // a step lies inside one page of the pool (pages of 32 keys)
    const int pg = (kb0 >> 5) + step;
    return ((int64_t)table[pg >> page_run] << page_run) + (pg & ((1 << page_run) - 1));
  };
  // every lane loads, whatever its piece and block, from an address inside the page: loads under branches would be
  // waited for one by one. What is read past the row's end meets zeros of the queries.
  auto load_keys = [&](uint4 (&kf)[2][CPW], int64_t page) {
#pragma unroll
    for (int tau = 0; tau < 2; ++tau) {
      const bf16_t* krow = k_cache + page * kp + (int64_t)(8 * (r >> 2) + 4 * tau + (r & 3)) * ks;
#pragma unroll
      for (int i = 0; i < CPW; ++i) kf[tau][i] = *(const uint4*)(krow + min(32 * (wave + LM_WAVES * i) + 8 * g, row - 8));
    }
  };
  auto load_values = [&](uint4 (&vf)[VPW], int64_t page) {
#pragma unroll
    for (int i = 0; i < VPW; ++i)
      vf[i] = *(const uint4*)(v_cache + page * vp + (int64_t)min(16 * (wave + LM_WAVES * i) + r, rank - 1) * vd + 8 * g);
  };
  uint4 kf[2][CPW], vf[VPW], kn[2][CPW], vn[VPW];
  if (first <= last) {
    const int64_t page = page_of(first);
    load_keys(kf, page);
    load_values(vf, page);
  }
  for (int step = first; step <= last; ++step) {
    const int64_t page_next = page_of(min(step + 1, last));  // (the last step asks for itself again)
    load_keys(kn, page_next);
    load_values(vn, page_next);
    const int kb = kb0 + 32 * step, par = (step - first) & 1;
#pragma unroll
    for (int rt = 0; rt < LM_RT; ++rt)
#pragma unroll
      for (int tau = 0; tau < 2; ++tau) {
        float4_t st = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < CPW; ++i) {
          const int c = wave + LM_WAVES * i;
          if (c < nks) st = mfma32(kf[tau][i], *(const uint4*)&q_s[16 * rt + r][32 * c + 8 * g], st);
        }
        s_part[par][wave][rt][tau][lane] = st;
      }
    __syncthreads();                                         // (one a step: the next step writes the other half)
    uint4 hi[LM_RT], lo[LM_RT];
    float alpha[LM_RT];
#pragma unroll
    for (int rt = 0; rt < LM_RT; ++rt) {
      float s[8];
#pragma unroll
      for (int tau = 0; tau < 2; ++tau) {
        float4_t st = s_part[par][0][rt][tau][lane];
#pragma unroll
        for (int w = 1; w < LM_WAVES; ++w) {
          const float4_t o = s_part[par][w][rt][tau][lane];
#pragma unroll
          for (int j = 0; j < 4; ++j) st[j] += o[j];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int key = kb + 8 * g + 4 * tau + j;
          s[4 * tau + j] = (key >= my_lo[rt] && key <= my_pos[rt]) ? st[j] * scale_log2 : -INFINITY;
        }
      }
      float top = s[0];
#pragma unroll
      for (int j = 1; j < 8; ++j) top = fmaxf(top, s[j]);
      const float m_new = fmaxf(m[rt], row_max(top));
      const float m_safe = m_new == -INFINITY ? 0.f : m_new;
      alpha[rt] = fast_exp2(m[rt] - m_safe);                 // (m = -inf: nothing summed yet, and 2^-inf = 0)
      float p[8], sum = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        p[j] = fast_exp2(s[j] - m_safe);
        sum += p[j];
      }
      l[rt] = l[rt] * alpha[rt] + sum;
      m[rt] = m_new;
      uint32_t* hw = (uint32_t*)&hi[rt];
      uint32_t* lw = (uint32_t*)&lo[rt];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        hw[j] = pack_bf16(p[2 * j], p[2 * j + 1]);
        const float r0 = p[2 * j] - __uint_as_float(hw[j] << 16), r1 = p[2 * j + 1] - __uint_as_float(hw[j] & 0xffff0000u);
        lw[j] = pack_bf16(r0, r1);
      }
    }
#pragma unroll
    for (int i = 0; i < VPW; ++i)
      if (wave + LM_WAVES * i < nvb) {
#pragma unroll
        for (int rt = 0; rt < LM_RT; ++rt) {
          float4_t a = acc[rt][i];
#pragma unroll
          for (int j = 0; j < 4; ++j) a[j] *= alpha[rt];
          a = mfma32(vf[i], hi[rt], a);
          acc[rt][i] = mfma32(vf[i], lo[rt], a);
        }
      }
#pragma unroll
    for (int tau = 0; tau < 2; ++tau)
#pragma unroll
      for (int i = 0; i < CPW; ++i) kf[tau][i] = kn[tau][i];
#pragma unroll
    for (int i = 0; i < VPW; ++i) vf[i] = vn[i];
  }
  // lane (r, g) holds, of row 16 rt + r, the columns 16 db + 4 g .. + 3 of its wave's blocks
#pragma unroll
  for (int rt = 0; rt < LM_RT; ++rt) {
    const int rr = 16 * rt + r;
    const int tok = rr / heads_here, head = heads_block * hb + rr % heads_here;
    const float total = row_sum(l[rt]);                      // (every lane takes part, whatever its row)
    if (tok >= count || tok >= tile_tokens) continue;
    const int64_t item = (int64_t)(t0 + tok) * nh + head;
    if (splits == 1) {
      const float inv = lm_scale(m[rt], total, sinks, head) * lm_gate(gate, (int64_t)(t0 + tok) * gate_token + head);
#pragma unroll
      for (int i = 0; i < VPW; ++i) {
        const int db = wave + LM_WAVES * i;
        if (db >= nvb) continue;
        TO* dst = out + item * rank + 16 * db + 4 * g;
#pragma unroll
        for (int j = 0; j < 4; ++j) Num<TO>::st(dst + j, acc[rt][i][j] * inv);
      }
    } else {
      float* dst = part_o + (item * splits + split) * rank;
#pragma unroll
      for (int i = 0; i < VPW; ++i) {
        const int db = wave + LM_WAVES * i;
        if (db >= nvb) continue;
        *(float4_t*)(dst + 16 * db + 4 * g) = acc[rt][i];
      }
      if (wave == 0 && g == 0) {
        part_ml[(item * splits + split) * 2] = m[rt];
        part_ml[(item * splits + split) * 2 + 1] = total;
      }
    }
  }
}

// One workgroup per (token, head), a thread per value column: the stretches' parts to one row. m is in units of log2.
template <typename TO>
__global__ void __launch_bounds__(LM_THREADS)
latent_attention_combine_kernel(TO* __restrict__ out, const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                int rank, int splits, int nh, const float* __restrict__ sinks, const float* __restrict__ gate,
                                int64_t gate_token) {
  const int64_t item = blockIdx.x;
  const int64_t tok = item / nh;
  const int head = (int)(item - tok * nh);
  const float* ml = part_ml + item * splits * 2;
  float ms[LM_MAX_SPLITS], ls[LM_MAX_SPLITS], top = -INFINITY;
#pragma unroll
  for (int z = 0; z < LM_MAX_SPLITS; ++z) {
    ms[z] = ml[2 * min(z, splits - 1)];
    ls[z] = ml[2 * min(z, splits - 1) + 1];
    top = fmaxf(top, ms[z]);
  }
  float weight[LM_MAX_SPLITS], total = 0.f;
#pragma unroll
  for (int z = 0; z < LM_MAX_SPLITS; ++z) {
    weight[z] = z < splits ? fast_exp2(ms[z] - top) : 0.f;   // (a stretch without keys: 2^-inf = 0)
    total += weight[z] * ls[z];
  }
  const float inv = lm_scale(top, total, sinks, head) * lm_gate(gate, tok * gate_token + head);
  for (int d = threadIdx.x; d < rank; d += LM_THREADS) {
    float part[LM_MAX_SPLITS];
#pragma unroll
    for (int z = 0; z < LM_MAX_SPLITS; ++z) part[z] = part_o[(item * splits + min(z, splits - 1)) * rank + d];
    float sum = 0.f;
#pragma unroll
    for (int z = 0; z < LM_MAX_SPLITS; ++z) sum = fmaf(weight[z], part[z], sum);
    Num<TO>::st(out + item * rank + d, sum * inv);
  }
}

// Whether the kernel is built for a cached row of `row` numbers of which `rank` are the values.
extern "C" int ts_latent_mfma_takes(int rank, int row) {
  return rank > 0 && rank % 16 == 0 && row % 8 == 0 && rank <= row && row <= 640 && rank <= 512;
}

// tiles: int32 [num_tiles, 2] (first token, token count <= tile_tokens), every tile inside one request, or null:
// every token a tile of its own. A tile's rows are tile_tokens tokens by heads_block heads (at most 32 together);
// heads beyond heads_block take further workgroups. splits > 1: part_o float32 [tokens, heads, splits, rank] and
// part_ml float32 [tokens, heads, splits, 2] receive the stretches' parts.
extern "C" int ts_paged_attention_latent_mfma(void* out, int out_dtype, const float* q, const void* k_cache, const void* v_cache,
                                              const int32_t* block_tables, const int32_t* seq_of_token, const int32_t* positions,
                                              const int32_t* tiles, int num_tiles, int tile_tokens, int num_tokens, int nh, int rank,
                                              int rot, int page_size, int64_t kp, int64_t ks, int64_t vp, int64_t vd,
                                              int64_t v_slot, int max_blocks, float scale, int window, int page_run, int splits,
                                              float* part_o, float* part_ml, const float* sinks, const float* gate,
                                              int64_t gate_token, hipStream_t stream) {
  if (num_tiles <= 0 || num_tokens <= 0) return TS_OK;
  const int row = rank + rot;
  const int heads_block = min(nh, LM_ROWS);
  if (!ts_latent_mfma_takes(rank, row) || nh <= 0 || page_size != 32 || v_slot != 1 || kp % 8 || ks % 8 || vp % 8 || vd % 8 ||
      ((uintptr_t)k_cache & 15) || ((uintptr_t)v_cache & 15) || max_blocks <= 0 || page_run < 0 || page_run > 16 ||
      tile_tokens < 1 || tile_tokens * heads_block > LM_ROWS || (!tiles && (num_tiles != num_tokens || tile_tokens != 1)) ||
      splits < 1 || splits > LM_MAX_SPLITS || (splits > 1 && (!part_o || !part_ml)))
    return TS_BAD_SHAPE;
  dim3 grid(((num_tiles + 7) / 8) * 8, (nh + heads_block - 1) / heads_block, splits);
  const float scale_log2 = scale * 1.4426950408889634f;
#define LM_LAUNCH(CPW, VPW, TO) \
  latent_attention_mfma_kernel<CPW, VPW, TO><<<grid, LM_THREADS, 0, stream>>>((TO*)out, part_o, part_ml, q, (const bf16_t*)k_cache, \
      (const bf16_t*)v_cache, block_tables, seq_of_token, positions, tiles, num_tiles, tile_tokens, heads_block, nh, rank, row, kp, ks, \
      vp, vd, max_blocks, scale_log2, window, page_run, splits, sinks, gate, gate_token)
#define LM_PICK(TO) \
  do { \
    if (row <= 256 && rank <= 128) LM_LAUNCH(2, 2, TO); \
    else if (row <= 384 && rank <= 256) LM_LAUNCH(3, 4, TO); \
    else if (row <= 512) LM_LAUNCH(4, 8, TO); \
    else LM_LAUNCH(5, 8, TO); \
    if (splits > 1) { \
      const int64_t items = (int64_t)num_tokens * nh; \
      latent_attention_combine_kernel<TO><<<(unsigned)items, LM_THREADS, 0, stream>>>((TO*)out, part_o, part_ml, rank, splits, nh, sinks, \
                                                                                        gate, gate_token); \
    } \
  } while (0)
  if (out_dtype == 0) LM_PICK(float);
  else if (out_dtype == 1) LM_PICK(bf16_t);
  else return TS_BAD_DTYPE;
#undef LM_PICK
#undef LM_LAUNCH
  return ts_check_launch();
}

// ---- steps of many tokens ---------------------------------------------------------------------------------------
// The same for steps that fill the chip with tiles of 128 rows (four tokens of 32 heads): a workgroup of eight waves, a wave
// 16 rows with their queries and whole outputs in registers, and every 32-key step's keys and values shared by all of them
// through LDS, where they go straight from memory, three steps in turn (one worked on, two under way). What bounds it: the
// matrix cores, 48 products a wave and step of 256 numbers (16 for the scores, 32 for the weights' two bfloat16 terms),
// beside the wave's softmax; the kernel above reads every token's keys from the second-level cache anew (2 GB for 2,048
// tokens over 256 numbers: 560 us, this one 112). The operands are read LP_AHEAD ahead of the products that take them, the
// first values ahead of the softmax: with each pair of reads waited for, as the compiler lays them out, it took 129 (heads of
// 320 numbers 118 and now 100, 130 heads of 80 388 and 351; 6 and 8 ahead the same). Waves of 32 rows, four to a workgroup and
// two workgroups to a unit, read half as much from LDS and took 138 to 160: no registers are left to read ahead into.
// In LDS a key's 16-byte pieces are turned by the key's place among the 16 that an operand takes, a value column's four by
// half the column's number: an operand's read then meets every bank once.
#define LP_WAVES 8
#define LP_ROWS (16 * LP_WAVES)
#define LP_RING 3
#define LP_AHEAD 4

// CP: 32-wide pieces of a cached row, VB: 16-wide blocks of value columns, both rounded up to what is built.
template <int CP, int VB, typename TO>
__global__ void __launch_bounds__(LP_WAVES * TS_WAVE, 2)
latent_attention_tiles_kernel(TO* __restrict__ out, const float* __restrict__ q, const bf16_t* __restrict__ k_cache,
                              const bf16_t* __restrict__ v_cache, const int32_t* __restrict__ block_tables,
                              const int32_t* __restrict__ seq_of_token, const int32_t* __restrict__ positions,
                              const int32_t* __restrict__ tiles, int num_tiles, int heads_block, int nh, int rank, int row,
                              int64_t kp, int64_t ks, int64_t vp, int64_t vd, int max_blocks, float scale_log2, int window,
                              int page_run, const float* __restrict__ sinks, const float* __restrict__ gate, int64_t gate_token) {
  constexpr int SL = (4 * CP + 15) / 16 * 16;               // 16-byte places of a key in LDS
  constexpr int KBYTES = 32 * SL * 16, STEP = KBYTES + VB * 1024;
  constexpr int NK = KBYTES / 1024 / LP_WAVES, NV = VB / LP_WAVES;       // kilobytes of a step that a wave fetches
  static_assert(VB % LP_WAVES == 0 && KBYTES % (1024 * LP_WAVES) == 0, "whole kilobytes a wave");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[LP_RING * STEP];
  const int tile = num_tiles - 1 - blockIdx.x;              // (the list ascends by the keys to walk: the longest first)
  const int t0 = tiles[2 * tile], count = tiles[2 * tile + 1], hb = blockIdx.y;
  const int heads_here = min(nh - heads_block * hb, heads_block);
  const int wave = wave_index(), lane = threadIdx.x & (TS_WAVE - 1), r = lane & 15, g = lane >> 4;
  // this lane's row of the tile: token t0 + i / heads_here, head heads_block hb + i % heads_here
  const int i_row = 16 * wave + r, tok = i_row / heads_here, head = heads_block * hb + i_row % heads_here;
  const bool valid = tok < count;
  const int pos0 = positions[t0], pos_max = pos0 + count - 1;
  const int my_pos = valid ? pos0 + tok : pos_max, my_lo = ts_first_key(my_pos, window);
  const int32_t* table = block_tables + (int64_t)seq_of_token[t0] * max_blocks;
  const int kb0 = ts_first_key(pos0, window) & ~31, steps = ((pos_max - kb0) >> 5) + 1;
  const int all_from = ts_first_key(pos_max, window);       // keys from here up to pos0 are seen by every row
  auto page_of = [&](int step) -> int64_t {                  // a step lies inside one page of the pool (pages of 32 keys)
    const int pg = (kb0 >> 5) + min(step, steps - 1);
    return ((int64_t)table[pg >> page_run] << page_run) + (pg & ((1 << page_run) - 1));
  };
  // ---- the loading side ----
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)lds;
  uint32_t koff[NK], voff[NV];
#pragma unroll
  for (int n = 0; n < NK; ++n) {
    const int place = (wave * NK + n) * 64 + lane, key = place / SL, kr = 4 * (key >> 3) + (key & 3);
    koff[n] = (uint32_t)(key * ks * 2) + min(8 * ((place % SL) ^ kr), row - 8) * 2;      // (past the row's end: zeros of the queries)
  }
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int d = (wave * NV + n) * 16 + lane / 4;
    voff[n] = (uint32_t)(min(d, rank - 1) * vd * 2) + ((lane % 4) ^ ((d >> 1) & 3)) * 16;
  }
  auto fetch = [&](int slot, int64_t page) {
    const __amdgpu_buffer_rsrc_t kb = load_base(k_cache + page * kp), vb = load_base(v_cache + page * vp);
    const uint32_t at = lds0 + slot * STEP;
#pragma unroll
    for (int n = 0; n < NK; ++n) load_to_lds(kb, at + (wave * NK + n) * 1024, koff[n], 0);
#pragma unroll
    for (int n = 0; n < NV; ++n) load_to_lds(vb, at + KBYTES + (wave * NV + n) * 1024, voff[n], 0);
  };
  fetch(0, page_of(0));
  fetch(1, page_of(1));
  int64_t page_next = page_of(2);
  // the wave's queries, rounded once, zeros where there is no row or no dimension
  u32x4_t qf[CP];
  {
    const float* src = q + ((int64_t)(t0 + (valid ? tok : 0)) * nh + (valid ? head : heads_block * hb)) * row;
#pragma unroll
    for (int c = 0; c < CP; ++c) {
      const int d = 32 * c + 8 * g;
      const float4 a = *(const float4*)(src + min(d, row - 8)), b = *(const float4*)(src + min(d, row - 8) + 4);
      const bool in = valid && d < row;
      qf[c] = in ? (u32x4_t){pack_bf16(a.x, a.y), pack_bf16(a.z, a.w), pack_bf16(b.x, b.y), pack_bf16(b.z, b.w)} : (u32x4_t){0, 0, 0, 0};
    }
  }
  // ---- the multiplying side ----
  uint32_t kat[4];                                          // this lane's place in a step for the pieces c, c + 4, ...
#pragma unroll
  for (int c = 0; c < 4; ++c) kat[c] = (uint32_t)((8 * (r >> 2) + (r & 3)) * SL * 16 + (((4 * c + g) ^ r) & 15) * 16);
  const uint32_t vat = KBYTES + r * 64 + ((g ^ (r >> 1)) & 3) * 16;
  float4_t acc[VB];
#pragma unroll
  for (int i = 0; i < VB; ++i) acc[i] = (float4_t){0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  int slot = 0;
  for (int step = 0; step < steps; ++step) {
    // this step has landed (the next one's loads may be under way) and every wave is done with the step before
    wait_for<NK + NV, 0>();
    __builtin_amdgcn_s_barrier();
    {
      const int into = slot == 0 ? LP_RING - 1 : slot - 1;
      fetch(into, page_next);
      page_next = page_of(step + 3);
    }
    const unsigned char* at = lds + slot * STEP;
    slot = slot + 1 == LP_RING ? 0 : slot + 1;
    const int kb = kb0 + 32 * step;
    // (a score's pieces in four sums, added in the order of the kernel above, whose scores these are bit for bit: in one sum
    // of all its pieces the rows were 1.9e-6 from 64 bits instead of 1.1e-6)
    float4_t st[2], piece[4][2];
    u32x4_t held[LP_AHEAD];                                 // (first keys, then values)
    auto key_piece = [&](int n) {
      const int c = n >> 1, tau = n & 1;
      return *(const u32x4_t*)(at + kat[c & 3] + (c >> 2) * 256 + tau * (4 * SL * 16));
    };
#pragma unroll
    for (int n = 0; n < LP_AHEAD; ++n) held[n] = key_piece(n);
#pragma unroll
    for (int n = 0; n < 2 * CP; ++n) {
      const int c = n >> 1, tau = n & 1;
      piece[c & 3][tau] = mfma32v(held[n % LP_AHEAD], qf[c], c < 4 ? (float4_t){0.f, 0.f, 0.f, 0.f} : piece[c & 3][tau]);
      if (n + LP_AHEAD < 2 * CP) held[n % LP_AHEAD] = key_piece(n + LP_AHEAD);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, LP_AHEAD, 0);
#pragma unroll
    for (int n = 0; n < 2 * CP; ++n) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      if (n + LP_AHEAD < 2 * CP) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
#pragma unroll
    for (int tau = 0; tau < 2; ++tau) st[tau] = piece[0][tau] + piece[1][tau] + piece[2][tau] + piece[3][tau];
#pragma unroll
    for (int i = 0; i < LP_AHEAD; ++i) held[i] = *(const u32x4_t*)(at + vat + i * 1024);
    float s[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] = st[j >> 2][j & 3] * scale_log2;
    if (kb < all_from || kb + 31 > pos0) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int key = kb + 8 * g + j;
        if (key < my_lo || key > my_pos) s[j] = -INFINITY;
      }
    }
    float top = fmaxf(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])), fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7])));
    // (the reference is the row's largest score so far, whose weight of 1 is exact in the first of its two terms: raised only
    // where a score exceeded it by 2^8, it cost rows that one key decides half as much precision again, 2.0e-6 for 1.3e-6)
    float alpha = 1.f;
    if (__any(top > m)) {                                    // (m = -inf: any key at all)
      const float m_new = fmaxf(m, row_max(top));
      alpha = m_new == -INFINITY ? 1.f : fast_exp2(m - m_new);
      m = m_new;
#pragma unroll
      for (int i = 0; i < VB; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] *= alpha;
    }
    const float m_safe = m == -INFINITY ? 0.f : m;
    u32x4_t hi, lo;
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float p0 = fast_exp2(s[2 * j] - m_safe), p1 = fast_exp2(s[2 * j + 1] - m_safe);
      sum += p0 + p1;
      hi[j] = pack_bf16(p0, p1);
      lo[j] = pack_bf16(p0 - __uint_as_float(hi[j] << 16), p1 - __uint_as_float(hi[j] & 0xffff0000u));
    }
    l = l * alpha + sum;
#pragma unroll
    for (int i = 0; i < VB; ++i) {
      acc[i] = mfma32v(held[i % LP_AHEAD], hi, acc[i]);
      acc[i] = mfma32v(held[i % LP_AHEAD], lo, acc[i]);
      if (i + LP_AHEAD < VB) held[i % LP_AHEAD] = *(const u32x4_t*)(at + vat + (i + LP_AHEAD) * 1024);
    }
#pragma unroll
    for (int i = 0; i < VB; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 1);
      if (i + LP_AHEAD < VB) __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
    }
  }
  wait_for<0>();                                            // (the steps fetched beyond the last land before the LDS is another's)
  const float total = row_sum(l);                           // (every lane takes part, whatever its row)
  if (!valid) return;
  const float inv = lm_scale(m, total, sinks, head) * lm_gate(gate, (int64_t)(t0 + tok) * gate_token + head);
  TO* dst = out + ((int64_t)(t0 + tok) * nh + head) * rank + 4 * g;
#pragma unroll
  for (int i = 0; i < VB; ++i)
    if (16 * i < rank) {
      if constexpr (sizeof(TO) == 4) *(float4_t*)(dst + 16 * i) = acc[i] * inv;
      else *(uint2*)(dst + 16 * i) = make_uint2(pack_bf16(acc[i][0] * inv, acc[i][1] * inv), pack_bf16(acc[i][2] * inv, acc[i][3] * inv));
    }
}

// Whether the kernel for steps of many tokens is built for these rows.
extern "C" int ts_latent_tiles_takes(int rank, int row) { return ts_latent_mfma_takes(rank, row) && rank <= 256 && row <= 384; }

// tiles as above, of at most LP_ROWS / min(heads, LP_ROWS) tokens.
extern "C" int ts_paged_attention_latent_tiles(void* out, int out_dtype, const float* q, const void* k_cache, const void* v_cache,
                                               const int32_t* block_tables, const int32_t* seq_of_token, const int32_t* positions,
                                               const int32_t* tiles, int num_tiles, int tile_tokens, int num_tokens, int nh, int rank,
                                               int rot, int page_size, int64_t kp, int64_t ks, int64_t vp, int64_t vd, int64_t v_slot,
                                               int max_blocks, float scale, int window, int page_run, const float* sinks,
                                               const float* gate, int64_t gate_token, hipStream_t stream) {
  if (num_tiles <= 0 || num_tokens <= 0) return TS_OK;
  const int row = rank + rot, heads_block = min(nh, LP_ROWS);
  if (!ts_latent_tiles_takes(rank, row) || nh <= 0 || page_size != 32 || v_slot != 1 || kp % 8 || ks % 8 || vp % 8 || vd % 8 || ks < row ||
      32 * ks >= (1 << 29) || rank * vd >= (1 << 29) || (((uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)q | (uintptr_t)out) & 15) ||
      max_blocks <= 0 || page_run < 0 || page_run > 16 || !tiles || tile_tokens < 1 || tile_tokens * heads_block > LP_ROWS)
    return TS_BAD_SHAPE;
  const dim3 grid(num_tiles, (nh + heads_block - 1) / heads_block);
  const float scale_log2 = scale * 1.4426950408889634f;
#define LP_LAUNCH(CP, VB, TO) \
  latent_attention_tiles_kernel<CP, VB, TO><<<grid, LP_WAVES * TS_WAVE, 0, stream>>>((TO*)out, q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, \
      block_tables, seq_of_token, positions, tiles, num_tiles, heads_block, nh, rank, row, kp, ks, vp, vd, max_blocks, scale_log2, window, \
      page_run, sinks, gate, gate_token)
#define LP_PICK(TO) \
  do { \
    if (row <= 128 && rank <= 128) LP_LAUNCH(4, 8, TO); \
    else if (row <= 256) LP_LAUNCH(8, 16, TO); \
    else LP_LAUNCH(12, 16, TO); \
  } while (0)
  if (out_dtype == 0) LP_PICK(float);
  else if (out_dtype == 1) LP_PICK(bf16_t);
  else return TS_BAD_DTYPE;
#undef LP_PICK
#undef LP_LAUNCH
  return ts_check_launch();
}

// ---- products per head on the matrix cores ---------------------------------------------------------------------
// y[t, h, n] = sum_k x[t, h, k] w[h][n][k] for bfloat16 matrices whose k runs along memory (a matrix stored [k, n]
// comes as a transposed copy), x 32-bit (rounded to bfloat16 once, as a projection's operand is) or bfloat16, 32-bit
// sums, times sigmoid(gate) on the way out if there is one. A wave makes RT blocks of 16 tokens by 64 columns of one head, a
// workgroup four waves' tokens: the matrix's rows are the instruction's rows, so that a lane ends with four adjacent columns of
// one token. Operands come straight from memory in 16-byte pieces; pieces past K are zeros of x against the matrix's last piece.
// What bounds it is loads and stores of 64 bytes of each of 16 rows: results are turned through shared memory into rows of 64
// columns (a twentieth less), and where that leaves enough waves a wave's pieces of the matrix serve two or four blocks of tokens.
// 2,048 tokens, 32 heads, 1, 2 and 4 blocks: K 64 by 256, 32-bit rows in and out 29.9, 26.9 and 23.6 us (31.3 before), K 256 by 64, bfloat16 23.6,
// 17.6 and 15.9 (24.0), of 32-bit rows 27.2, 21.7 and 27.3 (27.9); 300 tokens 7.7, 8.8 and 11.3. Every result is the same bits.
#define HM_TOKENS 64
#define HM_COLS 64

// BLOCKS 0: a workgroup takes one block of 16 tokens, and its waves 16 of the 64 columns each (with few tokens most waves had no token and the one
// that had them read the matrix by itself; which is better by the rule of ts_heads_gemm_few).
template <int BLOCKS, typename TX, typename TO>
__global__ void __launch_bounds__(LM_THREADS)
heads_gemm_mfma_kernel(TO* __restrict__ y, int64_t y_token, int64_t y_head, const TX* __restrict__ x, int64_t x_token,
                       int64_t x_head, const bf16_t* __restrict__ w, int64_t w_head, int64_t w_n, int num_tokens, int N, int K,
                       const float* __restrict__ gate, int64_t gate_token) {
  constexpr int RT = BLOCKS ? BLOCKS : 1, NB = BLOCKS ? HM_COLS / 16 : 1;      // blocks of 16 tokens and of 16 columns of a wave
  const int wave = wave_index(), lane = threadIdx.x & (TS_WAVE - 1);
  const int r = lane & 15, g = lane >> 4;
  const int h = blockIdx.y, n0 = blockIdx.z * HM_COLS + (BLOCKS ? 0 : 16 * wave);
  const int t0 = BLOCKS ? RT * (blockIdx.x * HM_TOKENS + 16 * wave) : 16 * blockIdx.x;
  const TX* xrow[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) xrow[rt] = x + (int64_t)min(t0 + 16 * rt + r, num_tokens - 1) * x_token + (int64_t)h * x_head;
  const bf16_t* wh = w + (int64_t)h * w_head;
  float4_t acc[RT][NB];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[rt][nb] = (float4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll(BLOCKS ? 4 : 8)
  for (int k0 = 0; k0 < K; k0 += 32) {
    const int k = k0 + 8 * g, kc = min(k, K - 8);
    uint4 b[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      if constexpr (sizeof(TX) == 4) {
        const float4 lo = *(const float4*)(xrow[rt] + kc), hi = *(const float4*)(xrow[rt] + kc + 4);
        b[rt] = make_uint4(pack_bf16(lo.x, lo.y), pack_bf16(lo.z, lo.w), pack_bf16(hi.x, hi.y), pack_bf16(hi.z, hi.w));
      } else {
        b[rt] = *(const uint4*)(xrow[rt] + kc);
      }
      if (k >= K) b[rt] = make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int n = min(n0 + 16 * nb + r, N - 1);
      const uint4 a = *(const uint4*)(wh + (int64_t)n * w_n + kc);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) acc[rt][nb] = mfma32(a, b[rt], acc[rt][nb]);
    }
  }
  // whole fours of columns go out in one store of a lane; 16 lanes' side by side, turned through shared memory by the wave, where
  // that pays (below: 16 tokens, 32 heads of 64 by 256 3.9 us as they are and 4.0 turned, 200 tokens, 24 of 40 by 100 with bfloat16
  // results 4.0 and 4.1, 32-bit ones 4.2 and 4.1)
  if (N % 4 == 0 && ((y_token | y_head) & 3) == 0 && ((uintptr_t)y & (4 * sizeof(TO) - 1)) == 0) {
    auto put = [&](int t, int n, float4_t v) {
      if (t >= num_tokens || n >= N) return;
      if (gate) {
        const float* gr = gate + (int64_t)t * gate_token + (int64_t)h * N + n;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = v[j] / (1.0f + expf(-gr[j]));
      }
      TO* yrow = y + (int64_t)t * y_token + (int64_t)h * y_head + n;
      if constexpr (sizeof(TO) == 4) *(float4_t*)yrow = v;
      else *(uint2*)yrow = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
    };
    __shared__ __attribute__((aligned(16))) float4_t turn[LM_WAVES][16][HM_COLS / 4 + 1];
    const bool turned = RT > 1 || (BLOCKS && sizeof(TO) == 4 && num_tokens >= HM_TOKENS);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      if (!turned) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) put(t0 + 16 * rt + r, n0 + 16 * nb + 4 * g, acc[rt][nb]);
        continue;
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) turn[wave][r][4 * nb + g] = acc[rt][nb];
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < 4; ++i) put(t0 + 16 * rt + 4 * i + g, n0 + 4 * r, turn[wave][4 * i + g][r]);
      __builtin_amdgcn_wave_barrier();
    }
    return;
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int t = t0 + 16 * rt + r;
    if (t >= num_tokens) continue;
    TO* yrow = y + (int64_t)t * y_token + (int64_t)h * y_head;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + 16 * nb + 4 * g + j;
      if (n >= N) continue;
      float v = acc[rt][nb][j];
      if (gate) v = v / (1.0f + expf(-gate[(int64_t)t * gate_token + (int64_t)h * N + n]));
      Num<TO>::st(yrow + n, v);
    }
  }
}

// The blocks of 16 tokens that a wave takes: two from 512 workgroups of one on, four from 2,048 (of bfloat16 rows, whose loads are
// half as many, from 1,024); one for reductions below 64, whose waves are over at once (40 by 100, 24 heads, 1,000 tokens 6.6 us, 7.2
// and 8.6), and for tokens that one workgroup of one holds, most of whose waves would have none (128 heads of 128 by 512, bfloat16
// rows, 5 tokens 10.4 us and in four blocks 12.7, 64 tokens 13.9 and 15.8, 100 tokens 24.1 and 17.2).
extern "C" int ts_heads_gemm_blocks(int num_tokens, int heads, int N, int K, int x_dtype) {
  const int64_t groups = (int64_t)((num_tokens + HM_TOKENS - 1) / HM_TOKENS) * heads * ((N + HM_COLS - 1) / HM_COLS);
  if (K < 64 || num_tokens <= HM_TOKENS || groups < 512) return 1;
  return groups >= 2048 || (groups >= 1024 && x_dtype == 1) ? 4 : 2;
}

// Whether a workgroup of one block of tokens a wave is better made one of 16 tokens whose waves share out the columns: where these are few workgroups,
// or one to a head's 64 columns. us, before and so: 8 tokens, 32 heads, K 256 by 64, bfloat16 rows 5.9 and 3.3, K 64 by 256, 32-bit rows 3.3 and 2.5,
// 128 heads of 512 by 128 12.1 and 6.8, 16 tokens of 128 by 512, 32-bit 11.7 and 8.2. From so many workgroups on each reads the matrix again for too few
// tokens: K 64 by 256, 32 heads, 48 tokens (384 of them) 3.7 and 3.4, 64 tokens (512, left) 3.8 and 3.9; 16 heads of 128 by 512, 33 tokens (384)
// 5.0 and 5.1, 65 tokens (640, left) 5.6 and 6.6; 128 heads of 128 by 512, 17 tokens (2,048, left) 11.8 and 14.0; K 256 by 64, 200 tokens (416, left) 7.5 and 5.9.
static bool ts_heads_gemm_few(int num_tokens, int heads, int N) {
  return num_tokens <= 16 || (int64_t)((num_tokens + 15) / 16) * heads * ((N + HM_COLS - 1) / HM_COLS) <= 384;
}

// w: bfloat16 [heads][N][K] with K along memory (stride w_n between rows, a multiple of 8; K a multiple of 8);
// x rows 16-byte aligned.
extern "C" int ts_heads_gemm_mfma(void* y, int y_dtype, int64_t y_token, int64_t y_head, const void* x, int x_dtype,
                                  int64_t x_token, int64_t x_head, const void* w, int64_t w_head, int64_t w_n, int num_tokens,
                                  int heads, int N, int K, const float* gate, int64_t gate_token, hipStream_t stream) {
  if (num_tokens <= 0) return TS_OK;
  const int x_size = x_dtype == 0 ? 4 : 2;
  if (heads <= 0 || heads > 65535 || N <= 0 || K < 8 || K % 8 || w_n % 8 || w_head % 8 || ((uintptr_t)w & 15) ||
      ((uintptr_t)x & 15) || (x_token * x_size) % 16 || (x_head * x_size) % 16 || (N + HM_COLS - 1) / HM_COLS > 65535)
    return TS_BAD_SHAPE;
  int blocks = ts_heads_gemm_blocks(num_tokens, heads, N, K, x_dtype);
  if (blocks == 1 && ts_heads_gemm_few(num_tokens, heads, N)) blocks = 0;
  const int tokens = blocks ? blocks * HM_TOKENS : 16;
  const dim3 grid((num_tokens + tokens - 1) / tokens, heads, (N + HM_COLS - 1) / HM_COLS);
#define HM_GO(RT, TX, TO) \
  heads_gemm_mfma_kernel<RT, TX, TO><<<grid, LM_THREADS, 0, stream>>>((TO*)y, y_token, y_head, (const TX*)x, x_token, x_head, \
      (const bf16_t*)w, w_head, w_n, num_tokens, N, K, gate, gate_token)
#define HM_LAUNCH(TX, TO) \
  do { \
    if (blocks == 0) HM_GO(0, TX, TO); \
    else if (blocks == 1) HM_GO(1, TX, TO); \
    else if (blocks == 2) HM_GO(2, TX, TO); \
    else HM_GO(4, TX, TO); \
  } while (0)
  if (x_dtype == 0 && y_dtype == 0) HM_LAUNCH(float, float);
  else if (x_dtype == 0 && y_dtype == 1) HM_LAUNCH(float, bf16_t);
  else if (x_dtype == 1 && y_dtype == 0) HM_LAUNCH(bf16_t, float);
  else if (x_dtype == 1 && y_dtype == 1) HM_LAUNCH(bf16_t, bf16_t);
  else return TS_BAD_DTYPE;
#undef HM_LAUNCH
#undef HM_GO
  return ts_check_launch();
}
