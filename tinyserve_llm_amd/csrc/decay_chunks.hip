// Linear attention with a decay per key channel over long portions, in chunks of 64 tokens on the matrix cores, in
// 32 bits or more (the walk token by token is in decay_scan.hip, with the two orders of decay and read). With W(s, t] the product of
// the decays of a channel over the tokens after s up to t, S0 the state before the chunk and tokens counted in the chunk:
//     o_t = sum_d q_td W(start, t] S0_d + sum_{s <= t} A_ts v_s,   A_ts = sum_d q_td k_sd W(s, t]
//     S   = W(start, end] S0 + sum_s (k_s W(s, end]) v_s^T
// (read first: the decay of t itself is left out of o_t's products, and A_tt has the bonus in the decay's place).
//   * `decay_chunk_sums`: what a chunk adds to the state, a workgroup per (chunk, head, 256 value columns).
//   * `decay_chunk_scan`: over a request's chunks in order, element by element, the state before every chunk.
//   * `decay_chunk_out`: A, then the read-outs.
// No decay is ever divided by: a product over many tokens may be 0 in 32 bits. A chunk is cut into four blocks of 16 tokens.
// Pairs of tokens in different blocks take their product apart at the blocks' edges (up to the end of s's block, the whole
// blocks between, from the start of t's block: all at most 1); pairs in one block are walked, the running k_s W(s, t] kept in
// registers, as the token-by-token kernel does it.
// What bounds it: the walk is a chain of tokens, 150 ns each however few heads there are (two
// requests of 2,048 tokens together: 532 µs for 8 heads of 128 x 256, 444 µs for 32 of 64 x 64; in
// chunks 130 and 130 µs). The same tokens in chunks are 3 and 2 GFLOP of 32-bit matrix instructions (157 TFLOP/s) beside the
// states' trips through memory (34 and 17 MB, three times): what is left is the chain of a workgroup's phases. Error against
// 64 bits (root mean square, 2,048 tokens): 1.7e-7 for the first heads (the walk: 7.0e-7), 0.81e-7 for the second (0.91e-7),
// of the states 1.5e-7 (7.8e-7) and 5.6e-8 (5.8e-8). A 32-bit instruction takes one number a lane
// and operand, so operands are fetched as 16 bytes of four steps where the order of the sum allows it, and a wave keeps all
// 64 tokens of its value columns so that every number of the state is read once.
#include <type_traits>

#include "chunk_ops.h"

#define DC_THREADS 256
#define DC_BLOCK 16             // tokens of a block

struct DecayChunks {
  float *out, *buf, *totals, *logs, *states;
  const float *q, *k, *v, *z, *z_bias, *bonus;
  int64_t q_stride, k_stride, v_stride, z_stride, slot_stride;
  const int32_t *chunks, *chunk_cu, *state_slots;
  int heads, vdim, form;
  float inv_tau, q_scale;
};

static __device__ __forceinline__ float4_t mfma_f32(float a, float b, float4_t acc) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0); }

static __device__ __forceinline__ float dc_fma(float a, float b, float c) { return fmaf(a, b, c); }
static __device__ __forceinline__ double dc_fma(float a, float b, double c) { return fma((double)a, (double)b, c); }

// The logarithm of one token's decay: of sigmoid(z)^(1 / tau) or exp(-exp(z)) (0 past a chunk's end, where q, k and v count as 0). A decay near 1 loses most of what tells it from 1 when it is stored in 32 bits; its logarithm does not,
// so products of decays are exponentials of sums of these (all of one sign: nothing cancels).
static __device__ __forceinline__ float dc_log(float z, int form, float inv_tau) {
  return form == 0 ? (fminf(z, 0.f) - log1pf(expf(-fabsf(z)))) * inv_tau : -expf(z);
}

// A channel's numbers of the 16 tokens of block b, in one go (no load waits for a test; tokens past the chunk's end: its last
// one, for which `dc_mask` puts 0). `src`: the chunk's first token, the same for every thread; places as 32-bit offsets from there.
static __device__ __forceinline__ void dc_fetch(float (&x)[DC_BLOCK], const float* src, int stride, int col, int b, int len) {
#pragma unroll
  for (int t = 0; t < DC_BLOCK; ++t) x[t] = src[(uint32_t)(min(b * DC_BLOCK + t, len - 1) * stride + col)];
}
static __device__ __forceinline__ void dc_mask(float (&x)[DC_BLOCK], int b, int len) {
#pragma unroll
  for (int t = 0; t < DC_BLOCK; ++t)
    if (b * DC_BLOCK + t >= len) x[t] = 0.f;
}
static __device__ __forceinline__ void dc_column(float (&x)[DC_BLOCK], const float* src, int stride, int col, int b, int len) {
  dc_fetch(x, src, stride, col, b, len);
  dc_mask(x, b, len);
}
static __device__ __forceinline__ void dc_log_column(float (&l)[DC_BLOCK], float bias, int form, float inv_tau, int b, int len) {
#pragma unroll
  for (int t = 0; t < DC_BLOCK; ++t) l[t] = b * DC_BLOCK + t < len ? dc_log(l[t] + bias, form, inv_tau) : 0.f;
}

// VT: 16-column tiles of a wave (four waves side by side). A workgroup takes DP of the head's channels: with all 128 in one, two
// requests of 2,048 tokens together were a workgroup a compute unit, whose loads and logarithms nothing hid (8 heads of
// 128 x 256: 45.6 µs, 37.7 in halves and 35.1 since these ask for both their columns at once, each element's sums in the same order; heads of
// 64 x 64 are one workgroup as before).
template <int D, int VT>
__global__ void __launch_bounds__(DC_THREADS) decay_chunk_sums_kernel(const DecayChunks a) {
  constexpr int DP = D < 64 ? D : 64, PARTS = D / DP;
  constexpr int ROW = DP + 16;                              // (four neighbouring tokens' rows 16 banks apart)
  __shared__ float k_s[SS_L][ROW], p_s[4][DP];
  const int d0 = blockIdx.z % PARTS * DP, vz = blockIdx.z / PARTS;
  const int c = blockIdx.x, h = blockIdx.y, tok0 = a.chunks[4 * c], len = a.chunks[4 * c + 1];
  // a thread takes a channel of a block (or two): the block's sum of logarithms, then k W(s, end] from the chunk's end back
  constexpr int ITEMS = 4 * DP;
  static_assert(ITEMS <= DC_THREADS, "a channel of a block a thread");
  const int d = threadIdx.x % DP, b0 = threadIdx.x / DP;
  const bool takes = ITEMS == DC_THREADS || threadIdx.x < ITEMS;
  float l[DC_BLOCK], kk[DC_BLOCK];
  // (both columns are asked for before either is looked at: the compiler otherwise waited for all of z before it asked for k, 32
  // heads of 64 x 64, 1,500 tokens 65.4 µs the three kernels and now 64.2, 8 of 128 x 256, 2,048 tokens 82.9 and 81.2)
  dc_fetch(l, a.z + (int64_t)tok0 * a.z_stride + h * D + d0, (int)a.z_stride, d, b0 % 4, len);
  dc_fetch(kk, a.k + (int64_t)tok0 * a.k_stride + h * D + d0, (int)a.k_stride, d, b0 % 4, len);
  __builtin_amdgcn_sched_barrier(0);
  dc_mask(kk, b0 % 4, len);
  if (takes) {
    dc_log_column(l, a.z_bias[h * D + d0 + d], a.form, a.inv_tau, b0, len);
    float all = 0.f;
#pragma unroll
    for (int t = DC_BLOCK - 1; t >= 0; --t) {
      all += l[t];
      if (vz == 0 && b0 * DC_BLOCK + t < len) a.logs[((int64_t)(tok0 + b0 * DC_BLOCK + t) * a.heads + h) * D + d0 + d] = l[t];
    }
    p_s[b0][d] = all;
  }
  __syncthreads();
  if (takes) {
    float after = 0.f;
    for (int m = 3; m > b0; --m) after += p_s[m][d];
#pragma unroll
    for (int t = DC_BLOCK - 1; t >= 0; --t) {
      k_s[b0 * DC_BLOCK + t][d] = kk[t] * expf(after);
      after += l[t];
    }
    if (b0 == 0 && vz == 0) a.totals[((int64_t)c * a.heads + h) * D + d0 + d] = expf(after);
  }
  __syncthreads();
  const int lane = threadIdx.x % TS_WAVE, r = lane % 16, g = lane / 16, wave = wave_index();
  const int v0 = vz * (64 * VT) + wave * (16 * VT);
  float4_t acc[DP / 16][VT];
#pragma unroll
  for (int i = 0; i < DP / 16; ++i)
#pragma unroll
    for (int j = 0; j < VT; ++j) acc[i][j] = (float4_t){0.f, 0.f, 0.f, 0.f};
  const float* v = a.v + (int64_t)tok0 * a.v_stride + h * a.vdim + v0 + r;
  float vv[2][4][VT];
  auto fetch = [&](int b, float (&x)[4][VT]) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int at = b * DC_BLOCK + 4 * s + g;
#pragma unroll
      for (int j = 0; j < VT; ++j) {
        const float y = v[(int64_t)min(at, len - 1) * a.v_stride + 16 * j];
        x[s][j] = at < len ? y : 0.f;
      }
    }
  };
  fetch(0, vv[0]);
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    if (b < 3) fetch(b + 1, vv[(b + 1) & 1]);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < DP / 16; ++i) {
        const float ka = k_s[b * DC_BLOCK + 4 * s + g][16 * i + r];
#pragma unroll
        for (int j = 0; j < VT; ++j) acc[i][j] = mfma_f32(ka, vv[b & 1][s][j], acc[i][j]);
      }
  }
  float* dst = a.buf + (((int64_t)c * a.heads + h) * D + d0) * a.vdim + v0 + r;
#pragma unroll
  for (int i = 0; i < DP / 16; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int j = 0; j < VT; ++j) dst[(int64_t)(16 * i + 4 * g + e) * a.vdim + 16 * j] = acc[i][j][e];
}

// A thread per four numbers of a head's state: over a request's chunks in order, what the chunk adds makes room for the state
// before the chunk. Requests without chunks keep their state as it is.
__global__ void __launch_bounds__(DC_THREADS) decay_chunk_scan_kernel(const DecayChunks a, int dim) {
  const int seq = blockIdx.x, h = blockIdx.y, per_head = dim * a.vdim;
  const int begin = a.chunk_cu[seq], end = a.chunk_cu[seq + 1];
  const int e = 4 * (blockIdx.z * DC_THREADS + threadIdx.x);
  if (begin >= end || e >= per_head) return;
  float* st = a.states + (int64_t)a.state_slots[seq] * a.slot_stride + (int64_t)h * per_head + e;
  float4 S = *(const float4*)st;
  float* p = a.buf + ((int64_t)begin * a.heads + h) * per_head + e;
  const float* keep_at = a.totals + ((int64_t)begin * a.heads + h) * dim + e / a.vdim;
  const int64_t next = (int64_t)a.heads * per_head, next_keep = (int64_t)a.heads * dim;
  constexpr int AHEAD = 8;                                   // chunks whose sums are on their way together
  for (int c = begin; c < end; c += AHEAD, p += AHEAD * next, keep_at += AHEAD * next_keep) {
    float4 add[AHEAD];
    float keep[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      const int k = min(i, end - 1 - c);
      add[i] = *(const float4*)(p + k * next);
      keep[i] = keep_at[k * next_keep];
    }
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
      if (c + i < end) {
        *(float4*)(p + i * next) = S;
        S.x = fmaf(keep[i], S.x, add[i].x);
        S.y = fmaf(keep[i], S.y, add[i].y);
        S.z = fmaf(keep[i], S.z, add[i].z);
        S.w = fmaf(keep[i], S.w, add[i].w);
      }
  }
  *(float4*)st = S;
}

// Channels go through shared memory DH at a time (64 at most: two workgroups a compute unit whatever the head's size).
template <int D, int VT, bool READ_FIRST>
__global__ void __launch_bounds__(DC_THREADS, 2) decay_chunk_out_kernel(const DecayChunks a) {
  constexpr int DH = D < 64 ? D : 64, ROW = DH + 4, AROW = SS_L + 4;      // (16 rows of 16-byte pieces in different banks)
  // Sums are cut short: 32-bit products run one after the other through a matrix instruction's accumulator, and a long run loses
  // more than the walk's sums over a few channels a lane. So every 16 channels (or tokens) have PARTS sums that start
  // from nothing, which are added to one of SETS totals (in runs of 32 products: 1.05e-7, the walk 0.91e-7).
  constexpr int SETS = VT == 4 ? 1 : 2, PARTS = VT == 4 ? 1 : 2;
  constexpr float4_t NONE = {0.f, 0.f, 0.f, 0.f};
  __shared__ __attribute__((aligned(16))) float q_s[SS_L][ROW], k_s[SS_L][ROW], w_s[SS_L][ROW], a_s[SS_L][AROW], p_s[4][DH];
  const int c = blockIdx.x, h = blockIdx.y, tok0 = a.chunks[4 * c], len = a.chunks[4 * c + 1];
  const int lane = threadIdx.x % TS_WAVE, wave = wave_index();
  int r = lane % 16, g = lane / 16;
  const int v0 = blockIdx.z * (64 * VT) + wave * (16 * VT);
  const int block = threadIdx.x / DH % 4;                   // this thread's block of tokens,
  int col = threadIdx.x % DH;                               // and its channel of DH
  const bool takes = threadIdx.x < 4 * DH;
  float4_t o[SETS][4][VT];
#pragma unroll
  for (int n = 0; n < SETS; ++n)
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int j = 0; j < VT; ++j) o[n][t][j] = (float4_t){0.f, 0.f, 0.f, 0.f};
  constexpr int AHEAD = VT == 4 ? 2 : DH / 16;              // rounds of 16 rows of the state on their way
  float sv[AHEAD][4][VT], vv[2][4][VT];
  const float* v = a.v + (int64_t)tok0 * a.v_stride + h * a.vdim + v0;
  auto fetch_values = [&](int s, float (&x)[4][VT]) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int j = 0; j < VT; ++j) x[e][j] = v[(uint32_t)(min(s * DC_BLOCK + 4 * g + e, len - 1) * (int)a.v_stride + r + 16 * j)];
  };
#pragma unroll 1
  for (int d0 = 0; d0 < D; d0 += DH) {
    asm volatile("" : "+v"(r), "+v"(g), "+v"(col));         // (or every place that depends on them is kept in registers over the loop)
    float l[DC_BLOCK];
    {
      float qq[DC_BLOCK], kk[DC_BLOCK];
      dc_column(l, a.logs + ((int64_t)tok0 * a.heads + h) * D + d0, a.heads * D, col, block, len);
      dc_column(qq, a.q + (int64_t)tok0 * a.q_stride + h * D + d0, (int)a.q_stride, col, block, len);
      dc_column(kk, a.k + (int64_t)tok0 * a.k_stride + h * D + d0, (int)a.k_stride, col, block, len);
      if (d0 > 0) __syncthreads();                          // (the channels before have been read)
      if (takes) {
        float all = 0.f;
#pragma unroll
        for (int t = 0; t < DC_BLOCK; ++t) {
          q_s[block * DC_BLOCK + t][col] = qq[t] * a.q_scale;
          k_s[block * DC_BLOCK + t][col] = kk[t];
          w_s[block * DC_BLOCK + t][col] = expf(l[t]);
          all += l[t];
        }
        p_s[block][col] = expf(all);
      }
    }
    // the state's rows that the read-outs begin with are asked for here, ahead of everything they wait for
    const float* S = a.buf + (((int64_t)c * a.heads + h) * D + d0) * a.vdim + v0;
    auto fetch_state = [&](int i, float (&x)[4][VT]) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < VT; ++j) x[e][j] = S[(uint32_t)((16 * i + 4 * g + e) * a.vdim + r + 16 * j)];
    };
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) fetch_state(i, sv[i]);
    __syncthreads();
    {
      // A of the pairs inside a block, a wave a block: a lane keeps a quarter of k_s W(s, t] of its s = r and goes through t
      const int t0 = wave * DC_BLOCK;
      float4 kp[DH / 16];
      float own = 0.f;                                      // (read first) the bonus in the decay's place
#pragma unroll
      for (int i = 0; i < DH / 16; ++i) kp[i] = *(const float4*)&k_s[t0 + r][16 * i + 4 * g];
      if constexpr (READ_FIRST) {
        float4 part = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int i = 0; i < DH / 16; ++i) {
          const float4 q4 = *(const float4*)&q_s[t0 + r][16 * i + 4 * g], u4 = *(const float4*)(a.bonus + h * D + d0 + 16 * i + 4 * g);
          part.x = fmaf(q4.x * u4.x, kp[i].x, part.x), part.y = fmaf(q4.y * u4.y, kp[i].y, part.y);
          part.z = fmaf(q4.z * u4.z, kp[i].z, part.z), part.w = fmaf(q4.w * u4.w, kp[i].w, part.w);
        }
        own = (part.x + part.y) + (part.z + part.w);
      }
      // (read first: these pairs and `own` are most of a row, and the walk's sums of a few channels a lane are good to 0.91e-7; in
      // 64 bits the rows are good to 0.81e-7, in 32 to 0.98e-7)
      using sum_t = std::conditional_t<READ_FIRST, double, float>;
      for (int t = 0; t < DC_BLOCK; ++t) {
        sum_t part[4] = {0, 0, 0, 0};
        const bool later = t > r;
#pragma unroll
        for (int i = 0; i < DH / 16; ++i) {
          const float4 q4 = *(const float4*)&q_s[t0 + t][16 * i + 4 * g], w4 = *(const float4*)&w_s[t0 + t][16 * i + 4 * g];
          float4& x = kp[i];
          const float4 y = make_float4(x.x * w4.x, x.y * w4.y, x.z * w4.z, x.w * w4.w);
          const float4 then = later ? y : x;
          if constexpr (!READ_FIRST) x = then;
          part[0] = dc_fma(q4.x, x.x, part[0]), part[1] = dc_fma(q4.y, x.y, part[1]);
          part[2] = dc_fma(q4.z, x.z, part[2]), part[3] = dc_fma(q4.w, x.w, part[3]);
          if constexpr (READ_FIRST) x = then;
        }
        sum_t sum = (part[0] + part[1]) + (part[2] + part[3]);
        if (READ_FIRST && t == r) sum = own;
        sum += __shfl_xor(sum, 16, TS_WAVE);
        sum += __shfl_xor(sum, 32, TS_WAVE);
        if (g == 0) a_s[t0 + t][t0 + r] = t >= r ? (d0 > 0 ? a_s[t0 + t][t0 + r] : 0.f) + (float)sum : 0.f;
      }
    }
    __syncthreads();
    // from here on q W(block's start, t] and k W(s, block's end]
    if (takes) {
      float before = 0.f, after = 0.f;
#pragma unroll
      for (int t = 0; t < DC_BLOCK; ++t) {
        if constexpr (!READ_FIRST) before += l[t];
        q_s[block * DC_BLOCK + t][col] *= expf(before);
        if constexpr (READ_FIRST) before += l[t];
        k_s[block * DC_BLOCK + DC_BLOCK - 1 - t][col] *= expf(after);
        after += l[DC_BLOCK - 1 - t];
      }
    }
    __syncthreads();
    // A of pairs in different blocks: six blocks of 16 x 16, two a wave for the first two waves and one for the others
    for (int n = wave; n < 6; n += 4) {
      const int jb = n < 3 ? 3 : n < 5 ? 2 : 1, ib = n < 3 ? n : n < 5 ? n - 3 : 0;      // (3,0) (3,1) (3,2) (2,0) (2,1) (1,0)
      float4_t part[DH / 8];
#pragma unroll
      for (int i = 0; i < DH / 16; ++i) {
        const float4 q4 = *(const float4*)&q_s[jb * DC_BLOCK + r][16 * i + 4 * g];
        float4 k4 = *(const float4*)&k_s[ib * DC_BLOCK + r][16 * i + 4 * g];
        for (int m = ib + 1; m < jb; ++m) {
          const float4 p4 = *(const float4*)&p_s[m][16 * i + 4 * g];
          k4.x *= p4.x, k4.y *= p4.y, k4.z *= p4.z, k4.w *= p4.w;
        }
        part[2 * i] = mfma_f32(q4.y, k4.y, mfma_f32(q4.x, k4.x, NONE));
        part[2 * i + 1] = mfma_f32(q4.w, k4.w, mfma_f32(q4.z, k4.z, NONE));
      }
#pragma unroll
      for (int n2 = DH / 16; n2 > 0; n2 /= 2)
#pragma unroll
        for (int i = 0; i < n2; ++i) part[i] += part[i + n2];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float& x = a_s[jb * DC_BLOCK + 4 * g + e][ib * DC_BLOCK + r];
        x = (d0 > 0 ? x : 0.f) + part[0][e];
      }
    }
    // the state's share, 16 channels a round
#pragma unroll
    for (int i = 0; i < DH / 16; ++i) {
      float4 upto = make_float4(1.f, 1.f, 1.f, 1.f);        // the blocks before t's
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const float4 q4 = *(const float4*)&q_s[t * DC_BLOCK + r][16 * i + 4 * g];
        const float qq[4] = {q4.x * upto.x, q4.y * upto.y, q4.z * upto.z, q4.w * upto.w};
        float4_t part[PARTS][VT];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int j = 0; j < VT; ++j) {
            float4_t& acc = part[e * PARTS / 4][j];
            acc = mfma_f32(qq[e], sv[i % AHEAD][e][j], e * PARTS % 4 ? acc : NONE);
          }
#pragma unroll
        for (int j = 0; j < VT; ++j) o[i % SETS][t][j] += PARTS == 2 ? part[0][j] + part[PARTS - 1][j] : part[0][j];
        const float4 p4 = *(const float4*)&p_s[t][16 * i + 4 * g];
        upto.x *= p4.x, upto.y *= p4.y, upto.z *= p4.z, upto.w *= p4.w;
      }
      if (i + AHEAD < DH / 16) fetch_state(i + AHEAD, sv[i % AHEAD]);
    }
  }
  fetch_values(0, vv[0]);
  __syncthreads();
  // the chunk's own share (values past its end count as 0)
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    if (s < 3) fetch_values(s + 1, vv[(s + 1) & 1]);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int j = 0; j < VT; ++j) vv[s & 1][e][j] = s * DC_BLOCK + 4 * g + e < len ? vv[s & 1][e][j] : 0.f;
#pragma unroll
    for (int t = s; t < 4; ++t) {
      const float4 a4 = *(const float4*)&a_s[t * DC_BLOCK + r][s * DC_BLOCK + 4 * g];
      const float aa[4] = {a4.x, a4.y, a4.z, a4.w};
      float4_t part[PARTS][VT];
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < VT; ++j) {
          float4_t& acc = part[e * PARTS / 4][j];
          acc = mfma_f32(aa[e], vv[s & 1][e][j], e * PARTS % 4 ? acc : NONE);
        }
#pragma unroll
      for (int j = 0; j < VT; ++j) o[s % SETS][t][j] += PARTS == 2 ? part[0][j] + part[PARTS - 1][j] : part[0][j];
    }
  }
  float* dst = a.out + (int64_t)tok0 * a.heads * a.vdim + h * a.vdim + v0 + r;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int at = t * DC_BLOCK + 4 * g + e;
      if (at < len)
#pragma unroll
        for (int j = 0; j < VT; ++j) {
          dst[(int64_t)at * a.heads * a.vdim + 16 * j] = SETS == 2 ? o[0][t][j][e] + o[SETS - 1][t][j][e] : o[0][t][j][e];
        }
    }
}

template <int D, int VT>
static int launch_decay_chunks(const DecayChunks& a, int num_chunks, int num_seqs, hipStream_t stream) {
  const dim3 grid(num_chunks, a.heads, a.vdim / (64 * VT));
  decay_chunk_sums_kernel<D, VT><<<dim3(num_chunks, a.heads, grid.z * (D < 64 ? 1 : D / 64)), DC_THREADS, 0, stream>>>(a);
  decay_chunk_scan_kernel<<<dim3(num_seqs, a.heads, (D * a.vdim / 4 + DC_THREADS - 1) / DC_THREADS), DC_THREADS, 0, stream>>>(a, D);
  if (a.bonus) decay_chunk_out_kernel<D, VT, true><<<grid, DC_THREADS, 0, stream>>>(a);
  else decay_chunk_out_kernel<D, VT, false><<<grid, DC_THREADS, 0, stream>>>(a);
  return ts_check_launch();
}

// Heads of 32, 64 or 128 key channels and a multiple of 64 value columns; q, k, v, z rows of 32-bit numbers that may lie
// apart. chunks: int32 [chunks, 4] (first token, tokens, request, 1 if the request's last); chunk_cu: int32 [requests + 1].
// buf: float32 [chunks, heads, dim, vdim], totals: [chunks, heads, dim], logs: [tokens, heads dim] (the decays' logarithms, made by
// the first kernel for the last). bonus (or null): [heads, dim], the read-first order.
extern "C" int ts_decay_chunks(float* out, const float* q, int64_t q_stride, const float* k, int64_t k_stride, const float* v,
                               int64_t v_stride, const float* z, int64_t z_stride, const float* z_bias, const float* bonus, float* states,
                               int64_t slot_stride, const int32_t* chunks, const int32_t* chunk_cu, const int32_t* state_slots, float* buf,
                               float* totals, float* logs, int num_chunks, int num_seqs, int heads, int dim, int vdim, float q_scale, int form,
                               float tau, hipStream_t stream) {
  if (num_chunks <= 0 || num_seqs <= 0) return TS_OK;
  if (heads <= 0 || heads > 65535 || (dim != 32 && dim != 64 && dim != 128) || vdim <= 0 || vdim % 64 || vdim > 65536 ||
      slot_stride < (int64_t)heads * dim * vdim || slot_stride % 4 || (form != 0 && form != 1) || !(tau > 0.f) ||
      (((uintptr_t)states | (uintptr_t)buf) & 15) || (bonus && ((uintptr_t)bonus & 15)))
    return TS_BAD_SHAPE;
  const int64_t widest = (1 << 23);                         // (a chunk's places go by 32-bit offsets)
  if (q_stride > widest || k_stride > widest || v_stride > widest || z_stride > widest || (int64_t)heads * dim > widest) return TS_TOO_LARGE;
  const DecayChunks a = {out, buf, totals, logs, states, q, k, v, z, z_bias, bonus, q_stride, k_stride, v_stride, z_stride, slot_stride,
                         chunks, chunk_cu, state_slots, heads, vdim, form, 1.f / tau, q_scale};
#define DC_GO(D) \
  return vdim % 256 == 0 ? launch_decay_chunks<D, 4>(a, num_chunks, num_seqs, stream) \
       : vdim % 128 == 0 ? launch_decay_chunks<D, 2>(a, num_chunks, num_seqs, stream) : launch_decay_chunks<D, 1>(a, num_chunks, num_seqs, stream);
  switch (dim) {
    case 32: DC_GO(32)
    case 64: DC_GO(64)
    default: DC_GO(128)
  }
#undef DC_GO
}
