// Split-key paged attention on the matrix cores for tokens that each bring one query (decoding),
// bfloat16. A workgroup takes one (token, key/value head, chunk of keys) and serves all query heads
// of that key/value head's group; its waves (up to 8; 4 for heads wider than 64 where a wave has more than one step) take the chunk's
// 32-key steps in turn:
//     S^T[key, head] = K[key, :] · Q[head, :]      v_mfma_f32_16x16x32_bf16, keys as rows
//     online softmax per head (32-bit), P = 2^(S - m)
//     O[head, :]    += P[head, key] · V[key, :]
// The result layout of the first product is the operand layout of the second, so P never leaves
// its registers. Keys are read as 16-byte pieces of their rows; values are read from pages that
// hold them transposed ([head_dim, page_size] per head), so that the eight consecutive keys an
// operand needs lie side by side in memory. The waves' partial results meet in LDS. With one chunk
// per token (few tokens, contexts short enough for one workgroup to stream) the workgroup
// normalises and writes the output itself. Otherwise a chunk's unnormalised output with its running
// max and sum goes to a 32-bit workspace, and a second kernel combines the chunks of a token in
// ascending order. Chunk boundaries are multiples of the chunk size counted from position 0.
// (The chunk's walk is attention_decode.h's, which a step with prompts beside the decoding tokens takes too: attn_step_kernel in attention_prefill.hip.)
#include "attention_decode.h"

template <int HD, bool ONE, bool GENERAL, bool ONCE>
__global__ void __launch_bounds__(DEC_WAVES_FOR(HD, ONE) * TS_WAVE)
attn_decode_mfma_kernel(bf16_t* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml,
                        const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
                        const int32_t* __restrict__ block_tables, const int32_t* __restrict__ seq_of_token,
                        const int32_t* __restrict__ positions, int nh, int G, int page_size, int page_shift, int page_run,
                        int64_t kp, int64_t ks, int64_t kh, int64_t vp, int64_t vh, int64_t vd, int max_blocks,
                        int num_splits, int chunk, float scale2, int window, float cap_in, float cap_out, int sink,
                        const float* __restrict__ sinks, const float* __restrict__ slopes, const float* __restrict__ gate,
                        int64_t gate_stride) {
  ts_fetch_arguments<GENERAL ? 192 : 164>();     // (nine pointers, five numbers, six strides, four more numbers and the scale; the caps, the sink and the gate)
  extern __shared__ __align__(16) float smem[];
  decode_chunk<HD, ONE, GENERAL, ONCE, false>(smem, blockDim.x / TS_WAVE, blockIdx.x, blockIdx.y, blockIdx.z, gridDim.z, out, part_o, part_ml, q, k_cache, v_cache,
                                              block_tables, seq_of_token, positions, nh, G, page_size, page_shift, page_run, kp, ks, kh, vp, vh, vd, max_blocks,
                                              num_splits, chunk, scale2, window, cap_in, cap_out, sink, sinks, slopes, gate, gate_stride);
}

// out[t, h, :] = sum_s o_s 2^{m_s - M} / sum_s l_s 2^{m_s - M} over the chunks s that hold visible keys
// (the running maxima are in units of log2).
// One 64-thread workgroup per (token, head): the lanes fetch the chunks' (m, l) side by side, then
// every lane sums its output dimensions over the chunks in ascending order.
#define COMBINE_MAX_SPLITS 1024
__global__ void __launch_bounds__(TS_WAVE)
attn_decode_combine_kernel(bf16_t* __restrict__ out, const float* __restrict__ part_o,
                           const float* __restrict__ part_ml, const int32_t* __restrict__ positions, int nh, int hd,
                           int num_splits, int chunk, int window, int sink, const float* __restrict__ sinks,
                           const float* __restrict__ gate, int64_t gate_stride) {
  __shared__ float wgt[COMBINE_MAX_SPLITS];
  const int t = blockIdx.x / nh, lane = threadIdx.x;
  const int64_t th = blockIdx.x;
  const int pos = positions[t];
  const int lo = ts_first_key(pos, window);
  const int s0 = min(lo / chunk, num_splits - 1), s1 = min(pos / chunk, num_splits - 1);  // the last chunk is open-ended
  const float* ml = part_ml + th * num_splits * 2;
  float M = -INFINITY;
  for (int s = s0 + lane; s <= s1; s += TS_WAVE) M = fmaxf(M, ml[2 * s]);
  M = wave_max(M);
  float L = 0.f;
  for (int s = s0 + lane; s <= s1; s += TS_WAVE) {
    const float w = fast_exp2(ml[2 * s] - M);
    wgt[s - s0] = w;
    L += ml[2 * s + 1] * w;
  }
  L = wave_sum(L);
  // the sink's score is 0, or its head's learned one
  if (sink) L += fast_exp2((sinks ? sinks[blockIdx.x % nh] * 1.44269504088896340736f : 0.f) - M);
  wave_sync();
  const float inv = 1.0f / L;
  const float* po = part_o + (th * num_splits + s0) * hd;
  for (int d = lane; d < hd; d += TS_WAVE) {
    float acc = 0.f;
#pragma unroll 4
    for (int s = 0; s <= s1 - s0; ++s) acc = fmaf(po[(int64_t)s * hd + d], wgt[s], acc);
    out[th * hd + d] = f2bf(acc * inv * ts_out_gate(gate, gate_stride, t, blockIdx.x % nh, hd, d));
  }
}

// What output dimension `d` has of chunks s0 to s1, up to MOST of them, whose (m, l) and parts are all asked for before the first is used (the last one's
// again for those that there are fewer): the sums are those above, in their order.
template <int MOST>
static __device__ __forceinline__ float
combine_few(const float* __restrict__ part_o, const float* __restrict__ part_ml, int64_t th, int s0, int s1, int num_splits, int hd, int d, float* sink) {
  const int lane = threadIdx.x % TS_WAVE;
  const float* const po = part_o + th * num_splits * hd + min(d, hd - 1);
  float v[MOST];
#pragma unroll
  for (int k = 0; k < MOST; ++k) v[k] = po[min(s0 + k, s1) * hd];
  const float* const ml = part_ml + 2 * (th * num_splits + min(s0 + lane, s1));
  const bool visible = s0 + lane <= s1;
  const float m = ml[0], l = ml[1];
  const float M = wave_max(visible ? m : -INFINITY);
  const float w = visible ? fast_exp2(m - M) : 0.f;
  float L = wave_sum(visible ? l * w : 0.f);
  if (sink) L += fast_exp2(*sink - M);
  const float inv = 1.0f / L;
  float acc = 0.f;
#pragma unroll
  for (int k = 0; k < MOST; ++k) {
    const float ws = __shfl(w, k, TS_WAVE);
    if (s0 + k <= s1) acc = fmaf(v[k], ws, acc);
  }
  return acc * inv;
}

// The same of up to MOST chunks, a thread an output dimension: the kernel is a chain of trips to memory (the position, the chunks' (m, l), their parts, which other
// dies have just written), so all that a token's visible chunks have left is asked for at once when its position is there, and no more of it (of up to
// four of them with a quarter of the loads). us, chain and here, with every chunk visible and with one: 32 heads of 64, 8 tokens of 8 chunks 3.14 and 2.50, 2.62 and 2.16, 64 of 8
// 4.95 and 4.32, 3.44 and 3.00, 64 of 12 5.88 and 5.16, 3.32 and 2.90, 300 of 8 13.3 and 11.2, 6.42 and 4.86; 32 of 128, 64 of 16 11.7 and 9.84, 3.70 and 3.08, 24 of 128, 8 of 8 2.98 and
// 2.23, 2.70 and 2.16. (The position asked for along with the parts of every chunk there is: no faster with all visible, 10.5 with one of the 16.)
template <int MOST>
__global__ void __launch_bounds__(4 * TS_WAVE)
attn_decode_combine_few_kernel(bf16_t* __restrict__ out, const float* __restrict__ part_o, const float* __restrict__ part_ml, const int32_t* __restrict__ positions,
                               int nh, int hd, int num_splits, int chunk, int window, int sink, const float* __restrict__ sinks, const float* __restrict__ gate,
                               int64_t gate_stride) {
  const int t = blockIdx.x / nh, d = threadIdx.x;
  const int64_t th = blockIdx.x;
  const int pos = positions[t], lo = ts_first_key(pos, window);
  const int s0 = min(lo / chunk, num_splits - 1), s1 = max(min(pos / chunk, num_splits - 1), s0);  // the last chunk is open-ended
  // the sink's score is 0, or its head's learned one
  float score = sink && sinks ? sinks[blockIdx.x % nh] * 1.44269504088896340736f : 0.f;
  const float y = s1 - s0 < 4 ? combine_few<4>(part_o, part_ml, th, s0, s1, num_splits, hd, d, sink ? &score : nullptr)
                              : combine_few<MOST>(part_o, part_ml, th, s0, s1, num_splits, hd, d, sink ? &score : nullptr);
  if (d < hd) out[th * hd + d] = f2bf(y * ts_out_gate(gate, gate_stride, t, blockIdx.x % nh, hd, d));
}

// The combining kernel alone: out [tokens, nh, hd] bfloat16 from the parts that ts_paged_attention_decode leaves
// with combine 0.
extern "C" int ts_attention_combine(void* out, const float* part_o, const float* part_ml, const int32_t* positions,
                                    int num_tokens, int nh, int hd, int num_splits, int chunk, int window, hipStream_t stream) {
  if (num_tokens <= 0) return TS_OK;
  if (!out || !part_o || !part_ml || !positions || nh <= 0 || hd <= 0 || num_splits < 1 || chunk <= 0) return TS_BAD_SHAPE;
  return ts_launch_attention_combine(out, part_o, part_ml, positions, num_tokens, nh, hd, num_splits, chunk, window, stream);
}

// The combining kernel alone, for the prefill kernel's split walks (declared in attention_mfma.h).
int ts_launch_attention_combine(void* out, const float* part_o, const float* part_ml, const int32_t* positions,
                                int num_tokens, int nh, int hd, int num_splits, int chunk, int window,
                                hipStream_t stream, int sink, const float* sinks, const float* gate, int64_t gate_stride) {
  if (num_splits > COMBINE_MAX_SPLITS) return TS_BAD_SHAPE;
#define TS_COMBINE(KERNEL, THREADS) \
  KERNEL<<<num_tokens * nh, THREADS, 0, stream>>>((bf16_t*)out, part_o, part_ml, positions, nh, hd, num_splits, chunk, window, sink, sinks, gate, gate_stride)
  const int threads = (hd + TS_WAVE - 1) / TS_WAVE * TS_WAVE;
  if (num_splits > 16 || hd > 4 * TS_WAVE) TS_COMBINE(attn_decode_combine_kernel, TS_WAVE);
  else if (num_splits > 8) TS_COMBINE(attn_decode_combine_few_kernel<16>, threads);
  else TS_COMBINE(attn_decode_combine_few_kernel<8>, threads);
#undef TS_COMBINE
  return ts_check_launch();
}

// part_o [tokens, nh, num_splits, hd] and part_ml [tokens, nh, num_splits, 2] are float workspaces
// (unused and may be null when num_splits is 1). num_splits * chunk must cover every position that
// `positions` holds; a workgroup has `waves` waves that take the chunk's 32-key steps in turn (chunk is a multiple of 32 waves). (Letting the last workgroup
// of a token combine its chunks inside the first kernel was tried and is slower: on a GPU of several
// dies the device-scope fences it needs write back and invalidate each die's L2.) Keys: rows dense in
// head_dim, strides kp/ks/kh (page, slot, head). Values: transposed pages, slot stride 1, strides
// vp/vh/vd (page, head, dimension). An entry of block_tables names 2^page_run consecutive pages of page_size
// keys (entry e: the pages e 2^page_run + j); max_blocks is the tables' width in entries.
static int launch_decode(void* out, float* part_o, float* part_ml, const void* q, const void* k_cache,
                         const void* v_cache, const int32_t* block_tables,
                         const int32_t* seq_of_token, const int32_t* positions, int num_tokens, int nh,
                         int nkv, int hd, int page_size, int64_t kp, int64_t ks, int64_t kh,
                         int64_t vp, int64_t vh, int64_t vd, int max_blocks, int num_splits, int chunk,
                         int waves, float scale, int window, int page_run, int combine, bool general, float softcap, int sink,
                         const float* sinks, const float* slopes, const float* gate, int64_t gate_stride, hipStream_t stream) {
  if (num_tokens <= 0) return TS_OK;
  if (gate && (!general || !combine || (gate_stride < (int64_t)nh * hd && -gate_stride < nh))) return TS_BAD_SHAPE;
  if (nkv <= 0 || nh % nkv || page_size <= 0 || page_size % 8 || max_blocks <= 0 || num_splits <= 0 || page_run < 0 || page_run > 16)
    return TS_BAD_SHAPE;
  if (waves < 1 || waves > DEC_WAVES_FOR(hd, chunk == 32 * waves) || chunk <= 0 || chunk % (32 * waves) || num_splits > COMBINE_MAX_SPLITS)
    return TS_BAD_SHAPE;
  if (num_splits > 1 && (!part_o || !part_ml)) return TS_BAD_SHAPE;
  if (num_tokens > 65535 || nkv > 65535) return TS_BAD_SHAPE;
  const int G = nh / nkv;
  if (G > 16 || G * hd > 2048) return TS_BAD_SHAPE;
  // 16-byte loads: key rows and the 8-key pieces of value rows must be 16-byte aligned
  if ((kp % 8) || (ks % 8) || (kh % 8) || (vp % 8) || (vh % 8) || (vd % 8)) return TS_BAD_SHAPE;
  if ((((uintptr_t)q) | ((uintptr_t)k_cache) | ((uintptr_t)v_cache)) & 15) return TS_BAD_SHAPE;
  const size_t smem = sizeof(float) * (2 * waves * 16 + (size_t)waves * G * hd);
  if (smem > 65536) return TS_BAD_SHAPE;
  int page_shift = -1;
  if ((page_size & (page_size - 1)) == 0) {
    page_shift = 0;
    while ((1 << page_shift) < page_size) ++page_shift;
  }
  dim3 grid(num_splits, nkv, num_tokens);
  const int64_t reach = (int64_t)num_splits * chunk, within = window < 0 ? -(int64_t)window : window, keys = within && within < reach ? within : reach;
  const bool once = (int64_t)num_tokens * nkv * hd * 4 * keys >= DEC_ONCE_BYTES;
  // capped: the cap's tanh takes the scale in and gives units of log2 out, and the softmax's own scale is 1
  const float log2e = 1.44269504088896340736f;
  const float cap_in = softcap > 0.f ? scale / softcap : 0.f, cap_out = softcap * log2e;
  const float scale2 = softcap > 0.f ? 1.0f : scale * log2e;
#define TS_DEC3(HH, ON, GG, NC)                                                                                 \
  attn_decode_mfma_kernel<HH, ON, GG, NC><<<grid, waves * TS_WAVE, smem, stream>>>(                                 \
      (bf16_t*)out, part_o, part_ml, (const bf16_t*)q, (const bf16_t*)k_cache, (const bf16_t*)v_cache,          \
      block_tables, seq_of_token, positions, nh, G, page_size, page_shift, page_run, kp, ks, kh, vp, vh, vd, max_blocks,  \
      num_splits, chunk, scale2, window, cap_in, cap_out, sink, sinks, slopes, gate, gate_stride)
#define TS_DEC2(HH, ON, GG) if (once) TS_DEC3(HH, ON, GG, true); else TS_DEC3(HH, ON, GG, false)
#define TS_DEC1(HH, ON) if (general) { TS_DEC2(HH, ON, true); } else { TS_DEC2(HH, ON, false); }
#define TS_DEC(HH) if (chunk == 32 * waves) { TS_DEC1(HH, true); } else { TS_DEC1(HH, false); }
  switch (hd) {
    case 32: TS_DEC(32); break;
    case 64: TS_DEC(64); break;
    case 96: TS_DEC(96); break;
    case 128: TS_DEC(128); break;
    default: return TS_BAD_SHAPE;
  }
#undef TS_DEC
#undef TS_DEC1
#undef TS_DEC2
#undef TS_DEC3
  int rc = ts_check_launch();
  if (rc || num_splits == 1 || !combine) return rc;     // (combine 0: the caller's next kernel reads the parts itself)
  return ts_launch_attention_combine(out, part_o, part_ml, positions, num_tokens, nh, hd, num_splits, chunk, window, stream, general ? sink : 0,
                                     general ? sinks : nullptr, gate, gate_stride);
}

extern "C" int ts_paged_attention_decode(void* out, float* part_o, float* part_ml, const void* q, const void* k_cache,
                                         const void* v_cache, const int32_t* block_tables,
                                         const int32_t* seq_of_token, const int32_t* positions, int num_tokens, int nh,
                                         int nkv, int hd, int page_size, int64_t kp, int64_t ks, int64_t kh,
                                         int64_t vp, int64_t vh, int64_t vd, int max_blocks, int num_splits, int chunk,
                                         int waves, float scale, int window, int page_run, int combine, hipStream_t stream) {
  return launch_decode(out, part_o, part_ml, q, k_cache, v_cache, block_tables, seq_of_token, positions, num_tokens, nh, nkv, hd,
                       page_size, kp, ks, kh, vp, vh, vd, max_blocks, num_splits, chunk, waves, scale, window, page_run, combine,
                       false, 0.f, 0, nullptr, nullptr, nullptr, 0, stream);
}

// The same with capped scores (softcap > 0: cap * tanh(score / cap)), a sink (one more in the softmax's
// denominator; `sinks`, float [nh], if given: exp(sinks[head]) more instead), a penalty of slopes[head] (float [nh],
// if given) per position of distance taken off every score, and weights carried in two bfloat16 terms; always combines.
// `gate` (float [tokens, >= nh hd], rows gate_stride apart; may be null): the output leaves multiplied by sigmoid(gate);
// a stride below zero: one number per head (`ts_out_gate`).
extern "C" int ts_paged_attention_decode_general(void* out, float* part_o, float* part_ml, const void* q, const void* k_cache,
                                                 const void* v_cache, const int32_t* block_tables,
                                                 const int32_t* seq_of_token, const int32_t* positions, int num_tokens,
                                                 int nh, int nkv, int hd, int page_size, int64_t kp, int64_t ks, int64_t kh,
                                                 int64_t vp, int64_t vh, int64_t vd, int max_blocks, int num_splits,
                                                 int chunk, int waves, float scale, int window, int page_run, float softcap,
                                                 int sink, const float* sinks, const float* slopes, const float* gate,
                                                 int64_t gate_stride, hipStream_t stream) {
  if (softcap < 0.f) return TS_BAD_SHAPE;
  return launch_decode(out, part_o, part_ml, q, k_cache, v_cache, block_tables, seq_of_token, positions, num_tokens, nh, nkv, hd,
                       page_size, kp, ks, kh, vp, vh, vd, max_blocks, num_splits, chunk, waves, scale, window, page_run, 1,
                       true, softcap, sink || sinks, sinks, slopes, gate, gate_stride, stream);
}
