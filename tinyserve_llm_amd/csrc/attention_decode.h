// One chunk of one decoding token's walk (attention_decode.hip says how the work is cut), for the kernel that decodes and for the one that takes a step's
// decoding tokens beside its prompts (attention_prefill.hip).
#pragma once
#include "attention_mfma.h"

#define DEC_MAX_WAVES 8
// heads wider than 64 keep two steps of wide rows in registers in the general loop: its workgroups
// have up to 4 waves then (with 8, a lane's 256 registers are overrun by 22, and 64 tokens over
// 2,560 keys take 137 µs instead of 122); the instance with a single step per wave has room for 8
#define DEC_WAVES_FOR(HD, ONE) ((HD) > 64 && !(ONE) ? 4 : DEC_MAX_WAVES)

// Bytes of keys and values, counted from what the tables have room for (from the window, where that is less), from which values go by the
// caches: they are put out before the next step reads them again, and what they put out are the weights' and the other kernels' lines. Decode steps of
// 12 layers of the 1B widths, through the caches and past them, us: over 2,048 keys 16 rows (67 MB a layer) 825 and 817, 64 rows 1,358 and 1,337, 96 rows 1,878 and 1,821, over 4,096
// keys 48 rows 1,644 and 1,572, 64 rows 2,059 and 1,911, over 1,024 keys 24 rows 770 both, 96 rows 1,398 and 1,384; 8 layers of heads of 128 over 2,048 keys, 16 rows 873 and 852, 64 rows 1,633 and 1,533; below,
// 8 rows over 2,048 keys (34 MB) 685 and 689, with the keys. With pages that all requests share as with their own: 64 rows over 2,048 keys, 7 of 9 pages shared, 1,096 and 1,081.
// Keys too where a wave has a single step of heads up to 64 wide: 16 rows over 2,048 keys 819 and 806, 48 rows 1,193 and 1,181; in the loop over several steps, where half of each
// line is asked for a second time, it has gone by then (20 rows over 3,072 keys 928 and 972, 96 rows over 1,024 keys 1,384 and 1,444). But not of pages that the next token's request
// has too, which reads them at once (16 rows over 2,048 keys, 8 of 9 pages shared: 759 and 766).
#define DEC_ONCE_BYTES (48ll << 20)

// ONE: a wave has a single 32-key step (chunk = 32 waves); without the second buffer of the
// general loop the kernel needs fewer registers and more workgroups share a compute unit
// GENERAL: capped scores, weights in two terms (attention_mfma.h), and optionally a sink: one more in the
// softmax's denominator, added where a token's chunks meet (here with one chunk, else in the combining kernel).
// ONCE: values by load_once, and some keys (DEC_ONCE_BYTES).
// `nw` waves share a chunk; SHARED: of a workgroup of another number, whose waves take those waves' keys in turn, each with sums of its own (the same bits).
struct DecodeArgs {
  bf16_t* out;
  float *part_o, *part_ml;
  const bf16_t *q, *k_cache, *v_cache;
  const int32_t *block_tables, *seq_of_token, *positions;
  int nh, G, page_size, page_shift, page_run;
  int64_t kp, ks, kh, vp, vh, vd;
  int max_blocks, num_splits, chunk;
  float scale2;
  int window;
  float cap_in, cap_out;
  int sink;
  const float *sinks, *slopes, *gate;
  int64_t gate_stride;
};

template <int HD, bool ONE, bool GENERAL, bool ONCE, bool SHARED>
static __device__ __forceinline__ void
decode_chunk(float* smem, int nw, int split, int kvh, int t, int tokens, bf16_t* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml,
             const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
             const int32_t* __restrict__ block_tables, const int32_t* __restrict__ seq_of_token,
             const int32_t* __restrict__ positions, int nh, int G, int page_size, int page_shift, int page_run,
             int64_t kp, int64_t ks, int64_t kh, int64_t vp, int64_t vh, int64_t vd, int max_blocks,
             int num_splits, int chunk, float scale2, int window, float cap_in, float cap_out, int sink,
             const float* __restrict__ sinks, const float* __restrict__ slopes, const float* __restrict__ gate,
             int64_t gate_stride) {
  constexpr int NC = HD / 32;    // 32-dimension pieces of a key row (one 16-byte load per lane each)
  constexpr int NDB = HD / 16;   // 16-dimension blocks of the output
  float* wm = smem;                       // [waves][16]
  float* wl = wm + nw * 16;               // [waves][16]
  float* wo = wl + nw * 16;               // [waves][G][HD]

  const int tid = threadIdx.x, wave = wave_index(), lane = tid & (TS_WAVE - 1);
  const int r = lane & 15, g = lane >> 4;
  int pos = positions[t];
  constexpr bool KEYS = ONCE && ONE && HD <= 64;
  int next = t, next_seq = 0;                   // KEYS: the token after this one (before it, of the last), and its request
  if constexpr (KEYS) {
    next = t + 1 < tokens ? t + 1 : max(t - 1, 0);
    next_seq = seq_of_token[next];
  }
  int seq = seq_of_token[t];                    // (asked for with the position: one trip to memory, not one after the other;
  asm volatile("" : "+s"(pos), "+s"(seq));      //  left to itself the compiler fetches it when it has seen that the chunk is visible)
  if constexpr (KEYS) asm volatile("" : "+s"(next_seq));
  const int lo = ts_first_key(pos, window);
  const int k0 = split * chunk;
  if (k0 > pos || k0 + chunk <= lo) return;     // nothing of this chunk is visible
  const int32_t* table = block_tables + (int64_t)seq * max_blocks;
  const PageMath pm{page_size, page_shift, page_run};

  uint4 qreg[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) qreg[c] = make_uint4(0, 0, 0, 0);
  if (r < G) {
    const bf16_t* qrow = q + ((int64_t)t * nh + (int64_t)kvh * G + r) * HD + 8 * g;
#pragma unroll
    for (int c = 0; c < NC; ++c) qreg[c] = *(const uint4*)(qrow + 32 * c);
  }
  // the chunk's visible keys, 32 at a time, dealt to the waves in turn (however few keys a request
  // has in the chunk, every wave gets its share of them, and the workgroup reads the chunk front to
  // back); the next step's loads are issued before this step's products
  const int stride = 32 * nw;
  int kend = k0 + chunk;
  if (kend > pos + 1) kend = pos + 1;
  // (the general variant: this row's head's penalty per position of distance, in the scores' units before scale2)
  const float slope = (GENERAL && slopes && r < G) ? slopes[kvh * G + r] * (1.44269504088896340736f / scale2) : 0.f;
#define TS_LOAD_AS(KEYS_ONCE, T, KB) load_tile<HD, KEYS_ONCE, ONCE>(T, KB, r, g, lo, pos, kvh, table, pm, k_cache, v_cache, kp, ks, kh, vp, vh, vd)
#define TS_LOAD(T, KB) TS_LOAD_AS(false, T, KB)
#define TS_USE(T, KB) use_tile_auto<HD, GENERAL>(T, KB, r, g, lo, pos, pos, lo, qreg, scale2, m, l, o, cap_in, cap_out, slope)
  const int here = SHARED ? (int)blockDim.x / TS_WAVE : nw;
  for (int w = wave; !SHARED || w < nw; w += here) {
    int kb = (k0 > (lo & ~31) ? k0 : (lo & ~31)) + 32 * w;
    float m = -INFINITY, l = 0.f;
    float4_t o[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db) o[db] = (float4_t){0.f, 0.f, 0.f, 0.f};
    if (ONE) {
      if (kb < kend) {
        KVTile<HD> A;
        const int entry = pm.page(kb) >> page_run;      // (KEYS: of this step, whose page is looked up in any case)
        if (KEYS && !(next != t && block_tables[(int64_t)next_seq * max_blocks + entry] == table[entry])) {
          TS_LOAD_AS(KEYS, A, kb);      // (the products in both arms: where these meet the compiler waits for every load)
          TS_USE(A, kb);
        } else {
          TS_LOAD(A, kb);
          TS_USE(A, kb);
        }
      }
    } else if (kb < kend) {
      // (the next step is asked for on every path, this step again where there is none: with a load that
      // may or may not have been issued the compiler waits for all of them before it uses any)
      KVTile<HD> A, B;
      TS_LOAD(A, kb);
      while (true) {
        const bool more_b = kb + stride < kend;
        TS_LOAD(B, more_b ? kb + stride : kb);
        TS_USE(A, kb);
        if (!more_b) break;
        kb += stride;
        const bool more_a = kb + stride < kend;
        TS_LOAD(A, more_a ? kb + stride : kb);
        TS_USE(B, kb);
        if (!more_a) break;
        kb += stride;
      }
    }
    // ---- the waves meet
    l = row_sum(l);
    if (g == 0) { wm[w * 16 + r] = m; wl[w * 16 + r] = l; }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int head = 4 * g + j;
      if (head < G) {
#pragma unroll
        for (int db = 0; db < NDB; ++db) wo[((int64_t)w * G + head) * HD + 16 * db + r] = o[db][j];
      }
    }
    if constexpr (!SHARED) break;
  }
#undef TS_LOAD
#undef TS_LOAD_AS
#undef TS_USE
  __syncthreads();
  for (int i = tid; i < G * HD; i += blockDim.x) {
    const int head = i / HD, d = i - head * HD;
    float M = -INFINITY;
    for (int w = 0; w < nw; ++w) M = fmaxf(M, wm[w * 16 + head]);
    float acc = 0.f, L = 0.f;
    for (int w = 0; w < nw; ++w) {
      const float wgt = fast_exp2(wm[w * 16 + head] - M);   // a wave without keys: 2^-inf = 0
      acc = fmaf(wo[((int64_t)w * G + head) * HD + d], wgt, acc);
      L = fmaf(wl[w * 16 + head], wgt, L);
    }
    if (num_splits == 1) {                  // the whole context was this workgroup's: position `pos` is always visible
      if (GENERAL && sink) L += fast_exp2((sinks ? sinks[kvh * G + head] * 1.44269504088896340736f : 0.f) - M);
      float y = acc / L;
      if (GENERAL) y *= ts_out_gate(gate, gate_stride, t, kvh * G + head, HD, d);
      out[((int64_t)t * nh + (int64_t)kvh * G + head) * HD + d] = f2bf(y);
    } else {
      const int64_t row = ((int64_t)t * nh + (int64_t)kvh * G + head) * num_splits + split;
      part_o[row * HD + d] = acc;
      if (d == 0) { part_ml[row * 2] = M; part_ml[row * 2 + 1] = L; }
    }
  }
}
