// The launchers that calls.cpp calls itself, instead of Python through ctypes. common.h includes this, so that a launcher whose
// parameters are other than here does not compile.
#pragma once
#include <stddef.h>
#include <stdint.h>

// Error codes returned by the extern "C" launchers (0 = launched).
#define TS_OK 0
#define TS_BAD_DTYPE 1
#define TS_BAD_SHAPE 2
#define TS_LAUNCH_FAILED 3
#define TS_TOO_LARGE 4

typedef struct ihipStream_t* hipStream_t;

extern "C" {
int ts_rmsnorm(void* out, void* res_out, const void* x, const void* res, const void* w, const int32_t* rows, int num_rows, int hidden,
               float eps, int dtype, int wdtype, hipStream_t stream);
int ts_rope_store(void* q_out, void* k_cache, void* v_cache, const void* qkv, const float* cos_sin, const int32_t* positions,
                  const int32_t* slots, int num_tokens, int nh, int nkv, int hd, int rot, int rotate, int page_size, int64_t kp, int64_t ks,
                  int64_t kh, int64_t vp, int64_t vs, int64_t vh, int64_t vd, int dtype, hipStream_t stream);
int ts_gemm_library_bf16(void* y, const void* x, const void* w, int M, int N, int K, int64_t ldx, int64_t ldw, int64_t ldy, int out_f32,
                         int tune, void* flush, size_t flush_bytes, hipStream_t stream);
int ts_gemm_slices_bf16(void* y, void* sum, void* parts, const void* x, const void* w, int M, int N, int K, int64_t ldx, int64_t ldw, int tile,
                        int slices, int out_f32, const void* res, const void* norm_w, float eps, hipStream_t stream);
int ts_gemm_slices_parts_bf16(float* parts, const void* x, const void* w, int M, int N, int K, int64_t ldx, int64_t ldw, int tile, int slices,
                              hipStream_t stream);
int ts_gemm_whole_bf16(int products, void* const* y, const void* const* x, const void* const* w, const int* N, int M, int K, int64_t ldx, int64_t ldw,
                       int tile, int chained, int out_f32, hipStream_t stream);
int ts_gemm_whole_rope_bf16(void* q_out, const void* x, const void* w, int M, int K, int64_t ldx, int64_t ldw, const float* cos_sin,
                            const int32_t* positions, const int32_t* slots, void* k_cache, void* v_cache, int nh, int nkv, int hd, int page_size,
                            int64_t kp, int64_t ks, int64_t kh, int64_t vp, int64_t vs, int64_t vh, int64_t vd, int tile, hipStream_t stream);
int ts_gemm_glu_bf16(void* y, const void* x, const void* w, int M, int F, int K, int64_t ldx, int64_t ldw, int64_t ldy, int tile, int act,
                     float limit, float slope, float up_shift, hipStream_t stream);
int ts_gemm_rows64_bf16(void* y, const void* x, const void* w16, int M, int N, int K, int64_t ldx, int64_t ldy, int glu, int out_f32,
                        const void* ssq_in, int ssq_parts, float eps, float limit, float slope, float up_shift, int few, hipStream_t stream);
int ts_gemm_rows64_group_bf16(int products, void* const* y, const void* const* x, const void* w16, const int* N, int M, int K, int64_t ldx,
                              hipStream_t stream);
int ts_gemm_rows64_sliced_bf16(void* y, void* parts, const void* x, const void* w16, int M, int N, int K, int64_t ldx, int slices,
                               const void* next_res, const void* next_nw, void* next_res_out, void* next_op, void* ssq_out, int64_t ld_op,
                               hipStream_t stream);
int ts_gemm_skinny8_bf16(void* y, const void* x, const void* w, int M, int N, int K, int64_t ldx, int64_t ldw, int64_t ldy, int out_dtype, int packed,
                         const void* next_res, const void* next_nw, void* next_res_out, void* next_op, void* ssq_out, int x_packed8, const float* comb_o,
                         const float* comb_ml, const int32_t* comb_pos, int comb_splits, int comb_chunk, int comb_window, int comb_hd, float cap,
                         hipStream_t stream);
int ts_skinny_tiles(int M, int N, int K);
int ts_gemm_skinny_bf16(void* y, const void* x, const void* w, const void* res, const void* nw, void* res_out, int M, int N, int K, int64_t ldx, int64_t ldw,
                        int64_t ldy, float eps, int mode, int glu, int out_dtype, int packed, const void* ssq_in, int ssq_parts, const void* next_res,
                        const void* next_nw, void* next_res_out, void* next_op, void* ssq_out, int y_pack8, float limit, float slope, float up_shift,
                        hipStream_t stream);
int ts_gemm_skinny_rope_bf16(void* q_out, const void* x, const void* w, const void* res, const void* nw, void* res_out, int M, int K, int64_t ldx,
                             int64_t ldw, float eps, int mode, int packed, const float* cos_sin, const int32_t* positions, const int32_t* slots,
                             void* k_cache, void* v_cache, int nh, int nkv, int hd, int rotate, int page_size, int64_t kp, int64_t ks, int64_t kh,
                             int64_t vp, int64_t vs, int64_t vh, int64_t vd, const void* ssq_in, int ssq_parts, hipStream_t stream);
int ts_gemm_rows64_sliced_rope_bf16(void* q_out, void* parts, const void* x, const void* w16, int M, int K, int64_t ldx, int slices,
                                    const void* ssq_in, int ssq_parts, float eps, const float* cos_sin, const int32_t* positions,
                                    const int32_t* slots, void* k_cache, void* v_cache, int nh, int nkv, int hd, int rotate, int page_size,
                                    int64_t kp, int64_t ks, int64_t kh, int64_t vp, int64_t vs, int64_t vh, int64_t vd, hipStream_t stream);
int ts_paged_attention_step(void* out, float* part_o, float* part_ml, const void* q, const void* k_cache, const void* v_cache, const int32_t* block_tables,
                            const int32_t* seq_of_token, const int32_t* positions, int num_tokens, int num_splits, int chunk, int decode_waves,
                            const int32_t* tiles, int num_tiles, int tile_tokens, int waves, int nh, int nkv, int hd, int page_size, int64_t kp, int64_t ks,
                            int64_t kh, int64_t vp, int64_t vh, int64_t vd, int max_blocks, float scale, int window, int page_run, int general, float softcap,
                            int sink, const float* sinks, const float* slopes, const float* gate, int64_t gate_stride, hipStream_t stream);
int ts_paged_attention_decode(void* out, float* part_o, float* part_ml, const void* q, const void* k_cache, const void* v_cache,
                              const int32_t* block_tables, const int32_t* seq_of_token, const int32_t* positions, int num_tokens, int nh,
                              int nkv, int hd, int page_size, int64_t kp, int64_t ks, int64_t kh, int64_t vp, int64_t vh, int64_t vd,
                              int max_blocks, int num_splits, int chunk, int waves, float scale, int window, int page_run, int combine,
                              hipStream_t stream);
int ts_paged_attention_decode_general(void* out, float* part_o, float* part_ml, const void* q, const void* k_cache, const void* v_cache,
                                      const int32_t* block_tables, const int32_t* seq_of_token, const int32_t* positions, int num_tokens,
                                      int nh, int nkv, int hd, int page_size, int64_t kp, int64_t ks, int64_t kh, int64_t vp, int64_t vh,
                                      int64_t vd, int max_blocks, int num_splits, int chunk, int waves, float scale, int window,
                                      int page_run, float softcap, int sink, const float* sinks, const float* slopes, const float* gate,
                                      int64_t gate_stride, hipStream_t stream);
int ts_paged_attention_prefill(void* out, const void* q, const void* k_cache, const void* v_cache, const int32_t* block_tables,
                               const int32_t* seq_of_token, const int32_t* positions, const int32_t* tiles, int num_tiles, int tile_tokens,
                               int waves, int nh, int nkv, int hd, int page_size, int64_t kp, int64_t ks, int64_t kh, int64_t vp, int64_t vh,
                               int64_t vd, int max_blocks, float scale, int window, int first_token, int num_tokens, int num_splits,
                               int chunk, float* part_o, float* part_ml, int page_run, hipStream_t stream);
int ts_paged_attention_prefill_general(void* out, const void* q, const void* k_cache, const void* v_cache, const int32_t* block_tables,
                                       const int32_t* seq_of_token, const int32_t* positions, const int32_t* tiles, int num_tiles,
                                       int tile_tokens, int waves, int nh, int nkv, int hd, int page_size, int64_t kp, int64_t ks, int64_t kh,
                                       int64_t vp, int64_t vh, int64_t vd, int max_blocks, float scale, int window, int first_token,
                                       int num_tokens, int num_splits, int chunk, float* part_o, float* part_ml, int page_run, float softcap,
                                       int sink, const float* sinks, const float* slopes, const float* gate, int64_t gate_stride,
                                       hipStream_t stream);
int ts_stream_post_norm(float* x, const float* a, const float* post_w, const float* scale, float post_eps, void* h, int h_dtype,
                        const float* w, float eps, int num_rows, int width, hipStream_t stream);
int ts_stream_post_norm_parts(float* x, const float* p, int64_t stride, int count, int scaled, float fa, float fb, const float* post_w, const float* scale,
                              float post_eps, void* h, int h_dtype, const float* w, float eps, int num_rows, int width, hipStream_t stream);
int ts_stream_post_norm_experts(float* x, const float* rows, const float* weights, const float* shared, int top, const int32_t* ids, int real, const void* input,
                                const float* gate, const float* post_w, const float* scale, float post_eps, void* h, int h_dtype, const float* w, float eps,
                                int num_rows, int width, hipStream_t stream);
int ts_stream_update_norm_parts(float* x, const float* a, const float* p, int64_t stride, int count, int scaled, float fa, float fb, float mult, void* h,
                                int h_dtype, const void* w, int w_dtype, float eps, int num_rows, int width, hipStream_t stream);
int ts_stream_update_norm(float* x, const void* a, int a_dtype, const void* b, int b_dtype, const void* bias, int bias_dtype, float mult,
                          void* h1, void* h2, int h_dtype, const void* w1, const void* w2, int w_dtype, float eps, const int32_t* rows,
                          int num_rows, int width, hipStream_t stream);
int ts_capped_glu(void* out, int out_dtype, const void* gate_up, int in_dtype, int64_t row_stride, int n, int ff, float limit, float slope,
                  float up_shift, int act, hipStream_t stream);
int ts_qkv_finish(void* q_out, void* k_cache, void* v_cache, const void* qkv, const double* freqs, const int32_t* positions,
                  const int32_t* slots, int num_tokens, int nh, int nkv, int hd, int vd_size, int rot, int interleaved, int qk_norm,
                  float qk_eps, int v_norm, float v_eps, int page_size, int64_t kp, int64_t ks, int64_t kh, int64_t vp, int64_t vs,
                  int64_t vh, int64_t vd, int in_dtype, int out_dtype, float amplitude, int64_t row, hipStream_t stream);
int ts_mlstm_finish(void* out, int out_dtype, const float* o, const float* weight, const float* gate, int64_t gate_stride, int num_tokens,
                    int heads, int vdim, float eps, int weight_head, int silu_gate, hipStream_t stream);
}

// 32-wide steps of k that a wave of the 8-row form takes for a reduction of K (it covers 64 of k in each): the fewest that fit 8 waves, else 16 in up to
// 16 waves; 0: it does not serve K.
static inline int ts_skinny8_steps(int K) {
  for (int steps : {4, 8, 16})
    if (K % (64 * steps) == 0 && K / (64 * steps) <= 8) return steps;
  return K % 1024 == 0 && K / 1024 <= 16 ? 16 : 0;
}
