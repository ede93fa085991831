// The entry points that the layers of a dense model launch: declared once, for the files that define them and for the one that
// calls them again for further layers (layer_launches.hip).
#pragma once
#include <hip/hip_runtime.h>

extern "C" {
int jllm_rmsnorm(const float* x, const int* rows, int n_rows, int d, const void* gain, int gain_dtype, float eps, void* out, int out_dtype,
        int ldo, hipStream_t stream);
int jllm_gemm_generic(const void* A, int a_dtype, int lda, const void* W, const void* W2, int w_dtype, const void* bias, int bias_dtype,
        void* out, int out_dtype, int ldo, int M, int N, int K, int epilogue, float gate_limit, hipStream_t stream);
int jllm_gemm_skinny_bf16(const void* A, int lda, const void* W, const void* W2, const void* bias, int bias_dtype, void* out, int out_dtype,
        int ldo, int M, int N, int K, int epilogue, float gate_limit, int rows, hipStream_t stream);
int jllm_gemm_skinny_norm_bf16(const void* A, int lda, const void* W, const void* W2, const void* bias, int bias_dtype, void* out, int
        out_dtype, int ldo, int M, int N, int K, int epilogue, float gate_limit, int rows, void* emit_rows, const void* emit_gain, int
        emit_gain_dtype, float* emit_partial, int emit_parts, const float* norm_partial, int norm_parts, float norm_eps, hipStream_t
        stream);
int jllm_gemm_mfma_bf16(const void* A, int lda, const void* W, const void* W2, const void* bias, int bias_dtype, void* out, int out_dtype,
        int ldo, int M, int N, int K, int epilogue, float gate_limit, int tile, int splits, float* partial, const void* norm_gain, int
        norm_gain_dtype, float norm_eps, void* norm_rows, int norm_ld, hipStream_t stream);
int jllm_gemm_pingpong_bf16(const void* A, int lda, const void* W, const void* W2, const void* bias, int bias_dtype, void* out, int
        out_dtype, int ldo, int M, int N, int K, int epilogue, float gate_limit, int tile_rows, int splits, float* partial, const void*
        norm_gain, int norm_gain_dtype, float norm_eps, void* norm_rows, int norm_ld, hipStream_t stream);
int jllm_gemm_stream_bf16(const void* A, int lda, const void* W, const void* W2, const void* bias, int bias_dtype, void* out, int out_dtype,
        int ldo, int M, int N, int K, int epilogue, float gate_limit, int rows, int tile_m, int parts, float* partial, int* arrivals, void*
        emit_rows, int emit_ld, const void* emit_gain, int emit_gain_dtype, float* emit_partial, int emit_parts, const float* norm_partial,
        int norm_parts, float norm_eps, hipStream_t stream);
int jllm_qk_norm_rope_store(void* qkv, int dtype, int ld, const int* positions, const int* slots, const float* cos_t, const float* sin_t,
        const void* gq, const void* gk, int gain_dtype, float eps, int n_tokens, int H, int Hkv, int hd, int rot, int page_size, void*
        kcache, void* vcache, int write_kv, hipStream_t stream);
int jllm_paged_attention_generic(const void* q, int ldq, void* out, int ldo, int dtype, const void* kcache, const void* vcache, const int*
        block_table, int max_blocks, const int* row_req, const int* positions, int n_tokens, int n_requests, int H, int Hkv, int hd, int
        page_size, int window, float scale, const float* slopes, hipStream_t stream);
int jllm_decode_attention_bf16(const void* q, int ldq, void* out, int ldo, const void* kcache, const void* vcache, const int* block_table,
        int max_blocks, const int* row_req, const int* positions, int n_rows, int H, int Hkv, int hd, int page_size, int window, float
        scale, int max_pos, float* part_acc, float* part_ml, int max_splits, int split, hipStream_t stream);
int jllm_decode_attention_fused_bf16(const void* qkv, int ldqkv, void* out, int ldo, void* kcache, void* vcache, const int* block_table, int
        max_blocks, int table_rows, const int* row_req, const int* positions, const int* slots, const float* cos_t, const float* sin_t,
        const void* gq, const void* gk, int gain_dtype, float eps, int rot, int write_kv, int n_rows, int H, int Hkv, int hd, int page_size, int window,
        float scale, int max_pos, float* part_acc, float* part_ml, int max_splits, int split, int* arrivals, hipStream_t stream);
int jllm_prefill_attention_bf16(const void* q, int ldq, void* out, int ldo, const void* kcache, const void* vcache, const int* block_table,
        int max_blocks, const int* tiles, const int* positions, int n_tiles, int n_requests, int H, int Hkv, int hd, int page_size, int
        window, int max_context, float scale, int key_groups, hipStream_t stream);
}

// name by name, for a table of them
#define JLLM_LAYER_ENTRIES(X) \
  X(jllm_rmsnorm) \
  X(jllm_gemm_generic) \
  X(jllm_gemm_skinny_bf16) \
  X(jllm_gemm_skinny_norm_bf16) \
  X(jllm_gemm_mfma_bf16) \
  X(jllm_gemm_pingpong_bf16) \
  X(jllm_gemm_stream_bf16) \
  X(jllm_qk_norm_rope_store) \
  X(jllm_paged_attention_generic) \
  X(jllm_decode_attention_bf16) \
  X(jllm_decode_attention_fused_bf16) \
  X(jllm_prefill_attention_bf16)
