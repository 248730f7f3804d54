// pk_block_kernels.h - device-side entry points of the conformer-block
// operations (pk_block_kernels.hip).  All pointers are device pointers;
// activations are time-major rows.
#pragma once

#include <hip/hip_runtime.h>

namespace pkgpu {

// Longest chunk of the fast attention, and of pk_gpu_attention_dev, which takes
// no workspace.  The reference's encoder never attends over more than 500 frames
// unless chunking is forced off (PK_CHUNK_THRESHOLD, parakeet.h;
// encoder.c:595-610).
constexpr int kAttnMaxT = 512;
constexpr int kAttnRows = 32;          // query rows per workgroup (fast and long)
// Row stride of a workgroup's score rows in AttnArgs::scores.
__host__ __device__ constexpr int attn_sld(int T) { return ((T + 31) & ~31) + 8; }
// Row stride of the exact attention's score rows in LDS: 4 more than a multiple
// of 32 floats, so that the 4 x 16 scores a wave instruction stores (rows 4
// apart) reach every bank twice, and the softmax's 4 rows x 16 lanes nearly so.
__host__ __device__ constexpr int attn4_sld(int T) { return ((T + 31) & ~31) + 4; }
// LDS of its workgroup of 16 rt rows and nw waves (160 KB in a CU): the score
// rows and, staged, 16 rows of 132 floats per wave and for each 16 rows of Q.
constexpr int kLdsBytes = 160 * 1024;
constexpr size_t attn_lds_bytes(int T, int rt, int nw, bool stage)
{
    return 4u * ((stage ? (size_t)(rt + nw) * 16 * 132 : 0) + (size_t)16 * rt * attn4_sld(T));
}
// Whether the exact attention keeps the score rows in LDS (T <= 1344); those of
// longer sequences go through AttnArgs::scores.
constexpr bool attn_scores_in_lds(int T) { return attn_lds_bytes(T, 1, 8, true) <= kLdsBytes; }

// Sequences of at most kAttnShortT rows never take the fast attention.
constexpr int kAttnShortT = 64;

// Relative-position attention of n chunks (encoder.c:300-408); chunk z has
// chunk_T[z] <= T rows (all T when chunk_T is null).
//   qkv  [rows][ldq]: Q | K | V (H*128 columns each, bias added); chunk z
//        starts at row chunk_rows[z]
//   P    [2T-1][ldp]: linear_pos(pe_slice(T)); a chunk of Tz rows uses its
//        rows [T - Tz, T + Tz - 1), which are linear_pos(pe_slice(Tz))
//   out  [rows][ldo]: the concatenated head outputs, chunk z at chunk_rows[z]
struct AttnArgs {
    const float* qkv; int ldq;
    const float* P; int ldp;
    const float* pos_bias_u;   // [H*128]
    const float* pos_bias_v;
    float* out; int ldo;
    const int* chunk_rows;     // device, n entries (null: one chunk at row 0)
    const int* chunk_T;        // device, n entries, each in [1, T] (null: all T)
    int T, H;
    // unless attn_scores_in_lds(T): attn_score_rows_floats(T, H, n) floats of
    // device workspace, one slice of score rows per workgroup
    float* scores;
};
// Floats of all score rows of n chunks of up to T rows.
inline size_t attn_score_rows_floats(int T, int H, int n_chunks)
{
    return (size_t)((T + kAttnRows - 1) / kAttnRows) * H * n_chunks * kAttnRows * attn_sld(T);
}
// Workspace floats the exact attention of them reads.
inline size_t attn_scores_floats(int T, int H, int n_chunks)
{
    return attn_scores_in_lds(T) ? 0 : attn_score_rows_floats(T, H, n_chunks);
}

// Depthwise convolution over time with optional Swish (tensor_ops.c:476-548,
// encoder.c:467-469), channel c of chunk z: x[chunk_rows[z] + t][c] for t in
// [0, chunk_T[z]) (all T when chunk_T is null).
struct DwArgs {
    const float* x; int ldx;
    const float* w;            // [C][K]
    const float* b;            // [C] or null
    float* out; int ldo;
    const int* chunk_rows;     // device, n entries (null: one chunk at row 0)
    const int* chunk_T;        // device, n entries, each in [1, T] (null: all T)
    int T, C, K;
    int swish;
    // x holds the pointwise convolution's 2C-wide rows and each input value
    // is their GLU, gated = x[t][c] * (1 / (1 + exp(-x[t][C + c]))), formed
    // as the GLU kernel forms it (the GLU fused: the same bits)
    int glu;
};

hipError_t launch_layer_norm(const float* x, int ldx, const float* gamma, const float* beta,
                             float* out, int ldo, int rows, int D, hipStream_t s);
// The same LayerNorm with its output pre-split for the split GEMM kernels
// (GemmProblem::a_presplit): the fp32 row's bytes hold, per group of 8
// columns, the 8 bf16 hi then the 8 bf16 lo halves.
hipError_t launch_layer_norm_split(const float* x, int ldx, const float* gamma, const float* beta,
                                   float* out, int ldo, int rows, int D, hipStream_t s);
hipError_t launch_attention(const AttnArgs& a, int n_chunks, hipStream_t s);
// The same attention on split bf16 operands (fast numerics, within about 1e-5
// of launch_attention; not bit-identical), for T <= kAttnMaxT: a first
// launch splits the chunks' keys and values and the launch's position rows
// into ws, in the matrix cores' fragment order, which must hold
// attn_fast_ws_floats(a.T, a.H, n_chunks) floats.
size_t attn_fast_ws_floats(int T, int H, int n_chunks);
hipError_t launch_attention_fast(const AttnArgs& a, int n_chunks, float* ws, size_t ws_floats, hipStream_t s);
hipError_t launch_glu(const float* in, int ldi, float* out, int ldo, int rows, int D, hipStream_t s);
hipError_t launch_depthwise(const DwArgs& a, int n_chunks, hipStream_t s);
hipError_t launch_transpose(const float* in, float* out, int R, int C, hipStream_t s);

// Pre-encode subsampling (encoder.c:103-174), channel-last [H][W][256].
hipError_t launch_conv0_conv2(const float* mel, int T, int n_mels, const float* w0, const float* b0,
                              const float* w2, const float* b2, float* out, int H1, int W1, int H2, int W2,
                              hipStream_t s);
hipError_t launch_dwconv3x3s2(const float* in, int H, int W, const float* w, const float* b,
                              float* out, int Ho, int Wo, hipStream_t s);
hipError_t launch_flatten_rows(const float* in, float* out, int H, int W, hipStream_t s);
hipError_t launch_scale(float* x, long long n, float sc, hipStream_t s);

}  // namespace pkgpu
