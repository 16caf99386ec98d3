// Host-side launchers of the gfx950 kernels.  Every launcher enqueues on the
// given stream and returns the launch status; none of them synchronises.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>

namespace mch {

// storage type of a device buffer: fp32 or bf16 (the library's 16-bit storage)
enum DType { F32 = 0, BF16 = 1 };

typedef uint16_t bf16_t;

__host__ __device__ inline float bf16_to_f32(bf16_t v)
{
    union { uint32_t u; float f; } c;
    c.u = ((uint32_t)v) << 16;
    return c.f;
}

// round to nearest even; NaN stays NaN
__host__ __device__ inline bf16_t f32_to_bf16(float f)
{
    union { uint32_t u; float f; } c;
    c.f = f;
    if ((c.u & 0x7fffffffu) > 0x7f800000u)
        return (bf16_t)((c.u >> 16) | 0x40);
    uint32_t r = 0x7fffu + ((c.u >> 16) & 1u);
    return (bf16_t)((c.u + r) >> 16);
}

// the largest scratch allocation a kernel object makes, in bytes: no limit, or MYCAFFE_HIP_SCRATCH_LIMIT of the environment at
// its creation
inline size_t scratch_limit()
{
    const char* v = getenv("MYCAFFE_HIP_SCRATCH_LIMIT");
    return v && *v ? (size_t)strtoull(v, nullptr, 10) : SIZE_MAX;
}

// ---- elementwise and layout kernels (ew_kernels.hip) ----------------------
hipError_t k_set(hipStream_t s, DType dt, void* y, size_t n, float v);
hipError_t k_convert(hipStream_t s, DType sdt, const void* src, DType ddt, void* dst, size_t n);
hipError_t k_axpy(hipStream_t s, DType dt, size_t n, float alpha, const void* x, void* y);
hipError_t k_scale(hipStream_t s, DType dt, size_t n, float alpha, const void* x, void* y);
hipError_t k_add(hipStream_t s, DType dt, size_t n, const void* a, const void* b, void* y, float alpha);
hipError_t k_mul(hipStream_t s, DType dt, size_t n, const void* a, const void* b, void* y);
hipError_t k_silu(hipStream_t s, DType dt, size_t n, const void* x, void* y);
hipError_t k_swiglu(hipStream_t s, DType dt, size_t n, const void* a, const void* b, void* y);
hipError_t k_mask(hipStream_t s, DType dt, size_t n, int maskDim, float search, float replace, const void* x,
                  const void* mask, void* y, float xscale = 1.0f);
hipError_t k_mask_batch(hipStream_t s, DType dt, size_t n, int batch, int maskDim, float search, float replace,
                        const void* x, const void* mask, void* y, float xscale = 1.0f);
hipError_t k_transpose(hipStream_t s, DType dt, size_t n, const void* x, void* y, const float* xc, const float* yc,
                       const float* map, int axes);
// the two halves of k_transpose: fetching the stride / map blobs costs a device round trip, so callers keep the result
struct PermuteArgs { int xs[8]; int ys[8]; int map[8]; int axes; };
hipError_t k_transpose_fetch(hipStream_t s, const float* xc, const float* yc, const float* map, int axes, PermuteArgs* out);
hipError_t k_transpose_run(hipStream_t s, DType dt, size_t n, const void* x, void* y, const PermuteArgs& a);
hipError_t k_transpose_hw(hipStream_t s, DType dt, int nc, int h, int w, const void* x, void* y);
hipError_t k_channel_copy(hipStream_t s, DType dt, size_t n, int channels, int blocks, int inner, int offset,
                          void* x, void* y, int dir);
hipError_t k_embed(hipStream_t s, DType wdt, size_t count, const float* ids, const void* w, int N, void* top);
// softmax over `len` for outer x inner independent series; element (o, l, i) at (o*len + l)*inner + i
hipError_t k_softmax(hipStream_t s, DType dt, const void* x, void* y, size_t outer, int len, int inner, bool logsm);
// softmax of mask(x) in one pass (mask semantics of k_mask / k_mask_batch with md1 = maskDim / batch, dd1 = n / batch);
// hipErrorNotSupported when the shape does not fit
// zeroFlag (causal only): a row whose masked entries do not all come out as exact zeros writes `epoch` there
hipError_t k_softmax_masked(hipStream_t s, DType dt, const void* x, void* y, size_t rows, int len, bool logsm, const void* mask,
                            size_t md1, size_t dd1, float search, float replace, float xscale, bool causal = false,
                            int* zeroFlag = nullptr, int epoch = 0);
// gradient with respect to the softmax input from the output y and its gradient dy (dx may alias dy)
// causalT: y is causal (rows of causalT over causalT queries, entries above the diagonal exact zeros unless *zeroFlag == epoch);
// taken into account for inner == 1 and len <= 2048, where dx then has the same zeros, or the flag is raised
// (softmax_bwd_keeps_zeros)
hipError_t k_softmax_bwd(hipStream_t s, DType dt, const void* y, const void* dy, void* dx, size_t outer, int len, int inner, bool logsm,
                         int causalT = 0, int* zeroFlag = nullptr, int epoch = 0);
// *flag = epoch if one of n values at a 16-byte aligned address is infinite or no number
hipError_t k_flag_nonfinite(hipStream_t s, const float* x, size_t n, int* flag, int epoch);
inline bool softmax_bwd_keeps_zeros(int len, int inner) { return inner == 1 && len <= 2048; }
// adjacent-pair rotary embedding with the CudaDnnDLL index rule; x == y allowed
hipError_t k_rope(hipStream_t s, DType dt, size_t n, const void* x, void* y, const float* fcos, const float* fsin,
                  int seqLen, int heads, int hs, int tableOff, bool grad = false);
// LayerNorm without affine part over rows x inner; stdev[rows] keeps sqrt(var + eps) of every row for the gradient.
// Norms with `add`: forward normalises total = x + add (stored), backward adds `add` to dx.
hipError_t k_layernorm_fwd(hipStream_t s, DType dt, int rows, int inner, const void* x, void* y, float* stdev, float eps, const void* add = nullptr,
                           void* total = nullptr);
hipError_t k_layernorm_bwd(hipStream_t s, DType dt, int rows, int inner, const void* y, const void* dy, void* dx,
                           const float* stdev, float bump, const void* add = nullptr);
hipError_t k_gelu_fwd(hipStream_t s, DType dt, size_t n, const void* x, void* y, bool bert);
hipError_t k_gelu_bwd(hipStream_t s, DType dt, size_t n, const void* dy, const void* x, void* dx, bool bert);
hipError_t k_relu_fwd(hipStream_t s, DType dt, size_t n, const void* x, void* y, float slope);
hipError_t k_relu_bwd(hipStream_t s, DType dt, size_t n, const void* dy, const void* y, void* dx, float slope);
hipError_t k_silu_bwd(hipStream_t s, DType dt, size_t n, const void* dy, const void* x, void* dx);
// primitives of the C# RMSNormLayer / LayerNormLayer chains
hipError_t k_powx(hipStream_t s, DType dt, size_t n, const void* a, float alpha, void* y);
hipError_t k_sqrt(hipStream_t s, DType dt, size_t n, const void* x, void* y, float eps);
hipError_t k_invert(hipStream_t s, DType dt, size_t n, const void* x, void* y, float num, float den);
hipError_t k_add_scalar(hipStream_t s, DType dt, size_t n, float alpha, void* y);
hipError_t k_div(hipStream_t s, DType dt, size_t n, const void* a, const void* b, void* y);
hipError_t k_sub(hipStream_t s, DType dt, size_t n, const void* a, const void* b, void* y, size_t nB);
hipError_t k_channel_mean(hipStream_t s, DType dt, size_t rows, int inner, const void* x, void* y);
// y[row] = scale * sum of the row's `inner` values; y[n, s] = sum over the channels of x[n, c, s]
hipError_t k_channel_rowsum(hipStream_t s, DType dt, size_t rows, int inner, const void* x, void* y, float scale);
hipError_t k_channel_colsum(hipStream_t s, DType dt, size_t outer, int channels, int spatial, const void* x, void* y);
// mode 0 fillfrom forward, 1 fillfrom backward, 2 copyall, 3 duplicate (index rules in ew_kernels.hip)
hipError_t k_channel_spread(hipStream_t s, DType dt, int mode, size_t n, size_t spatial, size_t period, size_t channels, void* x, void* y);
hipError_t k_rmsnorm(hipStream_t s, DType dt, int outer, int dim, const void* x, const void* w, void* y, float eps, const void* add = nullptr,
                     void* total = nullptr);
// dw (may be null) is overwritten with the sums of the first dwRows rows; rinv: scratch of `rows` floats, needed with dw
hipError_t k_rmsnorm_bwd(hipStream_t s, DType dt, int rows, int dim, const void* x, const void* w, const void* dy, const void* add, void* dx, void* dw,
                         int dwRows, float* rinv, float eps);
// dx (B*T, 3 H hs) from the head gradients (B,H,T,hs), rotated back when the tables are given (row % seq is the position)
hipError_t k_qkv_heads_grad(hipStream_t s, DType dt, int B, int Tn, int H, int hs, const void* dq, const void* dk, const void* dv, void* dx,
                            const float* fcos, const float* fsin, int seq);
hipError_t k_swiglu_bwd(hipStream_t s, DType dt, size_t n, const void* a, const void* b, const void* dy, void* da, void* db);
// primitives of the CAFFE-engine softmax chain: x is (num, channels, spatial), reduced tensors (num, spatial)
hipError_t k_exp(hipStream_t s, DType dt, size_t n, const void* a, void* y, float beta);
hipError_t k_log(hipStream_t s, DType dt, size_t n, const void* a, void* y, float beta, float alpha);
hipError_t k_channel_max(hipStream_t s, DType dt, size_t num, int channels, int spatial, const void* x, void* y, bool idx, bool across);
hipError_t k_channel_sub(hipStream_t s, DType dt, size_t count, int channels, int spatial, const void* a, const void* x, void* y);
hipError_t k_channel_div(hipStream_t s, DType dt, size_t count, int channels, int spatial, const void* x, void* y);
hipError_t k_channel_dot(hipStream_t s, DType dt, size_t num, int channels, int spatial, const void* x, const void* a, void* y);

// ---- GEMM family (gemm.hip) ------------------------------------------------
// row-major C[m,n] = alpha*op(A)*op(B) + beta*C; A, B, C all of storage type dt
// ws: k_gemm_workspace_bytes(...) bytes of scratch for contractions cut into parts (without it they are not)
hipError_t k_gemm(hipStream_t s, DType dt, bool tA, bool tB, int m, int n, int k, float alpha, const void* A,
                  const void* B, float beta, void* C, void* ws = nullptr, size_t wsBytes = 0);
size_t k_gemm_workspace_bytes(DType dt, bool tA, bool tB, int m, int n, int k, const void* A, const void* B, const void* C);
// Fused QKV projection of CausalSelfAttentionLayer: [q|k|v] = X W^T + bias with X (B*T, C), W (3C, C), C = H*hs, written
// straight into three (B,H,T,hs) tensors.  ws: k_gemm_qkv_heads_workspace_bytes(...) of scratch.
hipError_t k_gemm_qkv_heads(hipStream_t s, DType dt, int B, int T, int H, int hs, const void* X, const void* W, const void* bias,
                            void* q, void* k, void* v, void* ws, size_t wsBytes, const float* fcos = nullptr, const float* fsin = nullptr,
                            int ropeSeq = 0, bool fp32Sums = false);
// Y (m x n) = X (m x k) W^T + bias in one call; ws: k_gemm_bias_workspace_bytes(...) of scratch
hipError_t k_gemm_bias(hipStream_t s, DType dt, int m, int n, int k, const void* X, const void* W, const void* bias, void* Y, void* ws, size_t wsBytes,
                       bool fp32Sums = false);   // fp32Sums: GemmF32
// scratch of k_gemm_bias / k_gemm_qkv_heads with these operands (0: none)
hipError_t k_gemm_bias_heads(hipStream_t s, DType dt, int B, int T, int H, int hs, int k, const void* X, const void* W, const void* bias, void* Y,
                             void* ws, size_t wsBytes, bool fp32Sums = false);   // Y as (B,H,T,hs); scratch as k_gemm_bias
// several of those in 16-bit storage, of one width and contraction, as one launch, if that takes them (*done)
struct HeadsProjection { int m, T; const void *X, *W, *bias; void* Y; };
hipError_t k_gemm_bias_heads_group(hipStream_t s, int count, int n, int k, int H, const HeadsProjection* p, bool* done);
size_t k_gemm_bias_workspace_bytes(DType dt, int m, int n, int k, const void* X, const void* W, const void* Y, bool heads = false);
// whether the call fails without that scratch (otherwise its contraction stays in one part)
bool k_gemm_bias_needs_workspace(DType dt, int m, int n, int k, const void* X, const void* W);
size_t k_gemm_qkv_heads_workspace_bytes(DType dt, int B, int T, int H, int hs, const void* X, const void* W, const void* q, const void* k, const void* v);
// column-major strided batched gemm with BLAS semantics (fp32)
// C (fp32) = alpha X W^T + beta C on the bf16 matrix cores: W 16-bit (n x k), k % 64 == 0; A is X as bf16 (m x k) or,
// split, every row of X as two bf16 rows (nearest bf16, then the bf16 nearest to the remainder; m x 2k)
hipError_t k_gemm_bf16_f32(hipStream_t s, int m, int n, int k, float alpha, const void* A, bool split, const void* W, float beta, float* C);
// the same product with the epilogues of the Llama prompt pass: SwiGLU of the stacked W1 | W3 (bf16 rows of hid, or hi | lo
// rows of 2 hid), and rotation + scatter of the stacked Wq | Wk | Wv into head tensors and caches (gemm_bf16.hip, PromptEpilogue)
hipError_t k_gemm_bf16_swiglu(hipStream_t s, int m, int hid, int k, const void* A, bool split, const void* W13, void* out, bool outSplit);
hipError_t k_gemm_bf16_qkv_rope(hipStream_t s, int B, int P, int H, int kvH, int hs, int k, const void* A, bool split, const void* Wqkv,
                                void* q, void* kh, void* vh, bool heads16, void* kc, void* vc, bool cache16, int seqLen,
                                const float* fcos, const float* fsin);
// causalFlag != nullptr: op(B) (causalA: op(A)) is square, and what lies on one side of its diagonal is known to be exactly
// zero unless *causalFlag == epoch: B(k,j) for k > j, transposed for k < j; A(i,k) for k < i, transposed for k > i.  The
// contraction of a tile of C then stops or begins at the diagonal.
hipError_t k_gemm2(hipStream_t s, bool tA, bool tB, int m, int n, int k, float alpha, const float* A, const float* B,
                   float beta, float* C, int lda, int ldb, int ldc, long long sA, long long sB, long long sC,
                   int batch, const int* causalFlag = nullptr, int epoch = 0, bool skipAboveDiagonal = false, bool causalA = false);
// skipAboveDiagonal (no transposes, m == n, short contraction): entries C(i,j) of tiles that lie wholly at i > j need not
// be computed (their memory is left as it is); other shapes ignore the request
// A row-major (m,n) of type adt; x, y fp32.  y = alpha*A*x + beta*y, or with tA y = alpha*A^T*x + beta*y
size_t k_gemv_workspace_bytes(bool tA, int m, int n);   // scratch for the partial sums of a transposed product over many rows
hipError_t k_gemv(hipStream_t s, DType adt, bool tA, int m, int n, float alpha, const void* A, const float* x,
                  float beta, float* y, void* ws = nullptr, size_t wsBytes = 0);
// which kernel an fp32 product goes to (0 gemm_f32_kernel, 1 gemm_f32_split_kernel, 2 gemm_f32_small_kernel) + 4 its tile + 64 parts of the contraction
int gemm_f32_route(int m, int n, int k, int batch, bool causal, bool fp32Sums, bool heads);
int gemm_b16_route(int m, int n, int k);   // the same of a 16-bit product that goes to gemm_b16_kernel (0)
int linear_bwd_f32_route(int m, int n, int k);   // gradients and bias gradient of an fp32 inner product of m rows, n outputs: 1 one launch, 3 one that adds in levels, 0 neither
hipError_t linear_bwd_f32_small(hipStream_t s, int m, int n, int k, const float* X, const float* W, const float* dY, float* dW, float* db, float* dX, float beta,
                                bool* done);   // the gradients of an inner product as one launch, where sizes and memory allow (*done)
// dW (n x k) += dY^T X and db (n) += column sums of dY (m x n) together; workspace 0: not taken together, one after the other
size_t k_weight_bias_grad_workspace_bytes(DType dt, int m, int n, int k, const void* X, const void* dY, const void* dW, const void* db);
hipError_t k_weight_bias_grad(hipStream_t s, DType dt, int m, int n, int k, const void* X, const void* dY, void* dW, void* db, void* ws, size_t wsBytes);
size_t k_bias_grad_workspace_bytes(int m, int n);
hipError_t k_bias_grad(hipStream_t s, DType dt, int m, int n, const void* dY, void* db, void* ws, size_t wsBytes);   // db += column sums

// ---- attention (attn_prefill.hip, attn_decode.hip) --------------------------
enum MaskKind { MASK_NONE = 0, MASK_QK = 1, MASK_KEY = 2, MASK_BQK = 3, MASK_CAUSAL = 4 };
// q (B,H,Tq,hs), k/v (B,H,Tk,hs), y (B,H,Tq,hs), all dt.  mask is fp32:
//   MASK_QK (Tq,Tk) shared, MASK_KEY (B,Tk), MASK_BQK (B,Tq,Tk); zero entries are filled with -1e29.
//   MASK_CAUSAL needs no mask buffer (lower triangle kept).
// Attention dropout (training mode of the handle, attn.cu:455-486, 578-583): which probabilities survive is a pure
// function of (seed, batch*heads index, query, key), so the backward pass regenerates the mask of the forward call
// instead of storing it.  keep(i) = high 32 bits of splitmix64(seed * 0x9E3779B97F4A7C15 + i) >= threshold, with
// i = ((b*H + h)*Tq + query)*Tk + key and threshold = ratio * 2^32; survivors are scaled by 1 / (1 - ratio).
struct AttnDropout {
    uint64_t seed;
    uint32_t threshold;
    float keepScale;
};
__host__ __device__ inline bool attn_dropout_keep(uint64_t seed, uint64_t index, uint32_t threshold)
{
    uint64_t z = seed * 0x9E3779B97F4A7C15ull + index + 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (uint32_t)(z >> 32) >= threshold;
}
hipError_t k_attn_prefill(hipStream_t s, DType dt, const void* q, const void* k, const void* v, void* y, int B, int H,
                          int Tq, int Tk, int hs, float scale, const float* mask, MaskKind kind, float* lse2 = nullptr,
                          bool yMerged = false, const AttnDropout* dropout = nullptr, bool oneWave = false);
// oneWave: in fp32 a row's sums stay with one wavefront, in the order of its keys, at every size (csrc/flash_traits.h, flash_split_pays).
// yMerged: y is written as (B,Tq,H,hs), the head-merged layout the output projection reads, instead of (B,H,Tq,hs).
// With lse2 ([B*H*Tq] fp32) the forward pass also stores log2 of every row's softmax denominator (scores scaled, masked
// ones at -1e29; -inf marks a row whose keys are all masked), which is all the backward pass needs of the probabilities.
//
// Gradients of the same attention: dq, dk, dv from dy (attn_backward.hip).  lse2 as stored by the forward pass, or
// nullptr to have it recomputed (slow path).  workspace: attn_backward_workspace_bytes(B, H, Tq).
size_t attn_backward_workspace_bytes(int B, int H, int Tq);
hipError_t k_attn_backward(hipStream_t s, DType dt, const void* q, const void* k, const void* v, const void* y, const void* dy,
                           void* dq, void* dk, void* dv, int B, int H, int Tq, int Tk, int hs, float scale, const float* mask,
                           MaskKind kind, const float* lse2, void* workspace, size_t workspaceBytes,
                           const AttnDropout* dropout = nullptr);
// With dropout both calls take the general one-row-per-wavefront kernels (no matrix-core path), and the backward pass
// follows the reference's sequence literally: its softmax backward reads the probabilities AFTER dropout was applied to
// them in place (attn.cu:578-583, 637-646), which gives dS = M / (1 - ratio)^2 * P * (dP - dY.Y) and dV = (P M')^T dY.
size_t attn_decode_workspace_bytes(int B, int H, int hs, int len);
// one query per (b,h): q (B,H,hs), caches addressed as
//   cache[b*strideB + (h/kvMul)*strideH + t*strideT + i], y (B,H,hs).  All dt.
// With dlen set, `len` is only the upper bound used to size the launch and the
// actual number of cached positions is read from *dlen on the device.
hipError_t k_attn_decode(hipStream_t s, DType dt, const void* q, const void* kc, const void* vc, void* y, int B, int H,
                         int kvH, int hs, int len, long long strideB, long long strideH, long long strideT,
                         float scale, void* workspace, size_t workspaceBytes, const int* dlen = nullptr,
                         int* counters = nullptr, const struct DecodeAppend* app = nullptr);
// `counters`: B*H zero-initialised ints that stay zero between launches; when given, the last
// workgroup of every (batch, head) merges the split partials inside the kernel (no second launch).
// With `app` (counters set, no dlen, and attn_decode_appends says so) the call does k_rope_append's work at position len - 1 as well.
struct DecodeAppend { void* knew; const void* vnew; const float *fcos, *fsin; };
bool attn_decode_appends(DType dt, const void* q, const void* kc, const void* vc, const void* y, int B, int H, int kvH, int hs, int len,
                         long long strideB, long long strideH, long long strideT, const DecodeAppend& app);
//
// Decode step of the llama2 engine in one launch: rotate q / k at position *dlen - 1, append k, v to the caches
// ([B][seqLen][kvH*hs], stored as cacheType: fp32, or bf16 with hs a multiple of 8), attend over positions
// 0 .. *dlen - 1, which never exceeds `reach`.  qkv: [B][(H + 2 kvH) hs] raw fp32 projections, y: [B][H*hs] fp32.
// deferMerge (batch 1 with the whole cache in one iteration of rows per split; attn_decode_fused_deferred_splits says whether
// and how many splits): y is not written.  Split s leaves its accumulator of head h at workspace[s * H*hs + h * hs ..] and
// {running maximum, sum} at workspace[splits * H*hs + (s * H + h) * 2 ..] (fp32) for the next kernel of the stream, which
// merges the ceil(*dlen / rowsPerSplit) splits that hold rows (k_llama_matvec_merge in the engine).
hipError_t k_attn_decode_fused(hipStream_t s, const float* qkv, void* kc, void* vc, DType cacheType, float* y, int B, int H, int kvH,
                               int hs, int seqLen, int reach, float scale, const float* fcos, const float* fsin, const int* dlen, void* workspace,
                               size_t workspaceBytes, int* counters, bool deferMerge = false);
int attn_decode_fused_deferred_splits(int B, int H, int hs, int seqLen, int reach, DType cacheType, int* rowsPerSplit);
// rotate q (B,H,hs) and knew (B,kvH,hs) at position pos and append knew/vnew to the caches at pos
hipError_t k_rope_append(hipStream_t s, DType dt, void* q, void* knew, const void* vnew, void* kc, void* vc, int B,
                         int H, int kvH, int hs, int pos, long long strideB, long long strideH, long long strideT,
                         const float* fcos, const float* fsin);

}  // namespace mch
