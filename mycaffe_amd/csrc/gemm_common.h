// Pieces shared by the GEMM kernels (gemm.hip, gemm_f32.hip): vector types, MFMA steps by operand type, and the epilogue
// that adds a bias and writes head tensors.
#pragma once
#include <algorithm>
#include <type_traits>

#include "kernels.h"

namespace mch {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
typedef float floatx2v __attribute__((ext_vector_type(2)));

__device__ inline uint32_t pack2_bf16(float a, float b)
{
    floatx2v f = {a, b};
    bf16x2v r = __builtin_convertvector(f, bf16x2v);
    return *reinterpret_cast<uint32_t*>(&r);
}

template <typename T> __device__ inline float ldf(const T* p, size_t i);
template <> __device__ inline float ldf<float>(const float* p, size_t i) { return p[i]; }
template <> __device__ inline float ldf<bf16_t>(const bf16_t* p, size_t i) { return bf16_to_f32(p[i]); }
template <typename T> __device__ inline void stf(T* p, size_t i, float v);
template <> __device__ inline void stf<float>(float* p, size_t i, float v) { p[i] = v; }
template <> __device__ inline void stf<bf16_t>(bf16_t* p, size_t i, float v) { p[i] = f32_to_bf16(v); }
template <typename T> struct BigTraits;
template <> struct BigTraits<bf16_t> {
    static constexpr int E = 8;   // elements per 16-byte chunk
    __device__ static inline floatx16 mma(u32x4 a, u32x4 b, floatx16 c)
    {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<bf16x8*>(&a), *reinterpret_cast<bf16x8*>(&b), c, 0, 0, 0);
    }
    __device__ static inline float ld(const bf16_t* p) { return bf16_to_f32(*p); }
    __device__ static inline void st(bf16_t* p, float v) { *p = f32_to_bf16(v); }
    __device__ static inline void st4(bf16_t* p, float a, float b, float c, float d)
    {
        uint2 w;
        w.x = pack2_bf16(a, b);
        w.y = pack2_bf16(c, d);
        *(uint2*)p = w;
    }
};
template <> struct BigTraits<float> {
    static constexpr int E = 4;
    __device__ static inline floatx16 mma(u32x4 a, u32x4 b, floatx16 c)
    {
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.x), __uint_as_float(b.x), c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.y), __uint_as_float(b.y), c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.z), __uint_as_float(b.z), c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.w), __uint_as_float(b.w), c, 0, 0, 0);
        return c;
    }
    __device__ static inline float ld(const float* p) { return *p; }
    __device__ static inline void st(float* p, float v) { *p = v; }
    __device__ static inline void st4(float* p, float a, float b, float c, float d) { *(float4*)p = make_float4(a, b, c, d); }
};

// Epilogue of the fused QKV projection (HEADS): row r = (b, t) of the M = B*T rows, column c = (which, h, d) of the
// N = 3*H*hs columns goes, bias added, to element (b, h, t, d) of tensor `which` (q, k, v), i.e. the layout the
// attention kernels read, instead of to C[r][c].  Replaces the bias GEMM, the three channel copies and the three head
// transposes that follow the fused InnerProduct in CausalSelfAttentionLayer.forward (CausalSelfAttentionLayer.cs:526-557).
// With fcos / fsin set (tables [seq][hs/2]) the q and k thirds are also rotated, after their rounding to the storage type:
// adjacent pairs (2i, 2i+1) of row r by the angle of table row r % seq, column i - the rotary embedding that the layer
// applies to q and k in (B,T,H,hs) layout before the head transposes (CausalSelfAttentionLayer.cs:538-545, rope.cu:785-825).
struct HeadsEpilogue { const void* bias; void* dst[3]; int T, H, hs; const float* fcos; const float* fsin; int seq; };

template <typename T>
__device__ __forceinline__ T* heads_dst(const HeadsEpilogue& he, int row, int col)
{
    const int Cd = he.H * he.hs;
    const int which = col / Cd, w = col - which * Cd, h = w / he.hs, d = w - h * he.hs;
    const int b = row / he.T, t = row - b * he.T;
    return (T*)he.dst[which] + (((size_t)b * he.H + h) * he.T + t) * he.hs + d;
}

// (re, im) of one pair of q or k, rotated; the expressions of rope_kernel (ew_kernels.hip)
__device__ __forceinline__ void heads_rope_pair(float c, float sn, float& re, float& im)
{
    const float a = re * c - im * sn, b = re * sn + im * c;
    re = a; im = b;
}

// the rotation applied to one 16-byte piece (columns col .. col + 16 / sizeof(T) - 1 of row `row`; whole pairs of one head)
template <typename T>
__device__ __forceinline__ u32x4 heads_rope_piece(const HeadsEpilogue& he, int row, int col, u32x4 v)
{
    if (!he.fcos || col >= 2 * he.H * he.hs) return v;
    constexpr int NP = 8 / (int)sizeof(T);
    const size_t ti = (size_t)(row % he.seq) * (he.hs >> 1) + ((col % he.hs) >> 1);
    uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < NP; i++) {
        const float c = he.fcos[ti + i], sn = he.fsin[ti + i];
        if constexpr (sizeof(T) == 4) {
            float re = __uint_as_float(w[2 * i]), im = __uint_as_float(w[2 * i + 1]);
            heads_rope_pair(c, sn, re, im);
            w[2 * i] = __float_as_uint(re); w[2 * i + 1] = __float_as_uint(im);
        } else {
            float re = __uint_as_float(w[i] << 16), im = __uint_as_float(w[i] & 0xffff0000u);
            heads_rope_pair(c, sn, re, im);
            w[i] = (uint32_t)f32_to_bf16(re) | ((uint32_t)f32_to_bf16(im) << 16);
        }
    }
    u32x4 o; o.x = w[0]; o.y = w[1]; o.z = w[2]; o.w = w[3];
    return o;
}
template <typename T> struct Quad;
template <> struct Quad<float> {
    __device__ static inline void load(const float* p, float (&v)[4]) { const float4 a = *(const float4*)p; v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; }
    __device__ static inline void store(float* p, const float (&v)[4]) { *(float4*)p = make_float4(v[0], v[1], v[2], v[3]); }
};
template <> struct Quad<bf16_t> {
    __device__ static inline void load(const bf16_t* p, float (&v)[4])
    {
        const uint2 a = *(const uint2*)p;
        v[0] = __uint_as_float(a.x << 16); v[1] = __uint_as_float(a.x & 0xffff0000u);
        v[2] = __uint_as_float(a.y << 16); v[3] = __uint_as_float(a.y & 0xffff0000u);
    }
    __device__ static inline void store(bf16_t* p, const float (&v)[4]) { *(uint2*)p = make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3])); }
};
// C (m x n) = alpha op(A) op(B) + beta C in fp32, row-major (gemm_f32.hip).  op(A) is m x k: stored with k at unit stride
// (aK; row i at A + i lda) or with i at unit stride (row k at A + k lda); op(B) is k x n: stored with k at unit stride (bK;
// column j at B + j ldb) or with j at unit stride (row k at B + k ldb).
struct GemmF32 {
    int m, n, k;
    const float *A, *B;
    float* C;
    long long lda, ldb, ldc, sA, sB, sC;   // row distances; distances between the matrices of a batch
    bool aK, bK;
    float alpha, beta;
    int batch;
    // CAUSAL_*: op(A) (m == k) or op(B) (n == k) is known to be exactly zero on one side of the diagonal unless *flag == epoch
    int causal;
    const int* flag;
    int epoch;
    const HeadsEpilogue* heads;            // written through this epilogue instead of to C (alpha 1, beta 0, batch 1)
};
enum { CAUSAL_NO = 0, CAUSAL_A_LOWER /* A(i,k) zero for k > i */, CAUSAL_A_UPPER /* k < i */, CAUSAL_B_LOWER /* B(k,j) zero for k < j */, CAUSAL_B_UPPER /* k > j */ };
size_t gemm_f32_workspace_bytes(int m, int n, int k, int batch, bool causal);
hipError_t gemm_f32(hipStream_t s, const GemmF32& g, void* ws, size_t wsBytes);

}  // namespace mch
