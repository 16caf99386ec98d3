// Pieces shared by the GEMM kernels (gemm.hip, gemm_f32.hip, gemm_bf16.hip): vector types, MFMA steps by operand type, and the epilogue
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

#define LDS3(p) ((__attribute__((address_space(3))) void*)(p))

// One operand fragment of a bf16 MFMA.  The transposing reads are written as instructions: as builtins the compiler makes each of
// them wait for every fetch into LDS that is under way, the next stage's included (16-bit product of 8000 x 768 x 3072 with one such
// operand: 109 us).  tr_read issues the two reads of a k-step whose first element is OFF bytes from addr (ROWB bytes between k rows),
// tr_wait makes the values usable.  In between the compiler takes the registers for written: should it copy, spill or reuse one
// before the wait, the old contents would go on.  It has no reason to (every fragment is read once, or only after its wait), and
// what it makes of the files that use them is checked: tests/test_asm_pending_reads.py finds no instruction that names a pending
// register, in any of the kernels.
struct TrFragment { union { u32x4 w; uint2 h[2]; }; };
template <int ROWB> __device__ __forceinline__ void tr_read(uint32_t addr, int off, TrFragment& o)
{
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(o.h[0]) : "v"(addr), "n"(off) : "memory");
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(o.h[1]) : "v"(addr), "n"(off + 4 * ROWB) : "memory");
}
__device__ __forceinline__ void tr_wait(TrFragment& o) { asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(o.h[0]), "+v"(o.h[1]) : : "memory"); }

// BYTES (16 or 4) per lane from the buffer to LDS from `lds` on (wavefront-uniform), lane after lane
template <int BYTES> __device__ __forceinline__ void lds_fetch(__amdgpu_buffer_rsrc_t rs, void* lds, uint32_t voffset, int soffset)
{
    static_assert(BYTES == 16 || BYTES == 4, "");
    if constexpr (BYTES == 16) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, LDS3(lds), 16, voffset, soffset, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, LDS3(lds), 4, voffset, soffset, 0, 0);
}

// exchange of 32-row blocks (64 bytes, four 16-byte chunks) in row k of a [k][row] stage: four consecutive k of one block of
// rows have to lie on four different quarters of the 256 bytes of banks; rows are ROWB bytes apart
template <int ROWB> __device__ __forceinline__ int block_swizzle(int k)
{
    return ROWB % 256 == 0 ? (k & 3) * 4 : ((k >> 1) & 1) * 4;   // in chunks; rows 128 bytes apart modulo 256 alternate already
}

// the sum of p[0], p[stride], .. : eight loads under way, and eight sums, so that none is long
__device__ __forceinline__ float sum_partials(const float* p, int count, int stride)
{
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int p0 = 0; p0 < count; p0 += 8) {
        float x[8];
#pragma unroll
        for (int q = 0; q < 8; q++) x[q] = p[(size_t)min(p0 + q, count - 1) * stride];
#pragma unroll
        for (int q = 0; q < 8; q++) v[q] += p0 + q < count ? x[q] : 0.f;
    }
    return ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
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
    __device__ static inline float4 ld4(const bf16_t* p)   // aligned
    {
        const uint2 w = *(const uint2*)p;
        return make_float4(__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u), __uint_as_float(w.y << 16), __uint_as_float(w.y & 0xffff0000u));
    }
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
    __device__ static inline float4 ld4(const float* p) { return *(const float4*)p; }
    __device__ static inline void st4(float* p, float a, float b, float c, float d) { *(float4*)p = make_float4(a, b, c, d); }
};

// Epilogue of the fused QKV projection (HEADS): row r = (b, t) of the M = B*T rows, column c = (which, h, d) of the
// N = 3*H*hs columns goes, bias added, to element (b, h, t, d) of tensor `which` (q, k, v), i.e. the layout the
// attention kernels read, instead of to C[r][c].  Replaces the bias GEMM, the three channel copies and the three head
// transposes that follow the fused InnerProduct in CausalSelfAttentionLayer.forward (CausalSelfAttentionLayer.cs:526-557).
// With fcos / fsin set (tables [seq][hs/2]) the q and k thirds are also rotated, after their rounding to the storage type:
// adjacent pairs (2i, 2i+1) of row r by the angle of table row r % seq, column i - the rotary embedding that the layer
// applies to q and k in (B,T,H,hs) layout before the head transposes (CausalSelfAttentionLayer.cs:538-545, rope.cu:785-825).
// Positions are found without divisions: with m = floor(2^32 / d), n m / 2^32 is at most one below n / d for every n < 2^32.
// (Divided out per 16-byte piece they took 27 of the 74 us of 8000 x 3072 x 768 with its bias, 6 of the 14 us of 8192 x 512 x 512.)
struct HeadsEpilogue {
    const void* bias; void* dst[3]; int T, H, hs; const float* fcos; const float* fsin; int seq;
    uint32_t mT, mC, mhs, mseq;   // floor(2^32 / T), / (H hs), / hs, / seq
    unsigned long long perBatch;  // H T hs
};
static inline HeadsEpilogue heads_epilogue(const void* bias, void* q, void* k, void* v, int T, int H, int hs, const float* fcos, const float* fsin, int seq)
{
    auto magic = [](int d) { const unsigned long long m = (1ull << 32) / (unsigned long long)d; return (uint32_t)(m > 0xffffffffull ? 0xffffffffull : m); };
    HeadsEpilogue he;
    he.bias = bias; he.dst[0] = q; he.dst[1] = k; he.dst[2] = v; he.T = T; he.H = H; he.hs = hs;
    he.fcos = fcos; he.fsin = fsin; he.seq = seq;
    he.perBatch = (unsigned long long)H * T * hs;
    he.mT = magic(T); he.mC = magic(H * hs); he.mhs = magic(hs); he.mseq = magic(seq);
    return he;
}
// as a kernel argument: nothing where the kernel has no such epilogue (a launch with more than 200 bytes of arguments takes
// the host a microsecond longer)
template <bool HEADS> struct HeadsArg { HeadsEpilogue he; };
template <> struct HeadsArg<false> {};
template <bool HEADS> static inline HeadsArg<HEADS> heads_arg(const HeadsEpilogue* he)
{
    HeadsArg<HEADS> a;
    if constexpr (HEADS) a.he = *he;
    return a;
}
__device__ __forceinline__ int heads_div(int n, int d, uint32_t m, int& rem)
{
    int q = (int)__umulhi((uint32_t)n, m);
    rem = n - q * d;
    if (rem >= d) { rem -= d; q++; }
    return q;
}

// address of column `col` in row 0, and what row `row` adds to it
template <typename T>
__device__ __forceinline__ T* heads_col(const HeadsEpilogue& he, int col)
{
    int w, d;
    const int which = heads_div(col, he.H * he.hs, he.mC, w), h = heads_div(w, he.hs, he.mhs, d);
    return (T*)(which == 0 ? he.dst[0] : which == 1 ? he.dst[1] : he.dst[2]) + (size_t)h * he.T * he.hs + d;
}
__device__ __forceinline__ size_t heads_row(const HeadsEpilogue& he, int row, int& t)   // t: the row's position in its sequence
{
    const int b = heads_div(row, he.T, he.mT, t);
    return (size_t)((uint32_t)b * he.perBatch + (unsigned long long)(uint32_t)t * (uint32_t)he.hs);
}
__device__ __forceinline__ size_t heads_row(const HeadsEpilogue& he, int row)
{
    int t;
    return heads_row(he, row, t);
}
template <typename T>
__device__ __forceinline__ T* heads_dst(const HeadsEpilogue& he, int row, int col) { return heads_col<T>(he, col) + heads_row(he, row); }

// index into the rotation's tables for row `row`, column `col`
__device__ __forceinline__ size_t heads_rope_at(const HeadsEpilogue& he, int row, int col)
{
    int p, d;
    heads_div(row, he.seq, he.mseq, p);
    heads_div(col, he.hs, he.mhs, d);
    return (size_t)p * (he.hs >> 1) + (d >> 1);
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
    const size_t ti = heads_rope_at(he, row, col);
    uint32_t w[4] = {v.x, v.y, v.z, v.w};
    // a piece's pairs are whole aligned pieces of the tables too (hs is a multiple of the elements of a piece)
    typedef float Row __attribute__((ext_vector_type(NP)));
    const Row cs = *(const Row*)(he.fcos + ti), sns = *(const Row*)(he.fsin + ti);
#pragma unroll
    for (int i = 0; i < NP; i++) {
        const float c = cs[i], sn = sns[i];
        if constexpr (sizeof(T) == 4) {
            float re = __uint_as_float(w[2 * i]), im = __uint_as_float(w[2 * i + 1]);
            heads_rope_pair(c, sn, re, im);
            w[2 * i] = __float_as_uint(re); w[2 * i + 1] = __float_as_uint(im);
        } else {
            float re = __uint_as_float(w[i] << 16), im = __uint_as_float(w[i] & 0xffff0000u);
            heads_rope_pair(c, sn, re, im);
            w[i] = pack2_bf16(re, im);
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
// whether `n` values at p share memory with `m` values at q
template <typename T> inline bool values_meet(const T* p, long long n, const T* q, long long m)
{
    return p && q && n > 0 && m > 0 && (uintptr_t)p < (uintptr_t)(q + m) && (uintptr_t)q < (uintptr_t)(p + n);
}
// whether what a product of m rows and n columns writes, to C (`count` values) or through `heads`, shares memory with `operand`
template <typename T> inline bool result_meets(const T* C, long long count, const HeadsEpilogue* heads, int m, int n, const T* operand, long long values)
{
    if (!heads) return values_meet(C, count, operand, values);
    const int third = heads->H * heads->hs;
    for (int w = 0; w * third < n; w++)
        if (values_meet((const T*)heads->dst[w], (long long)m * third, operand, values)) return true;
    return false;
}

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
    const float* bias;                     // null, or n values added to every row of C (batch 1)
    const HeadsEpilogue* heads;            // written through this epilogue instead of to C (alpha 1, beta 0, batch 1, bias null)
    bool fp32Sums;                         // on the fp32 matrix cores, the k in order, whatever the size (gemm_f32_kernel)
    float* rowSum;                         // (m) += the sums of op(A)'s rows; dense operands, both with their rows at unit stride
};
enum { CAUSAL_NO = 0, CAUSAL_A_LOWER /* A(i,k) zero for k > i */, CAUSAL_A_UPPER /* k < i */, CAUSAL_B_LOWER /* B(k,j) zero for k < j */, CAUSAL_B_UPPER /* k > j */ };
// a result in the memory of an operand: taken by the kernels that always took such calls, and as before right where one workgroup has all
// that it overwrites (a single tile, or rows of A in place that one tile is wide enough for) or where the contraction is cut into parts
bool gemm_f32_shares(const GemmF32& g);
size_t gemm_f32_workspace_bytes(int m, int n, int k, int batch, bool causal);
size_t gemm_f32_row_sums_workspace_bytes(int m, int n, int k, bool vec);   // with rowSum; vec: operands in whole aligned 16-byte chunks; 0: not taken together
hipError_t gemm_f32(hipStream_t s, const GemmF32& g, void* ws, size_t wsBytes);

// The same in 16-bit storage, dense row-major operands (gemm_bf16.hip): op(A) stored (m, k) or (k, m), op(B) (n, k) or (k, n)
struct GemmB16 {
    int m, n, k;
    const bf16_t *A, *B;
    bf16_t* C;
    bool aK, bK;
    float alpha, beta;
    const bf16_t* bias;   // as in GemmF32
    const HeadsEpilogue* heads;
    bf16_t* rowSum = nullptr;   // (m) += the sums of op(A)'s rows; both operands with their rows at unit stride
};
bool gemm_b16_takes(const GemmB16& g);   // 16-byte chunks of both operands aligned and whole
size_t gemm_b16_workspace_bytes(const GemmB16& g);
size_t gemm_b16_row_sums_workspace_bytes(int m, int n, int k);   // with rowSum; 0: not taken together
hipError_t gemm_b16(hipStream_t s, const GemmB16& g, void* ws, size_t wsBytes);
bool gemm_b16_group(hipStream_t s, const GemmB16* q, int count, hipError_t* e);   // several with heads, of one n and k, as one launch

}  // namespace mch
