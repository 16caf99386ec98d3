// GEMM / GEMV kernels for gfx950; the choice of a kernel for a product (k_gemm, k_gemm_bias, k_gemm_qkv_heads).
//
//  * gemm_f32.hip, gemm_bf16.hip : the tiled matrix-core kernels behind most products.
//  * gemm_nt_wide_kernel  : A B^T of sizes that 256 x 288 or (16-bit) 256 x 192 tiles divide, one workgroup per CU.
//  * gemm_generic         : any transpose / stride combination (column-major strided-batched gemm2, sizes the tiles do not
//                           take), 64x64x16 LDS tiles, fp32 FMA.
//  * gemv                 : HBM-bound y = A x, one wavefront per row, 128-bit loads.
#include <algorithm>

#include "gemm_common.h"

namespace mch {

// ---------------------------------------------------------------------------
// generic strided GEMM: C(i,j) = alpha * sum_k A(i,k) B(k,j) + beta * C(i,j)
// element addresses: A[i*ai + k*ak], B[k*bk + j*bj], C[i*ci + j*cj]; blockIdx.z = batch
struct GemmStrides { long long ai, ak, bk, bj, ci, cj, sA, sB, sC; };

template <typename T>
__global__ __launch_bounds__(256) void gemm_generic_kernel(int M, int N, int K, float alpha, const T* __restrict__ A,
                                                           const T* __restrict__ B, float beta, T* __restrict__ C,
                                                           GemmStrides st)
{
    constexpr int BM = 64, BN = 64, BK = 16;
    __shared__ float As[BK][BM + 4];
    __shared__ float Bs[BK][BN + 4];
    A += (size_t)blockIdx.z * st.sA;
    B += (size_t)blockIdx.z * st.sB;
    C += (size_t)blockIdx.z * st.sC;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int tid = threadIdx.x;
    const int tm = (tid / 16) * 4, tn = (tid % 16) * 4;
    // pick the load order that walks the unit-stride axis with consecutive threads
    const bool a_k_fast = st.ak == 1;
    const bool b_k_fast = st.bk == 1;
    float acc[4][4] = {};
    for (int k0 = 0; k0 < K; k0 += BK) {
        for (int e = tid; e < BM * BK; e += 256) {
            int i, k;
            if (a_k_fast) { i = e / BK; k = e % BK; } else { k = e / BM; i = e % BM; }
            float v = 0.f;
            if (m0 + i < M && k0 + k < K) v = ldf(A, (size_t)((long long)(m0 + i) * st.ai + (long long)(k0 + k) * st.ak));
            As[k][i] = v;
        }
        for (int e = tid; e < BN * BK; e += 256) {
            int j, k;
            if (b_k_fast) { j = e / BK; k = e % BK; } else { k = e / BN; j = e % BN; }
            float v = 0.f;
            if (n0 + j < N && k0 + k < K) v = ldf(B, (size_t)((long long)(k0 + k) * st.bk + (long long)(n0 + j) * st.bj));
            Bs[k][j] = v;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < BK; k++) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; i++) a[i] = As[k][tm + i];
#pragma unroll
            for (int j = 0; j < 4; j++) b[j] = Bs[k][tn + j];
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] += a[i] * b[j];
        }
        __syncthreads();
    }
    for (int i = 0; i < 4; i++)
        for (int j = 0; j < 4; j++) {
            int r = m0 + tm + i, c = n0 + tn + j;
            if (r < M && c < N) {
                size_t ci = (size_t)((long long)r * st.ci + (long long)c * st.cj);
                float v = alpha * acc[i][j];
                if (beta != 0.f) v += beta * ldf(C, ci);
                stf(C, ci, v);
            }
        }
}

template <typename T>
static hipError_t launch_generic(hipStream_t s, int M, int N, int K, float alpha, const T* A, const T* B, float beta, T* C,
                                 GemmStrides st, int batch)
{
    if (M <= 0 || N <= 0 || batch <= 0) return hipSuccess;
    dim3 grid((N + 63) / 64, (M + 63) / 64, batch);
    if (grid.y > 65535 || grid.z > 65535) return hipErrorInvalidValue;
    hipLaunchKernelGGL(gemm_generic_kernel<T>, grid, 256, 0, s, M, N, K, alpha, A, B, beta, C, st);
    return hipGetLastError();
}

// A handful of outputs and a short contraction: one workgroup of the scalar kernel is done before a matrix-core tile has its
// first stage in LDS.
static inline bool gemm_is_tiny(int m, int n, int k) { return (long long)m * n <= 1024 && k <= 64; }

// ---------------------------------------------------------------------------
// ---------------------------------------------------------------------------
// NT, one 256 x 288 (WN = 9) or 256 x 192 (WN = 6) tile per workgroup and one workgroup per CU: 8192 x 2304 (the fused
// QKV projection of a 768-wide layer over 8192 tokens) is exactly 256 tiles of 256 x 288, one round of the chip, and a
// stage of K moves half the bytes per flop of the 128 x 128 tile from L2 to LDS.  Eight wavefronts stacked along M,
// 32 rows x 32 WN columns each (WN MFMA tiles, 144 accumulation registers at WN = 9), two per SIMD.
//   * Staging goes from global memory straight into LDS (global_load_lds_dwordx4: lane i of a wavefront lands 16 i bytes
//     past a wavefront-uniform address, so one instruction fills eight 128-byte rows): no staging registers and no
//     ds_write_b128, whose issue nothing covers when a SIMD holds one or two wavefronts.  Rows therefore lie 128 bytes
//     apart without padding, and the 16-byte piece c of row r is kept at position c ^ ((r >> 1) & 7) of its row (the
//     lane that fills position s of row r fetches piece s ^ ((r >> 1) & 7)): a 128-bit read serves sixteen lanes per
//     cycle out of 64 banks, and sixteen consecutive rows (two per 256 bytes of bank space) then fall on sixteen
//     different bank groups.
//   * A k-step is 32 rows of A and 32 WN of B; only RB fragments of B are held: fragment
//     f + RB - 1 of the (k-step, column) sequence is read while fragment f is multiplied.
//   * In 16 bits the products are 16 x 16 x 32, two for a fragment of B, which cost less power than 32 x 32 x 16 (gemm_bf16.hip): 8192 x
//     2304 x 768 34.9 -> 32.5 us, 8192 x 3072 x 768 53.5 -> 48.2, 8192 x 3072 x 12288 553 -> 515, the same bits.
// No edge handling: launched only where the tiles divide the matrix (wide_tile_fits).
// HEADS: 0 none, 1 without a rotation, 2 with.
template <typename T, int WN, int HEADS>
__global__ __launch_bounds__(512, 1) void gemm_nt_wide_kernel(int M, int N, int K, float alpha, const T* __restrict__ A,
                                                               const T* __restrict__ B, T* __restrict__ C, int tilesN,
                                                               int tilesTotal, HeadsEpilogue he)
{
    typedef BigTraits<T> TR;
    constexpr int E = TR::E, BK = 8 * E, BM = 256, BN = 32 * WN;   // a stage is 128 bytes of every row
    constexpr int F = sizeof(T) == 2 ? 16 : 32, TM = 32 / F, TN = WN * TM, PS = 64 / F, KS = 8 / PS;   // rows of a product; its tiles; 16-byte pieces of a row in a k-step
    constexpr int ROWS = BM + BN;                 // rows of one stage: A's 256, then B's 32 WN
    constexpr int STAGE = ROWS * BK;              // elements of one stage buffer
    constexpr int NP = (ROWS + 63) / 64;          // fetch instructions per thread and stage (a wavefront fills 8 rows with each)
    constexpr int RB = 5;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    T* smem = reinterpret_cast<T*>(smem_raw);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int per = (tilesTotal + 7) / 8;         // each XCD (workgroup index mod 8) takes a contiguous run of tiles
    const int tile = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if (tile >= tilesTotal) return;
    const int m0 = (tile / tilesN) * BM, n0 = (tile % tilesN) * BN;
    const int wm = wave * 32;

    typedef std::conditional_t<F == 16, floatx4, floatx16> Sums;
    Sums acc[TM][TN];
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int v = 0; v < F * F / 64; v++) acc[t][j][v] = 0.f;

    // fetch p of a stage: rows 64 p + 8 wave .. + 7 of the stage; this lane fills position tid & 7 of row 64 p + tid / 8.
    // The last fetch covers the 32 rows past a multiple of 64 only: wavefronts 0 .. 3.
    const int lr = tid >> 3;
    const int piece = ((tid & 7) ^ ((lr >> 1) & 7)) * E;
    const T* srcA = A + (size_t)(m0 + lr) * K + piece;
    const T* srcB = B + (size_t)(n0 + lr) * K + piece;
    const size_t passStride = (size_t)64 * K;
    auto fetch = [&](int p, int k0, T* stage) {
        if (p * 64 + wave * 8 >= ROWS) return;   // wavefront-uniform
        const T* src = p < BM / 64 ? srcA + p * passStride + k0 : srcB + (p - BM / 64) * passStride + k0;
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                         (__attribute__((address_space(3))) void*)(stage + (p * 64 + wave * 8) * BK), 16, 0, 0);
    };
    const int nk = K / BK;
#pragma unroll
    for (int p = 0; p < NP; p++) fetch(p, 0, smem);
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): the fetches have landed in LDS
    __syncthreads();

    // fragment of rows base + lane % F, k-step ks: piece PS ks + lane / F, kept at position piece ^ ((row >> 1) & 7)
    const int fr = lane & (F - 1), kp = lane / F;
    int koff[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) koff[ks] = ((PS * ks + kp) ^ ((fr >> 1) & 7)) * E;
    const T* fa = smem + (wm + fr) * BK;
    const T* fb = smem + (BM + fr) * BK;
    u32x4 a[2][TM], b[RB];
    for (int kt = 0; kt < nk; kt++) {
        const T* pa = fa + (kt & 1) * STAGE;
        const T* pb = fb + (kt & 1) * STAGE;
        T* next = smem + ((kt & 1) ^ 1) * STAGE;   // read during stage kt - 1; free since the barrier that ended it
        const int k1 = min(kt + 1, nk - 1) * BK;   // past the end the last stage is fetched again (valid memory, never read)
#pragma unroll
        for (int t = 0; t < TM; t++) a[0][t] = *(const u32x4*)(pa + t * F * BK + koff[0]);
#pragma unroll
        for (int f = 0; f < RB - 1; f++) b[f] = *(const u32x4*)(pb + (f % TN) * F * BK + koff[f / TN]);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            // written in issue order, one scheduling region per tile product: the product, a fragment read, and with
            // each of the stage's first products one fetch of the next stage
#pragma unroll
            for (int j = 0; j < TN; j++) {
#pragma unroll
                for (int t = 0; t < TM; t++) {
                    const u32x4 &x = b[(ks * TN + j) % RB], &y = a[ks & 1][t];
                    if constexpr (F == 16) acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)&x, *(const bf16x8*)&y, acc[t][j], 0, 0, 0);
                    else acc[t][j] = TR::mma(x, y, acc[t][j]);
                }
                const int f = ks * TN + j + RB - 1, fks = f / TN, fj = f % TN;
                if (fks < KS) b[f % RB] = *(const u32x4*)(pb + fj * F * BK + koff[fks]);
                if (j == TN / 2 && ks + 1 < KS)
#pragma unroll
                    for (int t = 0; t < TM; t++) a[(ks + 1) & 1][t] = *(const u32x4*)(pa + t * F * BK + koff[ks + 1]);
                const int n = ks * TN + j;
                if (n < NP) fetch(n, k1, next);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __builtin_amdgcn_s_waitcnt(0x0f70);
        __syncthreads();
    }

    // The products are the transposed tiles, a lane owns row lane % F and register v is column 4 (lane / F) + v (F = 32:
    // 8 (v / 4) + 4 (lane / 32) + v % 4).  Each wavefront passes its 32 rows, CH tiles of columns at
    // a time (in fp32 three: eight slices have to fit the LDS), through its own slice of LDS (free after the last barrier) and
    // stores 16-byte pieces, dealt to the lanes in row-major order.
    constexpr int CH = sizeof(T) == 2 ? WN : 3;
    static_assert(WN % CH == 0, "whole column chunks");
    // A lane keeps its columns while it walks the rows, five at a time: twelve lanes take 192 bytes of one (8192 x 2304 x
    // 768 into heads, 16 bits: 38.6 us with the place of every piece divided out and the bias read value by value, 36.8 so).
    constexpr int CW = 32 * CH, LDC = CW + E, LPR = 12, RPI = 5, NIT = (32 + RPI - 1) / RPI, GW = LPR * E;
    static_assert(CW % GW == 0, "whole groups of columns");
    const int col_l = kp * 4, rr = lane / LPR, cc = (lane % LPR) * E;
    const bool vecBias = ((uintptr_t)he.bias & (4 * sizeof(T) - 1)) == 0;
    T* cs = smem + wave * 32 * LDC;
#pragma unroll
    for (int c = 0; c < WN / CH; c++) {
#pragma unroll
        for (int jj = 0; jj < CH * TM; jj++)
#pragma unroll
            for (int g = 0; g < F * F / 256; g++) {
                const int j = c * CH * TM + jj;
                float4 b = make_float4(0.f, 0.f, 0.f, 0.f);
                if (he.bias) {
                    const T* bp = (const T*)he.bias + n0 + j * F + 8 * g + col_l;
                    if (vecBias) b = TR::ld4(bp);
                    else b = make_float4(TR::ld(bp), TR::ld(bp + 1), TR::ld(bp + 2), TR::ld(bp + 3));
                }
#pragma unroll
                for (int t = 0; t < TM; t++)
                    TR::st4(cs + (t * F + fr) * LDC + jj * F + 8 * g + col_l, alpha * acc[t][j][4 * g] + b.x, alpha * acc[t][j][4 * g + 1] + b.y,
                            alpha * acc[t][j][4 * g + 2] + b.z, alpha * acc[t][j][4 * g + 3] + b.w);
            }
        // same wavefront wrote and reads, and writes the next chunk after it has read this one: LDS operations of one
        // wavefront complete in order
#pragma unroll
        for (int q = 0; q < CW / GW; q++) {
            const int col = n0 + c * CW + q * GW + cc, r0 = m0 + wm + rr;
            T* to;
            size_t step = (size_t)RPI * N, wrap = 0;   // from a row to the one RPI further, and what the next sequence adds to that
            int t = 0;
            if constexpr (HEADS) {
                to = heads_col<T>(he, col) + heads_row(he, r0, t);
                step = (size_t)RPI * he.hs;
                wrap = (size_t)(he.perBatch - (unsigned long long)(uint32_t)he.T * (uint32_t)he.hs);
            } else {
                to = C + (size_t)r0 * N + col;
            }
#pragma unroll
            for (int it = 0; it < NIT; it++) {
                if (rr < RPI && it * RPI + rr < 32) {
                    u32x4 v = *(const u32x4*)(cs + (it * RPI + rr) * LDC + q * GW + cc);
                    if constexpr (HEADS == 2) v = heads_rope_piece<T>(he, r0 + it * RPI, col, v);
                    *(u32x4*)to = v;
                }
                to += step;
                if constexpr (HEADS)
                    for (t += RPI; t >= he.T; t -= he.T) to += wrap;
            }
        }
    }
}

// The wide tiles have no edge handling and one workgroup per CU: they are used where they divide the matrix, fill whole
// rounds of the 256 CUs to at least 85 % and K is long enough to pay for the larger prologue and epilogue.  Returns the
// tile width in MFMA tiles (9: 256 x 288, 6: 256 x 192) or 0.  One stage of K is 128 bytes of a row.
static int wide_tile_fits(int m, int n, int k, int stageElems, const void* A, const void* B, const void* C)
{
    if (m % 256 != 0 || k % stageElems != 0 || k < 8 * stageElems) return 0;
    if ((((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) & 15) != 0) return 0;
    for (int wn : {9, 6}) {
        if (n % (32 * wn) != 0) continue;
        const long long tiles = (long long)(m / 256) * (n / (32 * wn)), rounds = (tiles + 255) / 256;
        if (tiles <= (1ll << 30) && tiles * 100 >= rounds * 256 * 85) return wn;
    }
    return 0;
}

template <typename T, int WN, int HEADS>
static hipError_t launch_wide(hipStream_t s, int m, int n, int k, float alpha, const void* A, const void* B, void* C,
                              const HeadsEpilogue* heads = nullptr)
{
    HeadsEpilogue he = {};
    if (heads) he = *heads;
    constexpr int BN = 32 * WN, E = BigTraits<T>::E, CH = sizeof(T) == 2 ? WN : 3;
    const int tm = m / 256, tn = n / BN, total = tm * tn, per = (total + 7) / 8;
    // two stages of (256 + BN) rows x 128 bytes, or the epilogue's eight slices of 32 x (32 CH + E) elements, whichever is larger
    const size_t lds = std::max((size_t)2 * (256 + BN) * 128, (size_t)8 * 32 * (32 * CH + E) * sizeof(T));
    static bool attr = false;   // per instantiation: allow more than the default 64 KB of dynamic LDS
    if (!attr) {
        hipError_t e = hipFuncSetAttribute((const void*)gemm_nt_wide_kernel<T, WN, HEADS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        attr = true;
    }
    hipLaunchKernelGGL((gemm_nt_wide_kernel<T, WN, HEADS>), dim3(per * 8), 512, lds, s, m, n, k, alpha, (const T*)A, (const T*)B,
                       (T*)C, tn, total, he);
    return hipGetLastError();
}

template <typename T, int WN, bool HEADS>
static hipError_t launch_wide_heads(hipStream_t s, int m, int n, int k, float alpha, const void* A, const void* B, void* C, const HeadsEpilogue* heads)
{
    if constexpr (HEADS) return heads->fcos ? launch_wide<T, WN, 2>(s, m, n, k, alpha, A, B, C, heads) : launch_wide<T, WN, 1>(s, m, n, k, alpha, A, B, C, heads);
    else return launch_wide<T, WN, 0>(s, m, n, k, alpha, A, B, C, heads);
}

template <bool HEADS>
static bool launch_wide_if_fits(hipError_t* e, hipStream_t s, int m, int n, int k, float alpha, const void* A, const void* B, void* C,
                                const HeadsEpilogue* heads = nullptr)
{
    switch (wide_tile_fits(m, n, k, 64, A, B, C)) {
    case 9: *e = launch_wide_heads<bf16_t, 9, HEADS>(s, m, n, k, alpha, A, B, C, heads); return true;
    case 6: *e = launch_wide_heads<bf16_t, 6, HEADS>(s, m, n, k, alpha, A, B, C, heads); return true;
    }
    return false;
}
// fp32 sums (GemmF32): one round of 256 x 288 tiles where 128 x 128 tiles, two to a CU, would leave their last round mostly empty (8192 x
// 2304 x 768: 213 us, 214 us with the bias, against 226 us as three rounds of 128 x 192 and 232 us as 128 x 128); elsewhere
// the tiles of gemm_f32.hip cover the chip as well and hide their ends under a second workgroup.
template <bool HEADS>
static bool launch_wide_f32_if_fits(hipError_t* e, hipStream_t s, int m, int n, int k, float alpha, const void* A, const void* B, void* C,
                                    const HeadsEpilogue* heads = nullptr)
{
    const long long rem = (long long)((m + 127) / 128) * ((n + 127) / 128) % 512;
    if (rem == 0 || rem * 10 >= 512 * 4 || wide_tile_fits(m, n, k, 32, A, B, C) != 9) return false;
    *e = launch_wide_heads<float, 9, HEADS>(s, m, n, k, alpha, A, B, C, heads);
    return true;
}

// K = 1: the rank-1 update C[i,j] = alpha a[i] b[j] + beta C[i,j] that InnerProductLayer uses to add its bias
// (ones (M,1) x bias (1,N), InnerProductLayer.cs:405-414): one streaming pass over C, four columns per thread
template <typename T, bool VEC>
__global__ void gemm_rank1_kernel(int m, int n, float alpha, const T* __restrict__ a, const T* __restrict__ b, float beta, T* C)
{
    const size_t total = (size_t)m * n;
    const size_t items = VEC ? total / 4 : total;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < items; e += (size_t)blockDim.x * gridDim.x) {
        if (VEC) {
            const size_t idx = e * 4;
            const int i = (int)(idx / n), j = (int)(idx % n);
            const float ai = alpha * ldf(a, i);
            float bv[4], cv[4];
            Quad<T>::load(b + j, bv);
            if (beta != 0.f) Quad<T>::load(C + idx, cv);
#pragma unroll
            for (int q = 0; q < 4; q++) cv[q] = beta != 0.f ? ai * bv[q] + beta * cv[q] : ai * bv[q];
            Quad<T>::store(C + idx, cv);
        } else {
            const int i = (int)(e / n), j = (int)(e % n);
            float v = alpha * ldf(a, i) * ldf(b, j);
            if (beta != 0.f) v += beta * ldf(C, e);
            stf(C, e, v);
        }
    }
}

// Fallback of the fused QKV projection: the plain product in `tmp` (M x 3C) is split, bias added, into the three
// (B,H,T,hs) tensors in one pass.
__global__ void qkv_split_heads_kernel(const bf16_t* __restrict__ tmp, size_t total, int N, HeadsEpilogue he)
{
    // one pair of adjacent columns per step (hs is even when the rotation is asked for; otherwise N may be odd)
    const bool pairs = he.fcos != nullptr;
    const size_t steps = pairs ? total / 2 : total;
    for (size_t s = (size_t)blockIdx.x * blockDim.x + threadIdx.x; s < steps; s += (size_t)blockDim.x * gridDim.x) {
        const size_t i = pairs ? 2 * s : s;
        const int r = (int)(i / N), c = (int)(i - (size_t)r * N);
        float o = ldf(tmp, i);
        if (he.bias) o += ldf((const bf16_t*)he.bias, c);
        bf16_t* dp = heads_dst<bf16_t>(he, r, c);
        if (!pairs) { stf(dp, 0, o); continue; }
        float o1 = ldf(tmp, i + 1);
        if (he.bias) o1 += ldf((const bf16_t*)he.bias, c + 1);
        if (c < 2 * he.H * he.hs) {
            stf(dp, 0, o); stf(dp, 1, o1);
            o = ldf(dp, 0); o1 = ldf(dp, 1);                       // the values as the storage type holds them
            const size_t ti = heads_rope_at(he, r, c);
            heads_rope_pair(he.fcos[ti], he.fsin[ti], o, o1);
        }
        stf(dp, 0, o); stf(dp, 1, o1);
    }
}

static GemmB16 b16_product(bool tA, bool tB, int m, int n, int k, float alpha, const void* A, const void* B, float beta, void* C)
{
    return GemmB16{m, n, k, (const bf16_t*)A, (const bf16_t*)B, (bf16_t*)C, !tA, tB, alpha, beta, nullptr, nullptr, nullptr};
}
// X (m x kk) W^T (n x kk) through the tile kernels' HEADS epilogue `he`, or to Y; in 16-bit storage, operands the tile kernels do not
// take go through a scratch matrix (m x n) and a splitting pass
static size_t gemm_heads_workspace_bytes(DType dt, int m, int n, int kk, const void* X, const void* W, const HeadsEpilogue& he, const void* Y)
{
    if (dt == F32) return gemm_f32_workspace_bytes(m, n, kk, 1, false);
    GemmB16 g = b16_product(false, true, m, n, kk, 1.f, X, W, 0.f, (void*)Y);
    if (!Y) g.heads = &he;
    return gemm_b16_takes(g) ? gemm_b16_workspace_bytes(g) : (size_t)m * n * sizeof(bf16_t);
}
bool k_gemm_bias_needs_workspace(DType dt, int m, int n, int k, const void* X, const void* W)
{
    return dt != F32 && !gemm_b16_takes(b16_product(false, true, m, n, k, 1.f, X, W, 0.f, nullptr));
}
size_t k_gemm_bias_workspace_bytes(DType dt, int m, int n, int k, const void* X, const void* W, const void* Y, bool heads)
{
    return gemm_heads_workspace_bytes(dt, m, n, k, X, W, heads_epilogue(nullptr, (void*)Y, nullptr, nullptr, m, 1, n, nullptr, nullptr, 1), heads ? nullptr : Y);
}
size_t k_gemm_qkv_heads_workspace_bytes(DType dt, int B, int T, int H, int hs, const void* X, const void* W, const void* q, const void* k, const void* v)
{
    return gemm_heads_workspace_bytes(dt, B * T, 3 * H * hs, H * hs, X, W, heads_epilogue(nullptr, (void*)q, (void*)k, (void*)v, T, H, hs, nullptr, nullptr, 1), nullptr);
}

// Y: row-major result, only the bias of `he` is added; null: through `he`
static hipError_t gemm_heads_dispatch(hipStream_t s, DType dt, int m, int n, int kk, const void* X, const void* W, const HeadsEpilogue& he, void* Y,
                                      void* ws, size_t wsBytes, bool fp32Sums)
{
    if (dt == F32) {
        GemmF32 g = {};
        g.m = m; g.n = n; g.k = kk;
        g.A = (const float*)X; g.B = (const float*)W;
        g.lda = g.ldb = kk; g.ldc = n;
        g.aK = g.bK = true;
        g.alpha = 1.f; g.batch = 1;
        g.C = (float*)Y;
        if (Y) g.bias = (const float*)he.bias;
        else g.heads = &he;
        g.fp32Sums = fp32Sums;
        hipError_t fit;
        if ((fp32Sums || gemm_f32_shares(g)) && (Y ? launch_wide_f32_if_fits<false>(&fit, s, m, n, kk, 1.f, X, W, Y, &he)
                                                   : he.hs % 4 == 0 && (((uintptr_t)he.dst[1] | (uintptr_t)he.dst[2]) & 15) == 0 &&
                                                         launch_wide_f32_if_fits<true>(&fit, s, m, n, kk, 1.f, X, W, he.dst[0], &he))) return fit;
        return gemm_f32(s, g, ws, wsBytes);
    }
    hipError_t fit;
    if (Y ? launch_wide_if_fits<false>(&fit, s, m, n, kk, 1.f, X, W, Y, &he)
          : he.hs % 8 == 0 && (((uintptr_t)he.dst[1] | (uintptr_t)he.dst[2]) & 15) == 0 &&
                launch_wide_if_fits<true>(&fit, s, m, n, kk, 1.f, X, W, he.dst[0], &he)) return fit;
    GemmB16 g = b16_product(false, true, m, n, kk, 1.f, X, W, 0.f, Y);
    if (Y) g.bias = (const bf16_t*)he.bias;
    else g.heads = &he;
    if (gemm_b16_takes(g)) return gemm_b16(s, g, ws, wsBytes);
    // any other shape: plain product into the caller's scratch matrix, then one splitting pass
    if (!ws || wsBytes < (size_t)m * n * sizeof(bf16_t)) return hipErrorInvalidValue;
    hipError_t e = k_gemm(s, dt, false, true, m, n, kk, 1.f, X, W, 0.f, ws);
    if (e != hipSuccess) return e;
    const size_t total = (size_t)m * n;
    const int grid = (int)std::min<size_t>((total + 255) / 256, 8192);
    hipLaunchKernelGGL(qkv_split_heads_kernel, grid, 256, 0, s, (const bf16_t*)ws, total, n, he);
    return hipGetLastError();
}

hipError_t k_gemm_qkv_heads(hipStream_t s, DType dt, int B, int T, int H, int hs, const void* X, const void* W, const void* bias,
                            void* q, void* k, void* v, void* ws, size_t wsBytes, const float* fcos, const float* fsin, int ropeSeq, bool fp32Sums)
{
    if (fcos && (!fsin || ropeSeq < 1 || (hs & 1))) return hipErrorInvalidValue;
    const int m = B * T, C = H * hs, n = 3 * C, kk = C;
    if (m <= 0 || C <= 0) return hipSuccess;
    const HeadsEpilogue he = heads_epilogue(bias, q, k, v, T, H, hs, fcos, fcos ? fsin : nullptr, fcos ? ropeSeq : 1);
    return gemm_heads_dispatch(s, dt, m, n, kk, X, W, he, nullptr, ws, wsBytes, fp32Sums);
}

// Y (m x n) = X (m x k) W^T (n x k) + bias (n): the inner product layer's forward in one launch (InnerProductLayer.cs:
// 372-417 issues the product and a rank-1 update with a vector of ones).  (One head of n values over m positions, for the
// pass that splits a product the tile kernels do not take.)
hipError_t k_gemm_bias(hipStream_t s, DType dt, int m, int n, int k, const void* X, const void* W, const void* bias, void* Y, void* ws, size_t wsBytes,
                       bool fp32Sums)
{
    if (m <= 0 || n <= 0) return hipSuccess;
    const HeadsEpilogue he = heads_epilogue(bias, Y, Y, Y, m, 1, n, nullptr, nullptr, 1);
    return gemm_heads_dispatch(s, dt, m, n, k, X, W, he, Y, ws, wsBytes, fp32Sums);
}

// the same, Y written head by head: position t of sequence b and column h hs + d go to Y[b][h][t][d] (m = B T, n = H hs)
hipError_t k_gemm_bias_heads(hipStream_t s, DType dt, int B, int T, int H, int hs, int k, const void* X, const void* W, const void* bias, void* Y,
                             void* ws, size_t wsBytes, bool fp32Sums)
{
    if (B <= 0 || T <= 0 || H <= 0 || hs <= 0) return hipSuccess;
    const HeadsEpilogue he = heads_epilogue(bias, Y, Y, Y, T, H, hs, nullptr, nullptr, 1);
    return gemm_heads_dispatch(s, dt, B * T, H * hs, k, X, W, he, nullptr, ws, wsBytes, fp32Sums);
}

hipError_t k_gemm_bias_heads_group(hipStream_t s, int count, int n, int k, int H, const HeadsProjection* p, bool* done)
{
    *done = false;
    if (count < 2 || count > 3) return hipSuccess;
    HeadsEpilogue he[3];
    GemmB16 q[3];
    for (int i = 0; i < count; i++) {
        he[i] = heads_epilogue(p[i].bias, p[i].Y, p[i].Y, p[i].Y, p[i].T, H, n / H, nullptr, nullptr, 1);
        q[i] = b16_product(false, true, p[i].m, n, k, 1.f, p[i].X, p[i].W, 0.f, nullptr);
        q[i].heads = &he[i];
    }
    // a result over another product's operand or result: one after the other
    auto apart = [](const void* a, size_t na, const void* b, size_t nb) { return !a || !b || (const bf16_t*)a + na <= (const bf16_t*)b || (const bf16_t*)b + nb <= (const bf16_t*)a; };
    for (int i = 0; i < count; i++)
        for (int j = 0; j < count; j++) {
            const size_t out = (size_t)p[i].m * n;
            if (!apart(p[i].Y, out, p[j].X, (size_t)p[j].m * k) || !apart(p[i].Y, out, p[j].W, (size_t)n * k) || !apart(p[i].Y, out, p[j].bias, n) ||
                (i != j && !apart(p[i].Y, out, p[j].Y, (size_t)p[j].m * n))) return hipSuccess;
        }
    hipError_t e = hipSuccess;
    *done = gemm_b16_group(s, q, count, &e);
    return e;
}

size_t k_gemm_workspace_bytes(DType dt, bool tA, bool tB, int m, int n, int k, const void* A, const void* B, const void* C)
{
    if (m <= 0 || n <= 0 || k <= 1) return 0;
    if (dt == F32) return gemm_is_tiny(m, n, k) ? 0 : gemm_f32_workspace_bytes(m, n, k, 1, false);
    const GemmB16 g = b16_product(tA, tB, m, n, k, 1.f, A, B, 0.f, (void*)C);
    return gemm_b16_takes(g) ? gemm_b16_workspace_bytes(g) : 0;
}

hipError_t k_gemm(hipStream_t s, DType dt, bool tA, bool tB, int m, int n, int k, float alpha, const void* A,
                  const void* B, float beta, void* C, void* ws, size_t wsBytes)
{
    if (m <= 0 || n <= 0) return hipSuccess;
    if (dt == F32 && k > 1 && !gemm_is_tiny(m, n, k)) {
        GemmF32 g = {};
        g.m = m; g.n = n; g.k = k;
        g.A = (const float*)A; g.B = (const float*)B; g.C = (float*)C;
        g.aK = !tA; g.bK = tB;
        g.lda = tA ? m : k; g.ldb = tB ? k : n; g.ldc = n;
        g.alpha = alpha; g.beta = beta; g.batch = 1;
        hipError_t e;
        if (!tA && tB && beta == 0.f && gemm_f32_shares(g) && launch_wide_f32_if_fits<false>(&e, s, m, n, k, alpha, A, B, C)) return e;
        return gemm_f32(s, g, ws, wsBytes);
    }
    if (dt == BF16 && k > 1) {
        hipError_t e;
        if (!tA && tB && beta == 0.f && launch_wide_if_fits<false>(&e, s, m, n, k, alpha, A, B, C)) return e;
        const GemmB16 g = b16_product(tA, tB, m, n, k, alpha, A, B, beta, C);
        if (gemm_b16_takes(g)) return gemm_b16(s, g, ws, wsBytes);
    }
    if (k == 1) {
        const size_t es = dt == F32 ? 4 : 2;
        const bool vec = n % 4 == 0 && ((((uintptr_t)B | (uintptr_t)C) & (4 * es - 1)) == 0);
        const size_t items = vec ? (size_t)m * n / 4 : (size_t)m * n;
        const int g = (int)std::min<size_t>((items + 255) / 256, 256 * 16);
#define RANK1(TT, V) hipLaunchKernelGGL((gemm_rank1_kernel<TT, V>), g, 256, 0, s, m, n, alpha, (const TT*)A, (const TT*)B, beta, (TT*)C)
        if (dt == F32) { if (vec) RANK1(float, true); else RANK1(float, false); }
        else { if (vec) RANK1(bf16_t, true); else RANK1(bf16_t, false); }
#undef RANK1
        return hipGetLastError();
    }
    if (k <= 0) k = 0;
    GemmStrides st;
    st.ai = tA ? 1 : k;  st.ak = tA ? m : 1;   // A stored (m,k) or (k,m)
    st.bk = tB ? 1 : n;  st.bj = tB ? k : 1;   // B stored (k,n) or (n,k)
    st.ci = n;           st.cj = 1;
    st.sA = st.sB = st.sC = 0;
    if (dt == F32)
        return launch_generic<float>(s, m, n, k, alpha, (const float*)A, (const float*)B, beta, (float*)C, st, 1);
    return launch_generic<bf16_t>(s, m, n, k, alpha, (const bf16_t*)A, (const bf16_t*)B, beta, (bf16_t*)C, st, 1);
}

// ---------------------------------------------------------------------------
// The same product for a short contraction (K = KC of at most 128: Q K^T of the explicit attention chain, K = head size)
// with A(i,k) i-fast and B(k,j) k-fast.  A tile of such a product is all prologue and epilogue for the kernel above: one
// trip to memory for the operands, a few MFMAs, 64 KB of C to write.  Here a workgroup keeps its 128 rows of B (the j
// panel) in registers as MFMA operands for its whole life and walks `tilesPerWg` tiles of 128 i: the next tile's slice of
// A is requested before the current tile is multiplied, and the stores of one pair of 32 x 32 blocks drain under the
// MFMAs of the next (the loads are older than the stores, so waiting for them does not wait for the stores).
template <int KC>
__global__ __launch_bounds__(256, 2) void gemm2_panel_f32_kernel(int M, int N, float alpha, const float* __restrict__ A,
                                                              const float* __restrict__ B, float beta, float* __restrict__ C,
                                                              GemmStrides st, int iChunks, int tilesPerWg, int causal)
{
    constexpr int LDI = 128 + 4, NP = KC * 128 / 4 / 256;       // [k][i] row stride; float4 per thread and tile of A
    extern __shared__ __attribute__((aligned(16))) float panel_smem[];   // two stages of KC x LDI
    A += (size_t)blockIdx.y * st.sA;
    B += (size_t)blockIdx.y * st.sB;
    C += (size_t)blockIdx.y * st.sC;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int jp = blockIdx.x / iChunks;
    const int ic = blockIdx.x % iChunks;
    if (causal) {
        // One workgroup per j panel (iChunks == 1), which walks the tiles up to its diagonal: 1 to gridDim.x of them.
        // Panels are rotated by the batch index and taken in reverse in every other round of 256 workgroups, so that
        // neither a die (workgroup i goes to die i mod 8) nor a CU (i and i + 256 share one) collects the long ones.
        jp = (int)((blockIdx.x + blockIdx.y) % gridDim.x);
        if (((gridDim.x * blockIdx.y) >> 8) & 1) jp = (int)gridDim.x - 1 - jp;
    }
    const int j0 = jp * 128, wj = (wave >> 1) * 64, wi = (wave & 1) * 64;
    const int fr = lane & 31, fg = (lane >> 5) * 4;
    const int t0 = ic * tilesPerWg, nT = (M + 127) / 128;
    int t1 = min(nT, t0 + tilesPerWg);
    if (causal) t1 = min(t1, jp + 1);   // tile t holds i >= 128 t, the panel j <= 128 jp + 127
    if (t0 >= t1) return;

    // B fragments: block a holds rows j0 + wj + 32 a + fr, this lane's four k of every eight
    float4 qf[2][KC / 8];
#pragma unroll
    for (int a = 0; a < 2; a++) {
        const int j = j0 + wj + a * 32 + fr;
        const float* bp = B + (size_t)min(j, N - 1) * st.bj + fg;
#pragma unroll
        for (int q = 0; q < KC / 8; q++) qf[a][q] = *(const float4*)(bp + 8 * q);
    }
    float4 ra[NP];
    // whole: the tile lies inside the matrix (wavefront-uniform), so nothing is masked
    auto gload = [&](int t, bool whole) {
        const int i0 = t * 128;
        if (whole) {
#pragma unroll
            for (int p = 0; p < NP; p++) {
                const int e = tid + p * 256, ig = e & 31, k = e >> 5;
                ra[p] = *(const float4*)(A + (size_t)(i0 + 4 * ig) + (size_t)k * st.ak);
            }
            return;
        }
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const int e = tid + p * 256, ig = e & 31, k = e >> 5;
            ra[p] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (i0 + 4 * ig < M) ra[p] = *(const float4*)(A + (size_t)(i0 + 4 * ig) + (size_t)k * st.ak);
        }
    };
    auto sstore = [&](int buf) {
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const int e = tid + p * 256, ig = e & 31, k = e >> 5;
            *(float4*)(&panel_smem[buf * KC * LDI + k * LDI + 4 * ig]) = ra[p];
        }
    };
    const bool jWhole = j0 + 128 <= N;
    gload(t0, t0 * 128 + 128 <= M);
    sstore(0);
    __syncthreads();
    for (int t = t0; t < t1; t++) {
        const int buf = (t - t0) & 1;
        if (t + 1 < t1) gload(t + 1, (t + 1) * 128 + 128 <= M);
        const float* as = panel_smem + buf * KC * LDI;
        const bool plain = jWhole && t * 128 + 128 <= M && beta == 0.f;   // wavefront-uniform
#pragma unroll
        for (int b = 0; b < 2; b++) {
            floatx16 acc[2];
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[a][v] = 0.f;
#pragma unroll
            for (int q = 0; q < KC / 8; q++) {
                const float* ap = as + (8 * q + fg) * LDI + wi + b * 32 + fr;
                const float fi[4] = {ap[0], ap[LDI], ap[2 * LDI], ap[3 * LDI]};
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int a = 0; a < 2; a++)
                        acc[a] = __builtin_amdgcn_mfma_f32_32x32x2f32(((const float*)&qf[a][q])[e], fi[e], acc[a], 0, 0, 0);
            }
            // accumulator register v of a block: j = 8 (v / 4) + 4 (lane / 32) + v % 4, i = lane % 32
            const int i = t * 128 + wi + b * 32 + fr;
            if (plain) {
#pragma unroll
                for (int a = 0; a < 2; a++) {
                    float* cp = C + (size_t)i + (size_t)(j0 + wj + a * 32 + fg) * st.cj;
#pragma unroll
                    for (int v = 0; v < 16; v++) cp[(size_t)((v >> 2) * 8 + (v & 3)) * st.cj] = alpha * acc[a][v];
                }
            } else if (i < M) {
#pragma unroll
                for (int a = 0; a < 2; a++)
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        const int j = j0 + wj + a * 32 + (v >> 2) * 8 + fg + (v & 3);
                        if (j < N) {
                            const size_t ci = (size_t)i + (size_t)j * st.cj;
                            float o = alpha * acc[a][v];
                            if (beta != 0.f) o += beta * C[ci];
                            C[ci] = o;
                        }
                    }
            }
        }
        if (t + 1 < t1) sstore(buf ^ 1);
        // LDS only: a full __syncthreads() would also wait for this tile's stores of C
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
}

template <int KC>
static hipError_t launch_gemm2_panel(hipStream_t s, int M, int N, float alpha, const float* A, const float* B, float beta, float* C,
                                     const GemmStrides& st, int batch, bool causal)
{
    const int jPanels = (N + 127) / 128, nT = (M + 127) / 128;
    // enough workgroups for two rounds of two per CU, as long as a workgroup keeps two tiles
    int iChunks = 1;
    while (!causal && (long long)jPanels * iChunks * batch < 1024 && nT / (2 * iChunks) >= 2) iChunks *= 2;
    const int tilesPerWg = (nT + iChunks - 1) / iChunks;
    constexpr int lds = 2 * KC * (128 + 4) * 4;
    static bool attr = false;
    if (!attr) {
        hipError_t e = hipFuncSetAttribute((const void*)gemm2_panel_f32_kernel<KC>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return e;
        attr = true;
    }
    dim3 grid(jPanels * iChunks, batch);
    if (grid.y > 65535) return hipErrorInvalidValue;
    hipLaunchKernelGGL(gemm2_panel_f32_kernel<KC>, grid, 256, lds, s, M, N, alpha, A, B, beta, C, st, iChunks, tilesPerWg, causal ? 1 : 0);
    return hipGetLastError();
}

hipError_t k_gemm2(hipStream_t s, bool tA, bool tB, int m, int n, int k, float alpha, const float* A, const float* B,
                   float beta, float* C, int lda, int ldb, int ldc, long long sA, long long sB, long long sC, int batch,
                   const int* causalFlag, int epoch, bool skipAboveDiagonal, bool causalA)
{
    if (causalFlag && (causalA ? m : n) != k) return hipErrorInvalidValue;
    if (skipAboveDiagonal && (tA || tB || m != n || beta != 0.f)) return hipErrorInvalidValue;
    // column-major: op(A)(i,kk) = tA ? A[kk + i*lda] : A[i + kk*lda]
    GemmStrides st;
    st.ai = tA ? lda : 1;  st.ak = tA ? 1 : lda;
    st.bk = tB ? ldb : 1;  st.bj = tB ? 1 : ldb;
    st.ci = 1;             st.cj = ldc;
    st.sA = sA; st.sB = sB; st.sC = sC;
    if (m <= 0 || n <= 0 || batch <= 0) return hipSuccess;
    const bool aligned = ((((uintptr_t)A | (uintptr_t)B) & 15) == 0) && lda % 4 == 0 && ldb % 4 == 0 && sA % 4 == 0 && sB % 4 == 0;
    if (!tA && !tB && aligned && m % 4 == 0 && k % 4 == 0 && m >= 256 && n >= 128 && (long long)m * n * batch >= (1ll << 22)) {
        // a short contraction over large matrices (Q K^T of the attention chain): the j panel stays in registers
        if (k == 32) return launch_gemm2_panel<32>(s, m, n, alpha, A, B, beta, C, st, batch, skipAboveDiagonal);
        if (k == 64) return launch_gemm2_panel<64>(s, m, n, alpha, A, B, beta, C, st, batch, skipAboveDiagonal);
        if (k == 128) return launch_gemm2_panel<128>(s, m, n, alpha, A, B, beta, C, st, batch, skipAboveDiagonal);
    }
    if (k <= 0 || gemm_is_tiny(m, n, k)) return launch_generic<float>(s, m, n, k, alpha, A, B, beta, C, st, batch);
    // column-major C = op(A) op(B) is row-major C^T = op(B)^T op(A)^T
    GemmF32 g = {};
    g.m = n; g.n = m; g.k = k;
    g.A = B; g.B = A; g.C = C;
    g.lda = ldb; g.ldb = lda; g.ldc = ldc; g.sA = sB; g.sB = sA; g.sC = sC;
    g.aK = !tB; g.bK = tA;
    g.alpha = alpha; g.beta = beta; g.batch = batch;
    // MatMul as such keeps the sums it had: P V is one of the products whose rounding decides the mask of a ReLU behind it
    // (TransformerBlockLayer, fp32_sums), and the call does not say what follows.  Likeness, not accuracy, is what that keeps, and it costs
    // where no ReLU follows: 24 times 256 x 48 x 256 8.3 us here, 5.7 as gemm_f32_small_kernel takes it with a transposed operand, which the
    // products of its gradient have.
    g.fp32Sums = !tA && !tB;
    if (causalFlag) { g.causal = causalA ? (tA ? CAUSAL_B_UPPER : CAUSAL_B_LOWER) : (tB ? CAUSAL_A_UPPER : CAUSAL_A_LOWER); g.flag = causalFlag; g.epoch = epoch; }
    return gemm_f32(s, g, nullptr, 0);
}

// ---------------------------------------------------------------------------
// GEMV, not transposed: one wavefront per row, 128-bit loads along the row.
template <typename T> struct VecLoad;
template <> struct VecLoad<float> {
    static constexpr int W = 4;
    __device__ static inline float dot(const float* a, const float* x)
    {
        float4 av = *(const float4*)a, xv = *(const float4*)x;
        return av.x * xv.x + av.y * xv.y + av.z * xv.z + av.w * xv.w;
    }
};
template <> struct VecLoad<bf16_t> {
    static constexpr int W = 8;
    __device__ static inline float dot(const bf16_t* a, const float* x)
    {
        uint4 av = *(const uint4*)a;
        float4 x0 = *(const float4*)x, x1 = *(const float4*)(x + 4);
        const uint32_t u[4] = {av.x, av.y, av.z, av.w};
        const float xs[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            acc += __uint_as_float(u[i] << 16) * xs[2 * i];
            acc += __uint_as_float(u[i] & 0xffff0000u) * xs[2 * i + 1];
        }
        return acc;
    }
};

template <typename T>
__global__ __launch_bounds__(256) void gemv_n_kernel(int m, int n, float alpha, const T* __restrict__ A,
                                                     const float* __restrict__ x, float beta, float* __restrict__ y)
{
    constexpr int W = VecLoad<T>::W;
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= m) return;
    const T* a = A + (size_t)row * n;
    float acc = 0.f;
    const bool vec_ok = (n % W == 0) && (((uintptr_t)a % 16) == 0) && (((uintptr_t)x % 16) == 0);
    if (vec_ok) {
        for (int j = lane * W; j < n; j += 64 * W) acc += VecLoad<T>::dot(a + j, x + j);
    } else {
        for (int j = lane; j < n; j += 64) acc += ldf(a, j) * x[j];
    }
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if (lane == 0) {
        float v = alpha * acc;
        if (beta != 0.f) v += beta * y[row];
        y[row] = v;
    }
}

// transposed: y[j] = sum_i A[i,j] x[i]; consecutive threads walk consecutive columns
template <typename T>
__global__ void gemv_t_kernel(int m, int n, float alpha, const T* __restrict__ A, const float* __restrict__ x, float beta,
                              float* __restrict__ y)
{
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    float acc = 0.f;
    for (int i = 0; i < m; i++) acc += ldf(A, (size_t)i * n + j) * x[i];
    float v = alpha * acc;
    if (beta != 0.f) v += beta * y[j];
    y[j] = v;
}

// The transposed product over many rows (the bias gradient of an inner product layer: A = dY (rows x outputs), x = ones):
// the rows are dealt over workgroups, each leaves one partial row of sums, and a second launch adds the partials in the
// order of their rows - the same sum on every run.  A workgroup is 16 x 16 threads: 16 V columns (V = 4: 256 bytes of a
// row), sixteen rows at a time.
template <typename T, int V>
__global__ __launch_bounds__(256) void gemv_t_part_kernel(int m, int n, int rowsPer, const T* __restrict__ A,
                                                          const float* __restrict__ x, float* __restrict__ part)
{
    __shared__ float red[16][16 * V + 1];
    const int cl = threadIdx.x & 15, rl = threadIdx.x >> 4;
    const int j = (blockIdx.x * 16 + cl) * V;
    const int r0 = blockIdx.y * rowsPer, r1 = min(m, r0 + rowsPer);
    float acc[V];
#pragma unroll
    for (int v = 0; v < V; v++) acc[v] = 0.f;
    if (j < n) {
#pragma unroll 8
        for (int i = r0 + rl; i < r1; i += 16) {
            const float xi = x ? x[i] : 1.f;   // no vector: the plain sum of every column
            const T* a = A + (size_t)i * n + j;
            if (V == 4) {
                float av[4];
                if (sizeof(T) == 4) {
                    const float4 t = *(const float4*)a;
                    av[0] = t.x; av[1] = t.y; av[2] = t.z; av[3] = t.w;
                } else {
                    const uint2 t = *(const uint2*)a;
                    av[0] = __uint_as_float(t.x << 16); av[1] = __uint_as_float(t.x & 0xffff0000u);
                    av[2] = __uint_as_float(t.y << 16); av[3] = __uint_as_float(t.y & 0xffff0000u);
                }
#pragma unroll
                for (int v = 0; v < V; v++) acc[v] = __builtin_fmaf(av[v], xi, acc[v]);
            } else {
                acc[0] = __builtin_fmaf(ldf(a, 0), xi, acc[0]);
            }
        }
    }
#pragma unroll
    for (int v = 0; v < V; v++) red[rl][cl * V + v] = acc[v];
    __syncthreads();
    if (threadIdx.x < 16 * V) {
        const int jj = blockIdx.x * 16 * V + threadIdx.x;
        if (jj < n) {
            float t = 0.f;
#pragma unroll
            for (int r = 0; r < 16; r++) t += red[r][threadIdx.x];
            part[(size_t)blockIdx.y * n + jj] = t;
        }
    }
}

template <typename T>
__global__ void gemv_t_sum_kernel(int n, int chunks, float alpha, const float* __restrict__ part, float beta, T* __restrict__ y)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    float acc = 0.f;
#pragma unroll 8
    for (int c = 0; c < chunks; c++) acc += part[(size_t)c * n + j];
    float v = alpha * acc;
    if (beta != 0.f) v += beta * ldf(y, j);
    stf(y, j, v);
}

// y += column sums of A over at most a thousand rows, one launch: a workgroup takes 16 V columns, 64 rows a trip, and adds the
// sums of its 64 row lanes in order.  (Above that the rows are dealt over workgroups.)
template <typename T, int V>
__global__ __launch_bounds__(1024) void colsum_add_kernel(int m, int n, const T* __restrict__ A, T* __restrict__ y)
{
    __shared__ float red[64][16 * V + 1];
    const int cl = threadIdx.x & 15, rl = threadIdx.x >> 4, j = (blockIdx.x * 16 + cl) * V;
    float acc[V];
#pragma unroll
    for (int v = 0; v < V; v++) acc[v] = 0.f;
    if (j < n)
#pragma unroll 4
        for (int i = rl; i < m; i += 64) {
            const T* a = A + (size_t)i * n + j;
            if constexpr (V == 4 && sizeof(T) == 4) {
                const float4 t = *(const float4*)a;
                acc[0] += t.x; acc[1] += t.y; acc[2] += t.z; acc[3] += t.w;
            } else if constexpr (V == 4) {
                const uint2 t = *(const uint2*)a;
                acc[0] += __uint_as_float(t.x << 16); acc[1] += __uint_as_float(t.x & 0xffff0000u);
                acc[2] += __uint_as_float(t.y << 16); acc[3] += __uint_as_float(t.y & 0xffff0000u);
            } else acc[0] += ldf(a, 0);
        }
#pragma unroll
    for (int v = 0; v < V; v++) red[rl][cl * V + v] = acc[v];
    __syncthreads();
    const int jj = blockIdx.x * 16 * V + threadIdx.x;
    if (threadIdx.x < 16 * V && jj < n) {
        float t = 0.f;
#pragma unroll 8
        for (int q = 0; q < 64; q++) t += red[q][threadIdx.x];
        stf(y, jj, ldf(y, jj) + t);
    }
}

// how the rows of a transposed product are dealt: (columns per thread, rows per workgroup, workgroups along the rows)
static inline int gemv_t_chunks(int m, int colBlocks)
{
    int c = std::max(1, std::min(64, 4096 / colBlocks));
    return std::min(c, (m + 31) / 32);
}
static inline void gemv_t_split(DType adt, int m, int n, const void* A, int* V, int* rowsPer, int* chunks)
{
    const size_t es = adt == F32 ? 4 : 2;
    *V = (n % 4 == 0 && ((uintptr_t)A % (4 * es)) == 0) ? 4 : 1;
    const int c = gemv_t_chunks(m, (n + 16 * *V - 1) / (16 * *V));
    *rowsPer = (m + c - 1) / c;
    *chunks = (m + *rowsPer - 1) / *rowsPer;
}

size_t k_gemv_workspace_bytes(bool tA, int m, int n)
{
    if (!tA || m < 256 || n <= 0) return 0;
    // whichever column count per thread the alignment allows
    return (size_t)std::max(gemv_t_chunks(m, (n + 63) / 64), gemv_t_chunks(m, (n + 15) / 16)) * n * sizeof(float);
}

hipError_t k_gemv(hipStream_t s, DType adt, bool tA, int m, int n, float alpha, const void* A, const float* x, float beta,
                  float* y, void* ws, size_t wsBytes)
{
    if (m <= 0 || n <= 0) return hipSuccess;
    if (!tA) {
        int grid = (m + 3) / 4;
        if (adt == F32)
            hipLaunchKernelGGL(gemv_n_kernel<float>, grid, 256, 0, s, m, n, alpha, (const float*)A, x, beta, y);
        else
            hipLaunchKernelGGL(gemv_n_kernel<bf16_t>, grid, 256, 0, s, m, n, alpha, (const bf16_t*)A, x, beta, y);
    } else if (ws && m >= 256) {
        int V, rowsPer, chunks;
        gemv_t_split(adt, m, n, A, &V, &rowsPer, &chunks);
        if (wsBytes < (size_t)chunks * n * sizeof(float)) return hipErrorInvalidValue;
        float* part = (float*)ws;
        const dim3 grid((n + 16 * V - 1) / (16 * V), chunks);
        if (adt == F32) {
            if (V == 4) hipLaunchKernelGGL((gemv_t_part_kernel<float, 4>), grid, 256, 0, s, m, n, rowsPer, (const float*)A, x, part);
            else hipLaunchKernelGGL((gemv_t_part_kernel<float, 1>), grid, 256, 0, s, m, n, rowsPer, (const float*)A, x, part);
        } else {
            if (V == 4) hipLaunchKernelGGL((gemv_t_part_kernel<bf16_t, 4>), grid, 256, 0, s, m, n, rowsPer, (const bf16_t*)A, x, part);
            else hipLaunchKernelGGL((gemv_t_part_kernel<bf16_t, 1>), grid, 256, 0, s, m, n, rowsPer, (const bf16_t*)A, x, part);
        }
        hipLaunchKernelGGL(gemv_t_sum_kernel<float>, (n + 63) / 64, 64, 0, s, n, chunks, alpha, part, beta, y);
    } else {
        int grid = (n + 255) / 256;
        if (adt == F32)
            hipLaunchKernelGGL(gemv_t_kernel<float>, grid, 256, 0, s, m, n, alpha, (const float*)A, x, beta, y);
        else
            hipLaunchKernelGGL(gemv_t_kernel<bf16_t>, grid, 256, 0, s, m, n, alpha, (const bf16_t*)A, x, beta, y);
    }
    return hipGetLastError();
}

// Bias gradient of an inner product: db (n) += column sums of dY (m x n), both in the storage type.  In 16-bit storage the
// gemv call this replaces widened its vectors in launches of their own: six launches of some 5 us each at 8000 x 3072, two now.
size_t k_bias_grad_workspace_bytes(int m, int n) { return m <= 1024 ? 0 : k_gemv_workspace_bytes(true, m, n); }
template <typename T> static void bias_grad(hipStream_t s, DType dt, int m, int n, const T* dY, T* db, float* part)
{
    if (m <= 1024) {
        if (n % 4 == 0 && ((uintptr_t)dY % (4 * sizeof(T))) == 0) hipLaunchKernelGGL((colsum_add_kernel<T, 4>), (n + 63) / 64, 1024, 0, s, m, n, dY, db);
        else hipLaunchKernelGGL((colsum_add_kernel<T, 1>), (n + 15) / 16, 1024, 0, s, m, n, dY, db);
        return;
    }
    int V, rowsPer, chunks;
    gemv_t_split(dt, m, n, dY, &V, &rowsPer, &chunks);
    const dim3 grid((n + 16 * V - 1) / (16 * V), chunks);
    if (V == 4) hipLaunchKernelGGL((gemv_t_part_kernel<T, 4>), grid, 256, 0, s, m, n, rowsPer, dY, (const float*)nullptr, part);
    else hipLaunchKernelGGL((gemv_t_part_kernel<T, 1>), grid, 256, 0, s, m, n, rowsPer, dY, (const float*)nullptr, part);
    hipLaunchKernelGGL(gemv_t_sum_kernel<T>, (n + 63) / 64, 64, 0, s, n, chunks, 1.f, (const float*)part, 1.f, db);
}
// Weight and bias gradient as one pass over dY (16-bit storage, 8000 rows, 768 to 3072: 69.5 us one after the other, 55.9 together;
// 3072 to 768: 62.5, 56.8; 2048 rows, 512 to 512: 18.0, 11.7; fp32, 8000 rows,
// 768 to 3072: 210, 193).  A bias that
// shares memory with another operand, or a weight gradient that does, is left to the calls one after the other.
size_t k_weight_bias_grad_workspace_bytes(DType dt, int m, int n, int k, const void* X, const void* dY, const void* dW, const void* db)
{
    const size_t es = dt == F32 ? 4 : 2;
    const size_t mk = (size_t)m * k * es, mn = (size_t)m * n * es, nk = (size_t)n * k * es;
    auto meet = [](const void* a, size_t na, const void* b, size_t nb) { return values_meet((const char*)a, (long long)na, (const char*)b, (long long)nb); };
    if (meet(db, es * n, X, mk) || meet(db, es * n, dY, mn) || meet(db, es * n, dW, nk) || meet(dW, nk, X, mk) || meet(dW, nk, dY, mn)) return 0;
    if (dt == F32) return gemm_f32_row_sums_workspace_bytes(n, k, m, (((uintptr_t)X | (uintptr_t)dY) & 15) == 0 && n % 4 == 0 && k % 4 == 0);
    return gemm_b16_takes(b16_product(true, false, n, k, m, 1.f, dY, X, 1.f, nullptr)) ? gemm_b16_row_sums_workspace_bytes(n, k, m) : 0;
}
hipError_t k_weight_bias_grad(hipStream_t s, DType dt, int m, int n, int k, const void* X, const void* dY, void* dW, void* db, void* ws, size_t wsBytes)
{
    if (dt == F32) {
        GemmF32 g = {};
        g.m = n; g.n = k; g.k = m;
        g.A = (const float*)dY; g.B = (const float*)X; g.C = (float*)dW;
        g.lda = n; g.ldb = g.ldc = k;
        g.alpha = g.beta = 1.f; g.batch = 1;
        g.rowSum = (float*)db;
        return gemm_f32(s, g, ws, wsBytes);
    }
    GemmB16 g = b16_product(true, false, n, k, m, 1.f, dY, X, 1.f, dW);
    g.rowSum = (bf16_t*)db;
    return gemm_b16(s, g, ws, wsBytes);
}
hipError_t k_bias_grad(hipStream_t s, DType dt, int m, int n, const void* dY, void* db, void* ws, size_t wsBytes)
{
    if (m <= 0 || n <= 0) return hipSuccess;
    if (wsBytes < k_bias_grad_workspace_bytes(m, n)) return hipErrorInvalidValue;
    if (dt == F32) bias_grad<float>(s, dt, m, n, (const float*)dY, (float*)db, (float*)ws);
    else bias_grad<bf16_t>(s, dt, m, n, (const bf16_t*)dY, (bf16_t*)db, (float*)ws);
    return hipGetLastError();
}

}  // namespace mch
