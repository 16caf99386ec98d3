// Products of the double base type on the double matrix cores.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "gemm_f64.h"
#include "xcd_runs.h"

namespace mch {

// C(i,j) = alpha sum_k A(i,k) B(k,j) + beta C(i,j) with any element strides, on the double matrix cores
// (v_mfma_f64_16x16x4_f64: lane l holds A(l % 16, l / 16) and B(l / 16, l % 16) of a step, register v of the result is row
// 4 v + l / 16, column l % 16).  2 x 2 wavefronts of W x W MFMA tiles each, stages of 16 k double-buffered in LDS as
// [row][k] with 18 doubles a row (conflict-free 64-bit reads), the next stage held in registers meanwhile.  An operand is
// fetched along whichever index lies at unit stride.
// The layers of this type are small: a product is some dozens of tiles and what bounds it is the latency of one stage after
// the other.  G groups of four wavefronts of a workgroup therefore take every G-th stage each, with stages of their own, and
// their sums are added in order through LDS at the end (256 x 256 x 1024: 27 us with one group, 9 us with four; one output
// per thread took 45 us).
// zdiv: matrix z of C lies at (z / zdiv) sC + (z % zdiv) sC2.  bias (may be null): one value per column, added to every row.
typedef double d_vec4 __attribute__((ext_vector_type(4)));
template <int W, int G> __global__ __launch_bounds__(256 * G) void d_gemm_kernel(GemmD g)
{
    constexpr int BT = 32 * W, BK = 16, LD = BK + 2, NE = BT * BK / 256, STAGE = 2 * BT * LD;
    extern __shared__ double d_smem[];
    const int group = threadIdx.x >> 8, tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;
    double* stages = d_smem + group * 2 * STAGE;   // two of this group
    const int m0 = blockIdx.y * BT, n0 = blockIdx.x * BT, wm = (wave >> 1) * 16 * W, wn = (wave & 1) * 16 * W;
    const double* A = g.A + (size_t)blockIdx.z * g.sA;
    const double* B = g.B + (size_t)blockIdx.z * g.sB;
    double* C = g.C + (size_t)(blockIdx.z / g.zdiv) * g.sC + (size_t)(blockIdx.z % g.zdiv) * g.sC2;
    const bool ak = g.acs == 1, bk = g.brs == 1;
    d_vec4 acc[W][W];
#pragma unroll
    for (int i = 0; i < W; i++)
#pragma unroll
        for (int j = 0; j < W; j++) acc[i][j] = d_vec4{0.0, 0.0, 0.0, 0.0};
    double ra[NE], rb[NE];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int q = 0; q < NE; q++) {
            const int e = tid + 256 * q;
            const int ia = ak ? e / BK : e % BT, ka = ak ? e % BK : e / BT;
            const int jb = bk ? e / BK : e % BT, kb = bk ? e % BK : e / BT;
            ra[q] = (m0 + ia < g.m && k0 + ka < g.k) ? A[(long long)(m0 + ia) * g.ars + (long long)(k0 + ka) * g.acs] : 0.0;
            rb[q] = (n0 + jb < g.n && k0 + kb < g.k) ? B[(long long)(k0 + kb) * g.brs + (long long)(n0 + jb) * g.bcs] : 0.0;
        }
    };
    auto put = [&](int buf) {
        double *as = stages + buf * STAGE, *bs = as + BT * LD;
#pragma unroll
        for (int q = 0; q < NE; q++) {
            const int e = tid + 256 * q;
            as[ak ? (e / BK) * LD + e % BK : (e % BT) * LD + e / BT] = ra[q];
            bs[bk ? (e / BK) * LD + e % BK : (e % BT) * LD + e / BT] = rb[q];
        }
    };
    // trips are the same for every group: stages past the end are zeros
    const int trips = (g.k + BK * G - 1) / (BK * G), fr = lane & 15, fk = lane >> 4;
    fetch(group * BK);
    put(0);
    __syncthreads();
    for (int kt = 0; kt < trips; kt++) {
        const double *as = stages + (kt & 1) * STAGE, *bs = as + BT * LD;
        if (kt + 1 < trips) fetch(((kt + 1) * G + group) * BK);
#pragma unroll
        for (int kk = 0; kk < BK; kk += 4) {
            double a[W], b[W];
#pragma unroll
            for (int t = 0; t < W; t++) {
                a[t] = as[(wm + 16 * t + fr) * LD + kk + fk];
                b[t] = bs[(wn + 16 * t + fr) * LD + kk + fk];
            }
#pragma unroll
            for (int i = 0; i < W; i++)
#pragma unroll
                for (int j = 0; j < W; j++) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        if (kt + 1 < trips) put((kt & 1) ^ 1);
        __syncthreads();
    }
    if (G > 1) {
        // group q > 0 leaves its sums at [q - 1][register][thread]; group 0 adds them
        constexpr int NR = W * W * 4;
        if (group > 0) {
#pragma unroll
            for (int i = 0; i < W; i++)
#pragma unroll
                for (int j = 0; j < W; j++)
#pragma unroll
                    for (int v = 0; v < 4; v++) d_smem[((group - 1) * NR + (i * W + j) * 4 + v) * 256 + tid] = acc[i][j][v];
        }
        __syncthreads();
        if (group > 0) return;
        for (int q = 0; q < G - 1; q++)
#pragma unroll
            for (int i = 0; i < W; i++)
#pragma unroll
                for (int j = 0; j < W; j++)
#pragma unroll
                    for (int v = 0; v < 4; v++) acc[i][j][v] += d_smem[(q * NR + (i * W + j) * 4 + v) * 256 + tid];
    }
#pragma unroll
    for (int i = 0; i < W; i++)
#pragma unroll
        for (int j = 0; j < W; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int r = m0 + wm + 16 * i + 4 * v + fk, c = n0 + wn + 16 * j + fr;
                if (r >= g.m || c >= g.n) continue;
                double* cp = C + (long long)r * g.crs + (long long)c * g.ccs;
                double t = g.alpha * acc[i][j][v];
                if (g.bias) t += g.bias[c];
                *cp = g.beta == 0.0 ? t : t + g.beta * *cp;
            }
}
// ---------------------------------------------------------------------------
// Products of few tiles: 16 x 16 of C to a workgroup, every stage of the contraction dealt to its NW wavefronts, whose sums are added
// up through LDS at the end.  The 64 workgroups of 256 x 256 x 1024 in 32 x 32 tiles leave three quarters of the CUs idle and walk 16 k
// a trip; here there are 256 of them, a stage is 64 k, two stages are under way and three workgroups run on a CU.  What bounds it is
// the latency of the first fetch and of the end (2.7 us), the stages' latencies (0.13 us each beside 0.11 us of MFMA), and from some
// five workgroups a CU on the double matrix cores and what the tiles read.  Stages of 128 k (one workgroup to a CU): 256 x 768 x 256 8.6
// instead of 5.6 us, the same where a CU has one.
// Measured, before and now, us: 256 x 256 x 1024 19.7 -> 7.0, 256 x 256 x 256 7.2 -> 3.8, 256 x 768 x 256 7.6 -> 5.6, 512 x 384 x 1536
// 29.8 -> 17.5, 8 times 128 x 64 x 128 5.2 -> 3.3.
//
// A stage goes from memory straight into LDS.  k at unit stride: [row][k], the 16-byte piece c of row r at c ^ r.  Otherwise [k][row],
// of every eight k first the even ones: a step of the MFMA contracts k = 2 q + e over the four lane groups q, and their 128 bytes are
// then next to each other.  VEC: 16 bytes a lane; otherwise 4, whatever the strides and the alignment.
// rowSums: null, or a value for every row of C to which the sum of the row of A is added (by the tiles of the first columns).
constexpr int D_STAGES = 3;
constexpr int D_TILE_COST = 112;   // what a tile costs beside its contraction, in k (the last term of d_small_time)
template <int BYTES> __device__ __forceinline__ void d_lds_fetch(__amdgpu_buffer_rsrc_t rs, void* lds, uint32_t voffset)
{
    typedef __attribute__((address_space(3))) void* shared_ptr;
    static_assert(BYTES == 16 || BYTES == 4, "");
    if constexpr (BYTES == 16) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (shared_ptr)lds, 16, voffset, 0, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (shared_ptr)lds, 4, voffset, 0, 0, 0);
}

template <int NW, int BK, bool AK, bool BKC, bool VEC, bool HEADS>
__device__ __forceinline__ void d_small_tile(const GemmD& g, const HeadsD& he, int m0, int n0, int z, double* rowSums, double* smem)
{
    constexpr int NT = 64 * NW, S = D_STAGES, STAGE = 2 * 16 * BK;
    constexpr int W = VEC ? 4 : 1, P = 16 * BK * 2 / W / NT;   // 4-byte words per lane and fetch; fetches per thread, operand and stage
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr uint32_t OUTSIDE = 0x80000000u;
    auto resource = [](const void* base) { return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)(OUTSIDE - 16), 0x00020000); };
    // rows past the edge are clamped and never stored, k past the end reads as zeros; double e of a stage
    auto valueK = [&](bool kFast, int e) { return kFast ? (2 * (e % BK / 2 ^ (e / BK)) | (e & 1)) : ((e / 16) & ~7) | ((e / 16 & 3) << 1) | (e / 64 & 1); };
    auto valueRow = [&](bool kFast, int e, int left) { return min(kFast ? e / BK : e % 16, kFast || !VEC ? left - 1 : left - 2); };
    uint32_t va[P], vb[P];
#pragma unroll
    for (int p = 0; p < P; p++) {
        const int w = W * (tid + NT * p), e = w / 2;
        va[p] = 8 * ((uint32_t)valueRow(AK, e, g.m - m0) * (uint32_t)g.ars + (uint32_t)valueK(AK, e) * (uint32_t)g.acs) + 4 * (w & 1);
        vb[p] = 8 * ((uint32_t)valueRow(BKC, e, g.n - n0) * (uint32_t)g.bcs + (uint32_t)valueK(BKC, e) * (uint32_t)g.brs) + 4 * (w & 1);
    }
    const char* stageA = (const char*)(g.A + (size_t)z * g.sA + (size_t)m0 * g.ars);
    const char* stageB = (const char*)(g.B + (size_t)z * g.sB + (size_t)n0 * g.bcs);
    const int nk = (g.k + BK - 1) / BK;
    int fetched = 0;
    auto fetch = [&](double* stage) {
        if (fetched + 1 == nk) {   // what lies past the end of the contraction
#pragma unroll
            for (int p = 0; p < P; p++) {
                const int e = W * (tid + NT * p) / 2;
                if (fetched * BK + valueK(AK, e) >= g.k) va[p] = OUTSIDE;
                if (fetched * BK + valueK(BKC, e) >= g.k) vb[p] = OUTSIDE;
            }
        }
#pragma unroll
        for (int p = 0; p < P; p++) {
            float* to = reinterpret_cast<float*>(stage) + (p * NT + wave * 64) * W;
            d_lds_fetch<4 * W>(resource(stageA), to, va[p]);
            d_lds_fetch<4 * W>(resource(stageB), to + 2 * 16 * BK, vb[p]);
        }
        stageA += 8 * BK * g.acs;
        stageB += 8 * BK * g.brs;
        fetched++;
    };
    const int fr = lane & 15, fq = lane >> 4;
    // unit of eight k: a lane's two
    auto fragment = [&](bool kFast, const double* stage, int unit, double (&o)[2]) {
        if (kFast) {
            const double2 v = *(const double2*)(stage + fr * BK + 2 * ((4 * unit + fq) ^ fr));
            o[0] = v.x; o[1] = v.y;
        } else {
            const double* q = stage + (8 * unit + fq) * 16 + fr;
            o[0] = q[0]; o[1] = q[64];
        }
    };
    d_vec4 acc = {0.0, 0.0, 0.0, 0.0};
    // a row's sum as two, as in gemm_f32.hip
    const bool sumRows = rowSums && n0 == 0;
    constexpr int J = BK / 8 / NW;
    double rowSum[J] = {};
#pragma unroll
    for (int i = 0; i < S - 1; i++)
        if (i < nk) fetch(smem + i * STAGE);
    int buf = 0, free = S - 1;
    for (int kt = 0; kt < nk; kt++) {
        // the stage has landed, of this wavefront and then of all, while the next one is still on its way
        if (kt + S - 2 < nk) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(2 * P * (S - 2)) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" : : : "memory");
        const double* stage = smem + buf * STAGE;
        buf = buf == S - 1 ? 0 : buf + 1;
        const int units = (min(BK, g.k - kt * BK) + 7) / 8;
        double a[J][2], b[J][2];
#pragma unroll
        for (int j = 0; j < J; j++) {
            fragment(AK, stage, wave + NW * j, a[j]);
            fragment(BKC, stage + 16 * BK, wave + NW * j, b[j]);
        }
        if (kt + S - 1 < nk) {   // into the buffer of stage kt - 1, whose fragments every wavefront has had since the barrier
            fetch(smem + free * STAGE);
            free = free == S - 1 ? 0 : free + 1;
        }
#pragma unroll
        for (int j = 0; j < J; j++)
            if (NW * j < units) {
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[j][0], b[j][0], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[j][1], b[j][1], acc, 0, 0, 0);
            }
        if (sumRows)
#pragma unroll
            for (int j = 0; j < J; j++) rowSum[j] += a[j][0] + a[j][1];   // zeros past the end
    }
    __syncthreads();
    constexpr int LD = 17;
#pragma unroll
    for (int v = 0; v < 4; v++) smem[(wave * 16 + 4 * v + fq) * LD + fr] = acc[v];
    if (sumRows) {
        double t = 0.0;
#pragma unroll
        for (int j = 0; j < J; j++) t += rowSum[j];
        smem[NW * 16 * LD + tid] = t;
    }
    __syncthreads();
    if (sumRows && tid < 16 && m0 + tid < g.m) {
        double t = 0.0;
#pragma unroll
        for (int w = 0; w < 4 * NW; w++) t += smem[NW * 16 * LD + 16 * w + tid];
        rowSums[m0 + tid] += t;
    }
    if (tid >= 256) return;
    // along the index of C at unit stride
    const int rl = g.crs == 1 ? tid & 15 : tid >> 4, cl = g.crs == 1 ? tid >> 4 : tid & 15, r = m0 + rl, c = n0 + cl;
    if (r >= g.m || c >= g.n) return;
    auto value = [&](int col) {
        double t = 0.0;
#pragma unroll
        for (int w = 0; w < NW; w++) t += smem[(w * 16 + rl) * LD + col - n0];
        return g.alpha * t + (g.bias ? g.bias[col] : 0.0);
    };
    double v = value(c);
    if constexpr (HEADS) {
        const int C = he.H * he.hs, which = c / C, w = c - which * C, h = w / he.hs, d = w - h * he.hs;
        if (he.fcos && which < 2) {   // pairs of columns (the head size is even)
            const size_t ti = (size_t)(r % he.seq) * (he.hs >> 1) + (d >> 1);
            const double cs = he.fcos[ti], sn = he.fsin[ti], other = value(c ^ 1);
            v = d & 1 ? other * sn + v * cs : v * cs - other * sn;
        }
        he.dst[which][(((size_t)(r / he.T) * he.H + h) * he.T + r % he.T) * he.hs + d] = v;
        return;
    }
    double* cp = g.C + (size_t)(z / g.zdiv) * g.sC + (size_t)(z % g.zdiv) * g.sC2 + (long long)r * g.crs + (long long)c * g.ccs;
    *cp = g.beta == 0.0 ? v : v + g.beta * *cp;
}

// the workgroup's tile: each XCD (workgroup index mod 8) takes a contiguous run of them
__device__ __forceinline__ int d_xcd_item(int total) { return (int)(blockIdx.x % 8) * ((total + 7) / 8) + (int)(blockIdx.x / 8); }

template <int NW, int BK, bool AK, bool BKC, bool VEC, bool HEADS>
__global__ __launch_bounds__(64 * NW) void d_gemm_small_kernel(GemmD g, HeadsD he, int tilesN, int tiles, int total)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char d_smem_raw[];
    const int item = d_xcd_item(total);
    if (item >= total) return;
    const int z = item / tiles, tile = item - z * tiles;
    d_small_tile<NW, BK, AK, BKC, VEC, HEADS>(g, he, tile / tilesN * 16, tile % tilesN * 16, z, nullptr, reinterpret_cast<double*>(d_smem_raw));
}

// the gradients of an inner product as one launch: w is dW += dY^T X, whose first tiles add the column sums of dY to db, x is dX = dY W
// (calls in a row, us, apart and together, 256 rows: 256 to 256 10.6 and 5.1, 1024 to 256 18.4 and 12.0, 256 to 1024 20.6 and 12.1, 256 to 768 14.6 and 9.8; 1024 rows,
// 288 to 768 40 and 29); the longer contraction first, in runs of equal work (xcd_runs.h)
template <int NW, int BK, bool VEC>
__global__ __launch_bounds__(64 * NW) void d_linear_bwd_small_kernel(GemmD w, GemmD x, double* db, int tilesN, int tilesW, int tilesX, XcdRuns runs)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char d_smem_raw[];
    double* smem = reinterpret_cast<double*>(d_smem_raw);
    const int at = runs.first[blockIdx.x % 8] + (int)(blockIdx.x / 8), end = runs.first[blockIdx.x % 8 + 1];
    asm volatile("" : : "s"(w.k), "s"(x.k), "s"(tilesN), "s"(tilesW), "s"(tilesX), "s"(at), "s"(end));   // one trip for the arguments, not one after the other
    if (at >= end) return;
    const int item = w.k >= x.k ? at : at < tilesX ? tilesW + at : at - tilesX;
    if (item < tilesW) d_small_tile<NW, BK, false, false, VEC, false>(w, HeadsD(), item / tilesN * 16, item % tilesN * 16, 0, db, smem);
    else d_small_tile<NW, BK, true, false, VEC, false>(x, HeadsD(), (item - tilesW) / tilesN * 16, (item - tilesW) % tilesN * 16, 0, nullptr, smem);
}

template <int NW, int BK> constexpr int d_small_lds() { static_assert(D_STAGES * 2 * 16 * BK >= NW * (16 * 17 + 64) && D_STAGES * 2 * 16 * BK <= 8192, "room for the sums; no more than any launch gets"); return D_STAGES * 2 * 16 * BK * (int)sizeof(double); }

template <int NW, int BK, bool AK, bool BKC, bool VEC, bool HEADS>
static hipError_t d_launch_small(hipStream_t s, const GemmD& g, const HeadsD& he, int batch)
{
    constexpr int lds = d_small_lds<NW, BK>();
    const int tilesN = (g.n + 15) / 16, tiles = (g.m + 15) / 16 * tilesN, total = tiles * batch;
    hipLaunchKernelGGL((d_gemm_small_kernel<NW, BK, AK, BKC, VEC, HEADS>), (total + 7) / 8 * 8, 64 * NW, lds, s, g, he, tilesN, tiles, total);
    return hipGetLastError();
}

// Estimates in microseconds, fitted to 26 sizes (within 15 %).  Of d_gemm_kernel: one wave of tiles alone on their CUs, and what each
// further one on a CU adds; of the 16 x 16 tiles: what the workgroups of the busiest CU take for their products, and what each three
// of them that run at once (by LDS) take for their stages' latencies.
static double d_tiles_time(long long tiles, double once, double per256, double more, int k)
{
    const long long perCu = std::max(1ll, ((tiles + 7) / 8 + 31) / 32);
    return (once + per256 * k / 256) * (1.0 + more * (double)(perCu - 1));
}
static double d_small_time(long long tiles, int k)
{
    const long long perCu = ((tiles + 7) / 8 + 31) / 32;
    return 1.66 + (double)((perCu + 2) / 3) * (0.71 + 0.23 * k / 128) + (double)perCu * (0.28 + 0.32 * k / 128);
}
// 64 x 64 tiles once they give every CU one, 32 x 32 below; four groups while the workgroups leave CUs to spare (two of
// them fit a CU) and the contraction has stages for them
enum { D_BIG, D_GROUPS, D_PLAIN };
static int d_tiles(int m, int n, int k, int batch, double* time)
{
    const long long big = (long long)((m + 63) / 64) * ((n + 63) / 64) * batch, small = (long long)((m + 31) / 32) * ((n + 31) / 32) * batch;
    const int kind = big >= 256 ? D_BIG : small <= 512 && k >= 128 ? D_GROUPS : D_PLAIN;
    *time = kind == D_BIG ? d_tiles_time(big, 3.7, 17.6, 0.35, k) : kind == D_GROUPS ? d_tiles_time(small, 3.1, 4.15, 0.67, k) : d_tiles_time(small, 2.2, 7.9, 0.35, k);
    return kind;
}
// 31-bit byte offsets within 16 rows of a stage
static bool d_near(long long rowStride, long long kStride) { return rowStride >= 0 && kStride >= 0 && 16 * rowStride + 64 * kStride < (1ll << 27); }
// 16-byte chunks of an operand aligned and whole: along k, or along its rows
static bool d_chunks(const double* p, long long rowStride, long long kStride, int rows, int k, long long batchStride, int batch)
{
    const long long other = kStride == 1 ? rowStride : kStride;
    return (kStride == 1 || rowStride == 1) && ((uintptr_t)p & 15) == 0 && other % 2 == 0 && (kStride == 1 ? k : rows) % 2 == 0 && (batch == 1 || batchStride % 2 == 0);
}

template <bool VEC, bool HEADS> static hipError_t d_launch_layout(hipStream_t s, const GemmD& g, const HeadsD& he, int batch)
{
    // fetched along whichever index lies at unit stride (neither: along k)
    const bool ak = g.ars != 1 || g.acs == 1, bk = g.bcs != 1 || g.brs == 1;
    if constexpr (HEADS) return d_launch_small<4, 64, true, true, VEC, true>(s, g, he, batch);
    if (ak) return bk ? d_launch_small<4, 64, true, true, VEC, false>(s, g, he, batch) : d_launch_small<4, 64, true, false, VEC, false>(s, g, he, batch);
    return bk ? d_launch_small<4, 64, false, true, VEC, false>(s, g, he, batch) : d_launch_small<4, 64, false, false, VEC, false>(s, g, he, batch);
}

struct MemRange { const double* p; size_t n; };
// whether one of the first `out` ranges overlaps another one
static bool shared_memory(const MemRange* r, int out, int all)
{
    for (int i = 0; i < out; i++)
        for (int j = i + 1; j < all; j++)
            if (r[i].n && r[j].n && r[i].p < r[j].p + r[j].n && r[j].p < r[i].p + r[i].n) return true;
    return false;
}

hipError_t d_gemm(hipStream_t s, int batch, int m, int n, int k, double alpha, const double* A, long long ars, long long acs, const double* B,
                  long long brs, long long bcs, double beta, double* C, long long crs, long long ccs, long long sA, long long sB, long long sC,
                  int zdiv, long long sC2, const double* bias)
{
    GemmD g = {m, n, k, alpha, beta, A, B, C, ars, acs, brs, bcs, crs, ccs, sA, sB, sC, sC2, zdiv, bias};
    double time;
    const int kind = d_tiles(m, n, k, batch, &time);
    const long long tiles = (long long)((m + 15) / 16) * ((n + 15) / 16) * batch;
    // a result in an operand's memory stays with the larger tiles: right as before where one workgroup reads all that it overwrites
    auto shares = [&]() {
        const long long last = batch - 1, out = last / zdiv * sC + (zdiv > 1 ? std::min<long long>(last, zdiv - 1) * sC2 : 0) + (m - 1) * crs + (n - 1) * ccs + 1;
        const MemRange mem[] = {{C, (size_t)out}, {A, (size_t)(last * sA + (m - 1) * ars + (k - 1) * acs + 1)}, {B, (size_t)(last * sB + (k - 1) * brs + (n - 1) * bcs + 1)}};
        return shared_memory(mem, 1, 3);
    };
    if (k > 0 && m > 0 && n > 0 && batch > 0 && tiles < (1ll << 24) && d_small_time(tiles, k) < time && d_near(ars, acs) && d_near(bcs, brs) && !shares()) {
        if (d_chunks(A, ars, acs, m, k, sA, batch) && d_chunks(B, bcs, brs, n, k, sB, batch)) return d_launch_layout<true, false>(s, g, HeadsD(), batch);
        return d_launch_layout<false, false>(s, g, HeadsD(), batch);
    }
    const dim3 gridBig((n + 63) / 64, (m + 63) / 64, batch), gridSmall((n + 31) / 32, (m + 31) / 32, batch);
    if (gridSmall.y > 65535) return hipErrorInvalidValue;
    if (kind == D_BIG) hipLaunchKernelGGL((d_gemm_kernel<2, 1>), gridBig, 256, 2 * 2 * 64 * 18 * 8, s, g);
    else if (kind == D_GROUPS) {
        constexpr int lds = 4 * 2 * 2 * 32 * 18 * 8;
        static const hipError_t attr = hipFuncSetAttribute((const void*)d_gemm_kernel<1, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (attr != hipSuccess) return attr;
        hipLaunchKernelGGL((d_gemm_kernel<1, 4>), gridSmall, 1024, lds, s, g);
    } else hipLaunchKernelGGL((d_gemm_kernel<1, 1>), gridSmall, 256, 2 * 2 * 32 * 18 * 8, s, g);
    return hipGetLastError();
}

// X (m x k) W^T (n x k) + bias through `he`, where 16 x 16 tiles are what the size calls for (*done)
hipError_t d_gemm_heads(hipStream_t s, int m, int n, int k, const double* X, const double* W, const double* bias, const HeadsD& he, bool* done)
{
    *done = false;
    double time;
    d_tiles(m, n, k, 1, &time);
    const long long tiles = (long long)((m + 15) / 16) * ((n + 15) / 16);
    // the other kernels write the product first, and a second launch deals it out
    if (tiles >= (1ll << 24) || d_small_time(tiles, k) >= time + 4 || !d_near(k, 1)) return hipSuccess;
    const size_t part = (size_t)m * he.H * he.hs;   // ... after everything has been read: heads over an operand stay with that
    const bool parts = n != he.H * he.hs;
    const MemRange mem[] = {{he.dst[0], part}, {he.dst[1], parts ? part : 0}, {he.dst[2], parts ? part : 0}, {X, (size_t)m * k}, {W, (size_t)n * k}, {bias, bias ? (size_t)n : 0}};
    if (shared_memory(mem, 3, 6)) return hipSuccess;
    *done = true;
    const GemmD g = {m, n, k, 1.0, 0.0, X, W, nullptr, k, 1, 1, k, n, 1, 0, 0, 0, 0, 1, bias};
    if (d_chunks(X, k, 1, m, k, 0, 1) && d_chunks(W, k, 1, n, k, 0, 1)) return d_launch_layout<true, true>(s, g, he, 1);
    return d_launch_layout<false, true>(s, g, he, 1);
}

// The gradients of an inner product as one launch, if that is what the sizes call for (*done): dW (n x k) += dY^T (n x m) X (m x k),
// db (n, or null) += column sums of dY, dX (m x k) = dY W (n x k) + beta dX.
hipError_t d_linear_bwd_small(hipStream_t s, int m, int n, int k, const double* X, const double* W, const double* dY, double* dW, double* db, double* dX,
                              double beta, bool* done)
{
    *done = false;
    // what is written lies apart from everything else: the three calls, one after the other, may share memory
    const MemRange mem[] = {{dW, (size_t)n * k}, {dX, (size_t)m * k}, {db, db ? (size_t)n : 0}, {X, (size_t)m * k}, {W, (size_t)n * k}, {dY, (size_t)m * n}};
    if (shared_memory(mem, 3, 6)) return hipSuccess;
    const long long tilesN = (k + 15) / 16, tilesW = (n + 15) / 16 * tilesN, tilesX = (m + 15) / 16 * tilesN;
    if (tilesW + tilesX > (1ll << 20) || !d_near(1, n) || !d_near(1, k) || !d_near(n, 1)) return hipSuccess;
    double apartW, apartX;
    d_tiles(n, k, m, 1, &apartW);
    d_tiles(m, k, n, 1, &apartX);
    // against the launches apart: the column sums, and 2.5 us for each time that one launch waits for the last one's stores
    const double apart = std::min(apartW, d_small_time(tilesW, m)) + std::min(apartX, d_small_time(tilesX, n)) + 2.5 + (db ? 4.5 : 0.0);
    // the one launch, fitted to 23 sizes (0.8 .. 1.18 of what was measured, 4.6 to 93 us); a tenth on top of it, as both sides are estimates
    const double together = 3.1 + (0.49 * (double)(tilesW + tilesX) + 0.384 / 128 * ((double)tilesW * m + (double)tilesX * n)) / 256 + 0.15 * std::max(m, n) / 128;
    if (1.1 * together >= apart) return hipSuccess;
    const GemmD w = {n, k, m, 1.0, 1.0, dY, X, dW, 1, n, k, 1, k, 1, 0, 0, 0, 0, 1, nullptr}, x = {m, k, n, 1.0, beta, dY, W, dX, n, 1, k, 1, k, 1, 0, 0, 0, 0, 1, nullptr};
    const bool vec = d_chunks(dY, 1, n, n, m, 0, 1) && d_chunks(dY, n, 1, m, n, 0, 1) && d_chunks(X, 1, k, k, m, 0, 1) && d_chunks(W, 1, k, k, n, 0, 1);
    *done = true;
    constexpr int lds = d_small_lds<4, 64>();
    int most;
    const bool wFirst = w.k >= x.k;
    const XcdRuns runs = xcd_runs(wFirst ? tilesW : tilesX, std::max(w.k, x.k), wFirst ? tilesX : tilesW, std::min(w.k, x.k), D_TILE_COST, &most);
    const int grid = 8 * most;
    if (vec) hipLaunchKernelGGL((d_linear_bwd_small_kernel<4, 64, true>), grid, 256, lds, s, w, x, db, (int)tilesN, (int)tilesW, (int)tilesX, runs);
    else hipLaunchKernelGGL((d_linear_bwd_small_kernel<4, 64, false>), grid, 256, lds, s, w, x, db, (int)tilesN, (int)tilesW, (int)tilesX, runs);
    return hipGetLastError();
}

}  // namespace mch
