// fp32 GEMM on the fp32 matrix cores (v_mfma_f32_32x32x2_f32), any operand layout, gfx950.
//
// One kernel serves the inner products (A B^T), their gradients (A B and A^T B) and the batched products of the explicit
// attention chain.  2 x 2 wavefronts, each owning WM x WN MFMA tiles of 32 x 32, so a workgroup covers (64 WM) x (64 WN) of
// C and walks K in stages of 32 through a double-buffered LDS stage, one barrier per stage.  What bounds it is the matrix
// core: a 32x32x2 step is 64 cycles, so a stage of a 128 x 128 tile is 4096 cycles of MFMA per wavefront against some 40
// LDS and 16 global instructions, and everything else only has to stay out of its way - the instructions of the next
// fragments and stages are issued one by one between the products, in the order written (sched_barrier).
//
// An operand with k at unit stride lies in LDS as [row][k] (stride 36: conflict-free 128-bit reads; a lane's four k of every
// eight feed four MFMA steps, lane half h holding 4h .. 4h+3, step e contracting {e, 4 + e}).  One with the row index at unit
// stride lies as it is stored, [k][row], and a lane gathers its four k with 32-bit reads (stride the tile's rows, a multiple
// of 64 words, so that every read is an immediate offset from one address; odd groups of four k have rows r and r ^ 32
// swapped, so that the two lane halves, four k apart, fall on the two halves of the 64 banks): at the rate of the fp32 MFMA four reads cost
// no more than one, so no operand is transposed in memory first (transposing took 14 % of a weight gradient's time).
//
// Operands are fetched with buffer loads: an offset per chunk that never changes, the stage in the scalar offset, so a fetch
// is one instruction, and the contraction may end anywhere: a chunk past its end gets an offset out of the buffer's range,
// which reads as zeros.  (Vector instructions are not free next to the fp32 MFMA: a 64-bit address per fetch and a select per
// register on the way to LDS cost 6 % of a whole product.)
#include "gemm_common.h"

namespace mch {

struct GemmF32Args {
    int M, N, K;
    const float *A, *B;
    float* C;
    long long lda, ldb, ldc, sA, sB, sC;
    float alpha, beta;
    int tilesM, tilesN, parts, kChunk, causal, epoch;   // parts: of the contraction, or matrices of the batch
    const int* flag;
    float* part;              // kChunk < K: partial products, [split][M][N]
    bool vecC;                // C rows can be read and written in 16-byte pieces
    const float* bias;
};

// the bias of four columns from c on (0 past the matrix)
__device__ __forceinline__ float4 f32_bias4(const float* bias, int c, int N)
{
    if (!bias) return make_float4(0.f, 0.f, 0.f, 0.f);
    const float* b = bias + c;
    return make_float4(b[0], c + 1 < N ? b[1] : 0.f, c + 2 < N ? b[2] : 0.f, c + 3 < N ? b[3] : 0.f);
}

// four consecutive values of row r from column c on (a multiple of 4), bias added, through the heads epilogue; column c of
// row 0 is at col
__device__ __forceinline__ void heads_store4(const HeadsEpilogue& he, int r, int c, int N, bool vec, float* col, float (&v)[4])
{
    if (vec) {
        u32x4 p;
        p.x = __float_as_uint(v[0]); p.y = __float_as_uint(v[1]); p.z = __float_as_uint(v[2]); p.w = __float_as_uint(v[3]);
        *(u32x4*)(col + heads_row(he, r)) = heads_rope_piece<float>(he, r, c, p);
        return;
    }
#pragma unroll
    for (int q = 0; q < 4; q += 2) {
        // a rotation needs an even head size: a pair of columns is inside the matrix and one head, or outside
        if (c + q >= N) continue;
        if (he.fcos && c + q < 2 * he.H * he.hs) {
            const size_t ti = heads_rope_at(he, r, c + q);
            heads_rope_pair(he.fcos[ti], he.fsin[ti], v[q], v[q + 1]);
        }
        *heads_dst<float>(he, r, c + q) = v[q];
        if (c + q + 1 < N) *heads_dst<float>(he, r, c + q + 1) = v[q + 1];
    }
}

// VEC: every 16-byte chunk of an operand is aligned and lies inside it or outside as a whole
template <int WM, int WN, int OCC, bool AK, bool BKC, bool VEC, bool HEADS>
__global__ __launch_bounds__(256, OCC) void gemm_f32_kernel(GemmF32Args g, HeadsArg<HEADS> hp)
{
    constexpr int BK = 32, BM = 64 * WM, BN = 64 * WN, LDK = BK + 4;
    constexpr int LDA = AK ? LDK : BM, LDB = BKC ? LDK : BN;
    constexpr int SA = AK ? BM * LDK : BK * LDA, SB = BKC ? BN * LDK : BK * LDB;   // floats of one stage
    constexpr int PA = BM * BK / 4 / 256, PB = BN * BK / 4 / 256;                   // 16-byte chunks per thread and stage
    constexpr int KS = 4, NMF = WM * WN, HALF = KS / 2;
    constexpr int RF = (WM + WN + NMF - 1) / NMF;
    constexpr int SC = ((PA + PB + HALF - 1) / HALF + NMF - 1) / NMF;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    float* As = reinterpret_cast<float*>(smem_raw);
    float* Bs = As + 2 * SA;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // Work items are the tiles of every part of the contraction, or of every matrix of the batch; each XCD (workgroup index
    // mod 8) takes a contiguous run of them, so all dies get the same share whatever the tile count of one part.
    const int tiles = g.tilesM * g.tilesN, total = tiles * g.parts, per = (total + 7) / 8;
    const int item = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if (item >= total) return;
    const int part = item / tiles, tile = item - part * tiles;
    const bool split = g.kChunk < g.K;
    const int batch = split ? 0 : part;
    // tiles are numbered in groups of GROUP tile rows, down a group's rows first: the tiles an XCD has in flight then share
    // few enough rows of A and columns of B for its 4 MB of L2
    constexpr int GROUP = 8;
    const int group = tile / (GROUP * g.tilesN), inGroup = tile - group * GROUP * g.tilesN;
    const int groupRows = min(GROUP, g.tilesM - group * GROUP);
    int tr = group * GROUP + inGroup % groupRows;
    int tc = inGroup / groupRows;
    bool causal = false;
    if (g.causal) {
        // tiles differ in length along one side: every other round of an XCD's 32 CUs takes them in reverse, so that a CU
        // that had a long one gets a short one (decided per matrix, so that each of its tiles is still taken once)
        if (((batch * tiles) >> 5) & 1) {
            if (g.causal >= CAUSAL_B_LOWER) tc = g.tilesN - 1 - tc;
            else tr = g.tilesM - 1 - tr;
        }
        causal = *g.flag != g.epoch;
    }
    const int M = g.M, N = g.N;
    const int m0 = tr * BM, n0 = tc * BN;
    int kBegin = split ? part * g.kChunk : 0, kEnd = min(g.K, kBegin + g.kChunk);
    if (causal) {
        if (g.causal == CAUSAL_A_LOWER) kEnd = min(kEnd, m0 + BM);
        else if (g.causal == CAUSAL_A_UPPER) kBegin = m0;
        else if (g.causal == CAUSAL_B_LOWER) kBegin = n0;
        else kEnd = min(kEnd, n0 + BN);
    }
    const float* __restrict__ A = g.A + (size_t)batch * g.sA;
    const float* __restrict__ B = g.B + (size_t)batch * g.sB;
    const int wm = (wave >> 1) * (32 * WM), wn = (wave & 1) * (32 * WN);

    floatx16 acc[WM][WN];
#pragma unroll
    for (int i = 0; i < WM; i++)
#pragma unroll
        for (int j = 0; j < WN; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;

    // chunk c of a stage, k at unit stride: row tid / 8 + 32 c, k = 4 (tid % 8);
    // row at unit stride: k = (tid + 256 c) / (rows / 4), rows 4 ((tid + 256 c) % (rows / 4)) .. + 3
    const int lr = tid >> 3, lc = (tid & 7) * 4;
    // rows past the matrix edge are clamped: fetched (valid memory) and never stored
    const float* ga[PA];
    const float* gb[PB];
    // VEC: the same as byte offsets from a buffer resource that begins at the tile, and where the row index is at unit stride
    // at the stage, so that operands of any size are reached with 32 bits
    const float* baseA = A + (AK ? (size_t)m0 * g.lda : (size_t)m0);
    const float* baseB = B + (BKC ? (size_t)n0 * g.ldb : (size_t)n0);
    uint32_t va[PA], vb[PB];
#pragma unroll
    for (int p = 0; p < PA; p++) {
        const int e = tid + 256 * p, row = 4 * (e % (BM / 4));
        ga[p] = baseA + (AK ? (size_t)min(lr + p * 32, M - 1 - m0) * g.lda + lc : (size_t)(e / (BM / 4)) * g.lda + row);
        va[p] = 4 * (AK ? (uint32_t)min(lr + p * 32, M - 1 - m0) * (uint32_t)g.lda + lc : (uint32_t)(e / (BM / 4)) * (uint32_t)g.lda + min(row, M - 4 - m0));
    }
#pragma unroll
    for (int p = 0; p < PB; p++) {
        const int e = tid + 256 * p, row = 4 * (e % (BN / 4));
        gb[p] = baseB + (BKC ? (size_t)min(lr + p * 32, N - 1 - n0) * g.ldb + lc : (size_t)(e / (BN / 4)) * g.ldb + row);
        vb[p] = 4 * (BKC ? (uint32_t)min(lr + p * 32, N - 1 - n0) * (uint32_t)g.ldb + lc : (uint32_t)(e / (BN / 4)) * (uint32_t)g.ldb + min(row, N - 4 - n0));
    }
    constexpr uint32_t OUTSIDE = 0x80000000u;
    auto resource = [](const void* base) { return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)(OUTSIDE - 16), 0x00020000); };
    const __amdgpu_buffer_rsrc_t rsA = resource(baseA), rsB = resource(baseB);
    // where resources begin at stages: the stage that is fetched next, and the way to the one after it (0 from the last on).
    // Added up and not multiplied out: the scalar instructions of a stage show (gradients at 1000 x 32000 x 768: 0.5 %).
    const char *stageA = (const char*)(baseA + (size_t)kBegin * g.lda), *stageB = (const char*)(baseB + (size_t)kBegin * g.ldb);
    long long stepA = (long long)(BK * sizeof(float)) * g.lda, stepB = (long long)(BK * sizeof(float)) * g.ldb;
    auto advance = [&]() {
        if (!AK) stageA += stepA;
        if (!BKC) stageB += stepB;
    };
    u32x4 ra[PA], rb[PB];

    // before the last stage is fetched, once: the chunks past the end of the contraction
    auto lastStage = [&](int k0) {
        if (!VEC) return;
        stepA = stepB = 0;
#pragma unroll
        for (int p = 0; p < PA; p++)
            if (k0 + (AK ? lc : (tid + 256 * p) / (BM / 4)) >= kEnd) va[p] = OUTSIDE;
#pragma unroll
        for (int p = 0; p < PB; p++)
            if (k0 + (BKC ? lc : (tid + 256 * p) / (BN / 4)) >= kEnd) vb[p] = OUTSIDE;
    };
    // element-wise variant: any alignment, any extent
    auto fetchEach = [&](bool kfast, const float* base, long long ld, int rows0, int rowsEnd, int tileRows, int p, int k0) -> u32x4 {
        u32x4 v;
        if (kfast) {
            const uint32_t* q = (const uint32_t*)base;   // (base holds lc)
            const int left = kEnd - 1 - (k0 + lc);        // index of the last k inside, from this chunk's first
            v.x = q[k0 + min(0, left)]; v.y = q[k0 + min(1, left)]; v.z = q[k0 + min(2, left)]; v.w = q[k0 + min(3, left)];
            if (left < 0) v.x = 0;
            if (left < 1) v.y = 0;
            if (left < 2) v.z = 0;
            if (left < 3) v.w = 0;
        } else {
            const int e = tid + 256 * p, k = e / (tileRows / 4), back = min(0, kEnd - 1 - (k0 + k));
            const uint32_t* q = (const uint32_t*)(base + (k0 + back) * ld);   // (base holds this thread's k and row)
            const int left = rowsEnd - 1 - (rows0 + 4 * (e % (tileRows / 4)));   // index of the last row inside
            v.x = q[min(0, left)]; v.y = q[min(1, left)]; v.z = q[min(2, left)]; v.w = q[min(3, left)];
            if (back < 0) v.x = v.y = v.z = v.w = 0;
        }
        return v;
    };
    auto fetchA = [&](int p, int k0) {
        if (VEC && AK) ra[p] = __builtin_amdgcn_raw_buffer_load_b128(rsA, va[p], k0 * 4, 0);
        else if (VEC) ra[p] = __builtin_amdgcn_raw_buffer_load_b128(resource(stageA), va[p], 0, 0);
        else ra[p] = fetchEach(AK, ga[p], g.lda, m0, M, BM, p, k0);
    };
    auto fetchB = [&](int p, int k0) {
        if (VEC && BKC) rb[p] = __builtin_amdgcn_raw_buffer_load_b128(rsB, vb[p], k0 * 4, 0);
        else if (VEC) rb[p] = __builtin_amdgcn_raw_buffer_load_b128(resource(stageB), vb[p], 0, 0);
        else rb[p] = fetchEach(BKC, gb[p], g.ldb, n0, N, BN, p, k0);
    };
    auto put = [&](bool kfast, u32x4 v, float* dst, int ldrow, int tileRows, int p) {
        const int e = tid + 256 * p;
        if (kfast) *(u32x4*)(dst + (lr + 32 * p) * LDK + lc) = v;
        else *(u32x4*)(dst + (e / (tileRows / 4)) * ldrow + ((4 * (e % (tileRows / 4))) ^ ((e / tileRows & 1) * 32))) = v;
    };
    const int fr = lane & 31, fg = (lane >> 5) * 4;
    auto fragment = [&](bool kfast, const float* stage, int ldrow, int row, int ks) -> u32x4 {
        if (kfast) return *(const u32x4*)(stage + (row + fr) * LDK + ks * 8 + fg);
        const uint32_t* q = (const uint32_t*)(stage + fg * ldrow + ((row + fr) ^ (fg * 8)) + ks * 8 * ldrow);
        u32x4 v;
        v.x = q[0]; v.y = q[ldrow]; v.z = q[2 * ldrow]; v.w = q[3 * ldrow];
        return v;
    };

    const int nk = (kEnd - kBegin + BK - 1) / BK;
    if (nk == 1) lastStage(kBegin);
#pragma unroll
    for (int p = 0; p < PA; p++) fetchA(p, kBegin);
#pragma unroll
    for (int p = 0; p < PB; p++) fetchB(p, kBegin);
#pragma unroll
    for (int p = 0; p < PA; p++) put(AK, ra[p], As, LDA, BM, p);
#pragma unroll
    for (int p = 0; p < PB; p++) put(BKC, rb[p], Bs, LDB, BN, p);
    {
        const int k1 = kBegin + min(1, nk - 1) * BK;
        if (nk > 1) advance();
        if (nk == 2) lastStage(k1);
#pragma unroll
        for (int p = 0; p < PA; p++) fetchA(p, k1);
#pragma unroll
        for (int p = 0; p < PB; p++) fetchB(p, k1);
    }
    __syncthreads();
    u32x4 a[2][WM], b[2][WN];
    // One stage on LDS buffer kt & 1.  Between the products: in the first half of the k-steps the registers that hold stage
    // kt + 1 go to the other buffer, in the second half stage kt + 2 is fetched into them, and in every k-step but the last
    // the fragments of the next one are read.  Past the end the last stage is fetched again and never used.
    for (int kt = 0; kt < nk; kt++) {
        const int buf = kt & 1;
        const float* pa = As + buf * SA;
        const float* pb = Bs + buf * SB;
        float* wa = As + (buf ^ 1) * SA;
        float* wb = Bs + (buf ^ 1) * SB;
        const int k2 = kBegin + min(kt + 2, nk - 1) * BK;
        advance();
        if (kt + 3 == nk) lastStage(k2);
#pragma unroll
        for (int t = 0; t < WM; t++) a[0][t] = fragment(AK, pa, LDA, wm + t * 32, 0);
#pragma unroll
        for (int t = 0; t < WN; t++) b[0][t] = fragment(BKC, pb, LDB, wn + t * 32, 0);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int cur = ks & 1, nxt = cur ^ 1;
            const int c0 = (PA + PB) * (ks % HALF) / HALF, c1 = (PA + PB) * (ks % HALF + 1) / HALF;
#pragma unroll
            for (int q = 0; q < NMF; q++) {
                const int i = q / WN, j = q % WN;
                // the transposed tile (B as the row operand): a lane owns a row of C
                acc[i][j] = BigTraits<float>::mma(b[cur][j], a[cur][i], acc[i][j]);
                if (ks + 1 < KS) {
#pragma unroll
                    for (int r = q * RF; r < (q + 1) * RF; r++) {
                        if (r < WM) a[nxt][r] = fragment(AK, pa, LDA, wm + r * 32, ks + 1);
                        else if (r < WM + WN) b[nxt][r - WM] = fragment(BKC, pb, LDB, wn + (r - WM) * 32, ks + 1);
                    }
                }
#pragma unroll
                for (int c = c0 + q * SC; c < c0 + (q + 1) * SC; c++) {
                    if (c >= c1) break;
                    if (ks < HALF) {
                        if (c < PA) put(AK, ra[c], wa, LDA, BM, c);
                        else put(BKC, rb[c - PA], wb, LDB, BN, c - PA);
                    } else {
                        if (c < PA) fetchA(c, k2);
                        else fetchB(c - PA, k2);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();
    }
    // Register v of a tile is column 8 (v / 4) + 4 (lane / 32) + v % 4 of row lane % 32.  Each wavefront passes its tile, 32
    // rows at a time, through its own slice of LDS (free after the last barrier; operations of one wavefront complete in
    // order) and the lanes then walk the rows, so that a store instruction covers whole lines.
    constexpr int CW = 32 * WN, LDC = CW + 4, LPR = CW / 4, RPI = 64 / LPR, NIT = (32 + RPI - 1) / RPI;
    float* cs = reinterpret_cast<float*>(smem_raw) + wave * 32 * LDC;
    const int rr = lane / LPR, cc = (lane % LPR) * 4;
    float* C = split ? g.part + (size_t)part * M * N : g.C + (size_t)batch * g.sC;
    const long long ldc = split ? N : g.ldc;
    const float beta = split ? 0.f : g.beta;
    const bool vec = split ? (N & 3) == 0 : g.vecC;
    const int c = n0 + wn + cc;   // a lane keeps its columns while it walks the rows
    float4 bias = make_float4(0.f, 0.f, 0.f, 0.f);
    float* col = nullptr;
    if (!split && c < N) {
        bias = f32_bias4(g.bias, c, N);
        if constexpr (HEADS) col = heads_col<float>(hp.he, c);
    }
#pragma unroll
    for (int i = 0; i < WM; i++) {
#pragma unroll
        for (int j = 0; j < WN; j++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                *(float4*)(cs + fr * LDC + j * 32 + 8 * q + fg) =
                    make_float4(g.alpha * acc[i][j][4 * q], g.alpha * acc[i][j][4 * q + 1], g.alpha * acc[i][j][4 * q + 2], g.alpha * acc[i][j][4 * q + 3]);
#pragma unroll 4
        for (int it = 0; it < NIT; it++) {
            const int row = it * RPI + rr, r = m0 + wm + i * 32 + row;
            if (rr >= RPI || row >= 32 || r >= M || c >= N) continue;
            const float4 t = *(const float4*)(cs + row * LDC + cc);
            float v[4] = {t.x + bias.x, t.y + bias.y, t.z + bias.z, t.w + bias.w};
            if constexpr (HEADS) {
                if (!split) {
                    heads_store4(hp.he, r, c, N, vec, col, v);
                    continue;
                }
            }
            float* cp = C + (size_t)r * ldc + c;
            if (vec) {
                if (beta != 0.f) {
                    const float4 o = *(const float4*)cp;
                    v[0] += beta * o.x; v[1] += beta * o.y; v[2] += beta * o.z; v[3] += beta * o.w;
                }
                *(float4*)cp = make_float4(v[0], v[1], v[2], v[3]);
            } else {
#pragma unroll
                for (int q = 0; q < 4; q++)
                    if (c + q < N) cp[q] = v[q] + (beta != 0.f ? beta * cp[q] : 0.f);
            }
        }
    }
}

// C = sum over the S partial products, in their order (alpha is in them already), + beta C; or through the heads epilogue
template <bool HEADS>
__global__ __launch_bounds__(256) void gemm_f32_sum_kernel(const float* __restrict__ part, int S, int M, int N, long long ldc, float beta, bool vecC,
                                                           float* __restrict__ C, const float* __restrict__ bias, HeadsArg<HEADS> hp)
{
    const int quads = (N + 3) / 4;
    const size_t mn = (size_t)M * N;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < (size_t)M * quads; e += (size_t)blockDim.x * gridDim.x) {
        const int r = (int)(e / quads), c = (int)(e % quads) * 4;
        const float* p = part + (size_t)r * N + c;
        float v[4] = {0.f, 0.f, 0.f, 0.f};
        if ((N & 3) == 0) {
            for (int z = 0; z < S; z++) {
                const float4 t = *(const float4*)(p + z * mn);
                v[0] += t.x; v[1] += t.y; v[2] += t.z; v[3] += t.w;
            }
        } else {
            for (int z = 0; z < S; z++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    if (c + q < N) v[q] += p[z * mn + q];
        }
        const float4 b = f32_bias4(bias, c, N);
        v[0] += b.x; v[1] += b.y; v[2] += b.z; v[3] += b.w;
        if constexpr (HEADS) {
            heads_store4(hp.he, r, c, N, vecC, heads_col<float>(hp.he, c), v);
            continue;
        }
        float* cp = C + (size_t)r * ldc + c;
        if (vecC) {
            if (beta != 0.f) {
                const float4 o = *(const float4*)cp;
                v[0] += beta * o.x; v[1] += beta * o.y; v[2] += beta * o.z; v[3] += beta * o.w;
            }
            *(float4*)cp = make_float4(v[0], v[1], v[2], v[3]);
        } else {
            for (int q = 0; q < 4; q++)
                if (c + q < N) cp[q] = v[q] + (beta != 0.f ? beta * cp[q] : 0.f);
        }
    }
}

// ---------------------------------------------------------------------------
// How a product is cut: the tile and the number of parts of the contraction with the smallest estimated time.
struct GemmF32Plan { int wm, wn, splits, kChunk; };

static GemmF32Plan gemm_f32_plan(int m, int n, int k, int batch, bool causal)
{
    // Cycles of a tile: its products at 256 flops per cycle and CU over the efficiency of a CU's two or more workgroups, and
    // its first fetches and its stores; a workgroup alone on its CU shows every stage's latency.  Fitted to tiles of 768 and
    // 2304 k: 128 x 192 (one workgroup per CU: nothing covers its ends) 176k / 500k cycles, 128 x 128 111k / 332k, 64 x 128
    // 59k / 169k, 64 x 64 31k / 88k.  A split contraction pays for a second
    // launch and for the partial products' way through memory.
    static const struct { int wm, wn; double eff, ends, alone; } shapes[] = {{2, 3, 0.909, 14000, 1.10}, {2, 2, 0.89, 600, 1.30}, {1, 2, 0.895, 4000, 1.45}, {1, 1, 0.863, 2200, 1.60}};
    GemmF32Plan best = {1, 1, 1, k};
    double bestT = 1e30;
    for (const auto& sh : shapes) {
        const int bm = 64 * sh.wm, bn = 64 * sh.wn;
        const long long tiles = (long long)((m + bm - 1) / bm) * ((n + bn - 1) / bn) * batch;
        for (int S = 1; S <= 32; S++) {
            if (S > 1 && (batch > 1 || causal || k / S < 128)) break;
            const int chunk = ((k + S - 1) / S + 31) / 32 * 32;
            if ((k + chunk - 1) / chunk != S) continue;
            const double body = 2.0 * bm * bn * ((chunk + 31) / 32 * 32) / 256.0;
            const long long perCu = ((tiles * S + 7) / 8 + 31) / 32;
            const double cycles = perCu == 1 ? body * sh.alone + sh.ends : perCu * (body / sh.eff + sh.ends);
            double t = cycles / 2.4e9;
            if (S > 1) t += 4.5e-6 + (double)(S + 1) * m * n * 4.0 / 4.0e12;
            if (t < bestT) { bestT = t; best = {sh.wm, sh.wn, S, S > 1 ? chunk : k}; }
        }
    }
    return best;
}

size_t gemm_f32_workspace_bytes(int m, int n, int k, int batch, bool causal)
{
    if (m <= 0 || n <= 0 || k <= 0) return 0;
    const GemmF32Plan p = gemm_f32_plan(m, n, k, batch, causal);
    return p.splits > 1 ? (size_t)p.splits * m * n * sizeof(float) : 0;
}

template <int WM, int WN, int OCC, bool AK, bool BKC, bool VEC, bool HEADS>
static hipError_t launch_f32(hipStream_t s, const GemmF32Args& a, int splits, int batch, const HeadsEpilogue* he)
{
    constexpr int BM = 64 * WM, BN = 64 * WN;
    constexpr int SA = AK ? BM * 36 : 32 * BM, SB = BKC ? BN * 36 : 32 * BN;
    constexpr int lds = 4 * ((2 * (SA + SB)) > 4 * 32 * (32 * WN + 4) ? 2 * (SA + SB) : 4 * 32 * (32 * WN + 4));
    static const hipError_t attr = hipFuncSetAttribute((const void*)gemm_f32_kernel<WM, WN, OCC, AK, BKC, VEC, HEADS>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (attr != hipSuccess) return attr;
    GemmF32Args g = a;
    g.tilesM = (g.M + BM - 1) / BM;
    g.tilesN = (g.N + BN - 1) / BN;
    g.parts = splits > 1 ? splits : batch;
    const long long total = (long long)g.tilesM * g.tilesN * g.parts;
    if (total > (1ll << 27)) return hipErrorInvalidValue;
    const int per = (int)((total + 7) / 8);
    hipLaunchKernelGGL((gemm_f32_kernel<WM, WN, OCC, AK, BKC, VEC, HEADS>), dim3(per * 8), 256, lds, s, g, heads_arg<HEADS>(he));
    return hipGetLastError();
}

template <bool AK, bool BKC, bool VEC, bool HEADS>
static hipError_t launch_f32_tile(hipStream_t s, const GemmF32Args& a, const GemmF32Plan& p, int batch, const HeadsEpilogue* he = nullptr)
{
    if (p.wn == 3) return launch_f32<2, 3, 1, AK, BKC, VEC, HEADS>(s, a, p.splits, batch, he);
    if (p.wm == 2) return launch_f32<2, 2, 2, AK, BKC, VEC, HEADS>(s, a, p.splits, batch, he);
    if (p.wn == 2) return launch_f32<1, 2, 2, AK, BKC, VEC, HEADS>(s, a, p.splits, batch, he);
    return launch_f32<1, 1, 3, AK, BKC, VEC, HEADS>(s, a, p.splits, batch, he);
}

hipError_t gemm_f32(hipStream_t s, const GemmF32& q, void* ws, size_t wsBytes)
{
    if (q.m <= 0 || q.n <= 0 || q.batch <= 0) return hipSuccess;
    if (q.k <= 0 || (q.causal && ((q.causal >= CAUSAL_B_LOWER ? q.n : q.m) != q.k || !q.flag)) || (q.heads && (q.alpha != 1.f || q.beta != 0.f || q.batch != 1 || !q.aK || !q.bK)))
        return hipErrorInvalidValue;
    GemmF32Plan p = gemm_f32_plan(q.m, q.n, q.k, q.batch, q.causal != 0);
    if (p.splits > 1 && (!ws || wsBytes < (size_t)p.splits * q.m * q.n * sizeof(float) || ((uintptr_t)ws & 15))) { p.splits = 1; p.kChunk = q.k; }
    GemmF32Args a = {};
    a.M = q.m; a.N = q.n; a.K = q.k;
    a.A = q.A; a.B = q.B; a.C = q.C;
    a.lda = q.lda; a.ldb = q.ldb; a.ldc = q.ldc; a.sA = q.sA; a.sB = q.sB; a.sC = q.sC;
    a.alpha = q.alpha; a.beta = q.beta;
    a.kChunk = p.kChunk;
    a.causal = q.causal; a.flag = q.flag; a.epoch = q.epoch;
    a.part = (float*)ws;
    a.bias = q.heads ? (const float*)q.heads->bias : q.bias;
    if (q.heads) {
        const HeadsEpilogue& he = *q.heads;
        a.vecC = q.n % 4 == 0 && he.hs % 4 == 0 && (((uintptr_t)he.dst[0] | (uintptr_t)he.dst[1] | (uintptr_t)he.dst[2]) & 15) == 0;
    } else {
        a.vecC = q.n % 4 == 0 && q.ldc % 4 == 0 && (q.batch == 1 || q.sC % 4 == 0) && ((uintptr_t)q.C & 15) == 0;
    }
    // 31-bit byte offsets within a tile's rows of k (128 at most), or within the k rows of a stage
    auto near = [&](bool kFast, int rows, long long ld) { return (kFast ? (std::min(rows, 128) + 1) * ld : std::min(q.k, 32) * ld + 256) < (1ll << 29); };
    const bool vec = (((uintptr_t)q.A | (uintptr_t)q.B) & 15) == 0 && q.lda % 4 == 0 && q.ldb % 4 == 0 && (q.batch == 1 || (q.sA % 4 == 0 && q.sB % 4 == 0)) &&
                     (q.aK ? q.k % 4 == 0 : q.m % 4 == 0) && (q.bK ? q.k % 4 == 0 : q.n % 4 == 0) &&
                     near(q.aK, q.m, q.lda) && near(q.bK, q.n, q.ldb);
    hipError_t e;
    if (q.heads) e = vec ? launch_f32_tile<true, true, true, true>(s, a, p, 1, q.heads) : launch_f32_tile<true, true, false, true>(s, a, p, 1, q.heads);
#define LAYOUT(AKV, BKV) (vec ? launch_f32_tile<AKV, BKV, true, false>(s, a, p, q.batch) : launch_f32_tile<AKV, BKV, false, false>(s, a, p, q.batch))
    else if (q.aK) e = q.bK ? LAYOUT(true, true) : LAYOUT(true, false);
    else e = q.bK ? LAYOUT(false, true) : LAYOUT(false, false);
#undef LAYOUT
    if (e != hipSuccess || p.splits == 1) return e;
    const size_t quads = (size_t)q.m * ((q.n + 3) / 4);
    const int grid = (int)std::min<size_t>((quads + 255) / 256, 4096);
    if (q.heads) hipLaunchKernelGGL(gemm_f32_sum_kernel<true>, grid, 256, 0, s, (const float*)ws, p.splits, q.m, q.n, q.ldc, q.beta, a.vecC, q.C, a.bias, heads_arg<true>(q.heads));
    else hipLaunchKernelGGL(gemm_f32_sum_kernel<false>, grid, 256, 0, s, (const float*)ws, p.splits, q.m, q.n, q.ldc, q.beta, a.vecC, q.C, a.bias, HeadsArg<false>());
    return hipGetLastError();
}

}  // namespace mch
