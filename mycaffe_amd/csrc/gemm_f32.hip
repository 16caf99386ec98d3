// fp32 GEMM, any operand layout, gfx950: on the bf16 matrix cores with every value as three bf16 numbers (gemm_f32_split_kernel,
// below), and on the fp32 matrix cores (v_mfma_f32_32x32x2_f32) where that is not taken: gemm_f32_small_kernel for products that do not
// fill the chip, gemm_f32_kernel.
//
// gemm_f32_kernel serves the inner products (A B^T), their gradients (A B and A^T B) and the batched products of the explicit
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
#include "xcd_runs.h"

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
    int kTail;                // of the contraction's end, what the split kernel does not fetch in chunks of four
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

// Which tile of which part of the contraction, or of which matrix of the batch, a workgroup has, and its range of k.
struct F32Item { int part, batch, m0, n0, kBegin, kEnd; };
// Work items are the tiles of every part of the contraction, or of every matrix of the batch; each XCD (workgroup index mod 8)
// takes a contiguous run of them, so all dies get the same share whatever the tile count of one part.
__device__ __forceinline__ int xcd_item(int total) { return (int)(blockIdx.x % 8) * ((total + 7) / 8) + (int)(blockIdx.x / 8); }
template <int BM, int BN>
__device__ __forceinline__ void f32_item(const GemmF32Args& g, int item, F32Item& o)
{
    const int tiles = g.tilesM * g.tilesN;
    o.part = item / tiles;
    const int tile = item - o.part * tiles;
    const bool split = g.kChunk < g.K;
    o.batch = split ? 0 : o.part;
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
        if (((o.batch * tiles) >> 5) & 1) {
            if (g.causal >= CAUSAL_B_LOWER) tc = g.tilesN - 1 - tc;
            else tr = g.tilesM - 1 - tr;
        }
        causal = *g.flag != g.epoch;
    }
    o.m0 = tr * BM; o.n0 = tc * BN;
    o.kBegin = split ? o.part * g.kChunk : 0;
    o.kEnd = min(g.K, o.kBegin + g.kChunk);
    if (causal) {
        if (g.causal == CAUSAL_A_LOWER) o.kEnd = min(o.kEnd, o.m0 + BM);
        else if (g.causal == CAUSAL_A_UPPER) o.kBegin = o.m0;
        else if (g.causal == CAUSAL_B_LOWER) o.kBegin = o.n0;
        else o.kEnd = min(o.kEnd, o.n0 + BN);
    }
}

// The accumulators of a wavefront (the transposed tiles: register v is column 8 (v / 4) + 4 (lane / 32) + v % 4 of row lane % 32) to
// C, to the part's partial product or through the heads epilogue.  Each wavefront passes its tile, 32 rows at a time, through its
// own slice of LDS (free after the last barrier; operations of one wavefront complete in order) and the lanes then walk the rows,
// so that a store instruction covers whole lines.  (m, n): the wavefront's first row and column.
template <int WM, int WN, bool HEADS>
__device__ __forceinline__ void f32_store(const GemmF32Args& g, const HeadsArg<HEADS>& hp, floatx16 (&acc)[WM][WN], float* slice, int lane, int m, int n,
                                          int part, int batch)
{
    constexpr int CW = 32 * WN, LDC = CW + 4, LPR = CW / 4, RPI = 64 / LPR, NIT = (32 + RPI - 1) / RPI;
    const int M = g.M, N = g.N;
    const bool split = g.kChunk < g.K;
    const int fr = lane & 31, fg = (lane >> 5) * 4;
    const int rr = lane / LPR, cc = (lane % LPR) * 4;
    float* C = split ? g.part + (size_t)part * M * N : g.C + (size_t)batch * g.sC;
    const long long ldc = split ? N : g.ldc;
    const float beta = split ? 0.f : g.beta;
    const bool vec = split ? (N & 3) == 0 : g.vecC;
    const int c = n + cc;   // a lane keeps its columns while it walks the rows
    float4 bias = make_float4(0.f, 0.f, 0.f, 0.f);
    float* col = nullptr;
    if (!split && c < N) {
        bias = f32_bias4(g.bias, c, N);
        if constexpr (HEADS) col = heads_col<float>(hp.he, c);
    }
    // What the result is added to comes for eight rows at once; in the loop below each row would wait for memory (A^T B, added: 8000 x 512 x
    // 1000 65 us, 63 so, 32000 x 768 x 1000 255, 244, 5000 x 1000 x 1000 89, 82; A B: 8192 x 3072 x 768 214, 199, 1000 x 4096 x 512 41, 37).
    // Tiles with eight sums of 16 a lane have no registers for that (46 of them in memory, 9 without: 4096 x 4096 x 1024, A^T B, 172 us, 174
    // with it), and what goes head by head is not added.
    const bool add = !HEADS && WM * WN < 8 && vec && beta != 0.f;
    constexpr int AHEAD = NIT < 8 ? NIT : 8;
#pragma unroll
    for (int i = 0; i < WM; i++) {
#pragma unroll
        for (int j = 0; j < WN; j++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                *(float4*)(slice + fr * LDC + j * 32 + 8 * q + fg) =
                    make_float4(g.alpha * acc[i][j][4 * q], g.alpha * acc[i][j][4 * q + 1], g.alpha * acc[i][j][4 * q + 2], g.alpha * acc[i][j][4 * q + 3]);
        if (add) {
#pragma unroll 1
            for (int first = 0; first < NIT; first += AHEAD) {
                float4 old[AHEAD];
#pragma unroll
                for (int k = 0; k < AHEAD; k++)
                    old[k] = *(const float4*)(C + (size_t)min(m + i * 32 + (first + k) * RPI + rr, M - 1) * ldc + min(c, N - 4));
#pragma unroll
                for (int k = 0; k < AHEAD; k++) {
                    const int row = (first + k) * RPI + rr, r = m + i * 32 + row;
                    if (rr >= RPI || row >= 32 || r >= M || c >= N) continue;
                    const float4 t = *(const float4*)(slice + row * LDC + cc);
                    *(float4*)(C + (size_t)r * ldc + c) = make_float4(t.x + bias.x + beta * old[k].x, t.y + bias.y + beta * old[k].y, t.z + bias.z + beta * old[k].z, t.w + bias.w + beta * old[k].w);
                }
            }
            continue;
        }
#pragma unroll 4
        for (int it = 0; it < NIT; it++) {
            const int row = it * RPI + rr, r = m + i * 32 + row;
            if (rr >= RPI || row >= 32 || r >= M || c >= N) continue;
            const float4 t = *(const float4*)(slice + row * LDC + cc);
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
    const int total = g.tilesM * g.tilesN * g.parts, item = xcd_item(total);
    if (item >= total) return;
    F32Item it;
    f32_item<BM, BN>(g, item, it);
    const int M = g.M, N = g.N, m0 = it.m0, n0 = it.n0, kBegin = it.kBegin, kEnd = it.kEnd, part = it.part, batch = it.batch;
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
    f32_store<WM, WN, HEADS>(g, hp, acc, reinterpret_cast<float*>(smem_raw) + wave * 32 * (32 * WN + 4), lane, m0 + wm, n0 + wn, part, batch);
}

// ---------------------------------------------------------------------------
// The same products on the bf16 matrix cores, sixteen times the rate of the fp32 ones: every operand value is the sum of three
// bf16 numbers, x = h + m + l exactly (24 bits of significand are three times eight; each part is the bf16 nearest to what the
// parts before it leave), and of the nine products of parts the six down to 2^-18 of the first are added up in fp32:
// hh + (hm + mh + mm) + (hl + lh).  What is left out is 2^-25 of a product at most.  An MFMA adds sixteen products at a time
// where the fp32 one adds two, so the sums are rounded less often, and the error against 64 bits is below that of the fp32
// matrix cores from 64 k on (N(0, 1), 2-norm of the error over that of the result: 1.35e-7 against 1.45e-7 at 64 k, 4.3e-7 against
// 5.0e-7 at 768, 7.0e-7 against 8.0e-7 at 2048; the other way round at 16: 8.2e-8 against 7.4e-8); shorter contractions stay
// there (gemm_f32_choose).
//
// Exact results where parts do not hold a value.  An infinity or a value above the largest bf16 number leaves a NaN or an infinity
// among the parts and so in the sums.  Below 2^-109 the last part, or all of them, lose bits (bf16 ends at 2^-133): up to 2^-134 of
// the value, and of the sum that times the other factor, which may be any number.  It shows in what the last part is made of, eight
// bits of an fp32 number that end above its low half wherever bf16 holds them: the low halves of all of them are or-ed together
// (one v_or3 for two values).  A wavefront does its tile again on the fp32 matrix cores, straight from memory, if its sums hold a NaN, an
// infinity or anything nonzero below 2^-90, or if a value of the workgroup's operands lost bits and either some value is 2^16 or more (for which
// they are then read once more) or a sum, zeros among them, is so small that k products with up to 2^16 times those bits may be 2^-25 of
// it.  So an ordinary tile beside a stray tiny value (GELU of -10) is not made over: 8192 x 3072 x 768 with one in every tile takes 280 us, 218
// without, 570 with a row of zeros beside one.  (Looking for lost bits takes 1 - 2 % of an ordinary product under lasting load and 4 % in the
// first launches after a pause, whose clock is not at its limit yet; to keep the largest value along, and read nothing again, took 2 - 3 %.)
//
// What bounds it is power: at 8192 x 3072 x 768 operands of zeros take 136 us in 128 x 192 tiles, random ones 197 (same instructions), so what
// helps is fewer instructions and bytes per product.  Values are split once, on their way from registers to LDS (splitting whole
// operands in a pass of their own costs more than the repeats), the larger tiles split a value less often, and one LDS read of a
// fragment serves up to three products times WM or WN tiles.
//
// Measured, before (fp32 matrix cores) and now, us: 8192 x 3072 x 768 279 -> 188, 8192 x 768 x 3072 274 -> 190, 768 x 3072 x 8192
// (A^T B) 303 -> 191, 1000 x 32000 x 768 370 -> 231, 4096 x 4096 x 4096 935 -> 564 (244 TFLOP/s), 2800 x 768 x 768 40 -> 31.
//
//   * Global loads of a stage (16 KS k) are one stage ahead in registers; between the products of a stage they are split and
//     written to the other LDS buffer, and the stage after that is requested.
//   * LDS holds three planes (h, m, l) per operand.  k at unit stride: eight k of a row are 16 bytes, rows next to each other,
//     groups of eight k padded apart so that what a wavefront writes falls on different banks.  Row index at unit stride: [k][row],
//     the layout and the transposing reads of the 16-bit kernel (gemm_bf16.hip).
//   * One barrier a stage, placed before the last third of its products: by then every fragment of the stage has been read, and
//     the first fragments of the next stage arrive behind the remaining products.
__device__ __forceinline__ uint2 split_part(float (&v)[4], bool last)
{
    uint2 p;
    p.x = pack2_bf16(v[0], v[1]);
    p.y = pack2_bf16(v[2], v[3]);
    if (!last) {
        v[0] -= __uint_as_float(p.x << 16); v[1] -= __uint_as_float(p.x & 0xffff0000u);
        v[2] -= __uint_as_float(p.y << 16); v[3] -= __uint_as_float(p.y & 0xffff0000u);
    }
    return p;
}

// written as an instruction: the compiler would gather those of a stage at its end, and keep the values until then (14 registers; 256 x 256
// tiles spill)
__device__ __forceinline__ void or3(uint32_t& m, uint32_t a, uint32_t b) { asm("v_or3_b32 %0, %0, %1, %2" : "+v"(m) : "v"(a), "v"(b)); }

// what the workgroup's wavefronts leave in LDS for each other: whether a value lost bits, and whether one is LARGE or more
struct SplitFlags { uint32_t lost, large; };
constexpr float SPLIT_LARGE = 65536.f;

// whether this thread finds a value of SPLIT_LARGE or more in its share of an operand's R rows (`rows` of them there) from kBegin to kEnd
template <int R, int NT, bool KFAST> __device__ __forceinline__ bool split_large(const float* base, long long ld, int rows, int kBegin, int kEnd, int tid)
{
    constexpr int U = 16, W = KFAST ? 64 : 32;   // loads under way; lanes along the memory
    const int fast = tid % W, fastEnd = KFAST ? kEnd : min(R, rows), slowEnd = KFAST ? min(R, rows) : kEnd;
    bool found = false;
    for (int f = (KFAST ? kBegin : 0) + fast; f < fastEnd; f += W)
        for (int s0 = (KFAST ? 0 : kBegin) + tid / W; s0 < slowEnd; s0 += U * (NT / W)) {
            float x[U];
#pragma unroll
            for (int u = 0; u < U; u++) x[u] = base[(size_t)min(s0 + u * (NT / W), slowEnd - 1) * ld + f];
#pragma unroll
            for (int u = 0; u < U; u++) found |= fabsf(x[u]) >= SPLIT_LARGE;
        }
    return found;
}

// whether the parts may have lost something of these sums of k products (the same for the whole wavefront)
template <int WM, int WN> __device__ __forceinline__ bool split_lost(const floatx16 (&acc)[WM][WN], const SplitFlags& flags, int k)
{
    constexpr uint32_t TINY = (127u - 90u) << 24;   // 2^-90 without its sign
    if (flags.lost) {
        if (flags.large) return true;
        const float limit = (float)k * 0x1p-92f;   // 2 k values' 2^-134 times SPLIT_LARGE, 2^25 times that
        float least = limit;
#pragma unroll
        for (int i = 0; i < WM; i++)
#pragma unroll
            for (int j = 0; j < WN; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) least = fminf(least, fabsf(acc[i][j][v]));
        if (__any(least < limit)) return true;
    }
    uint32_t low = 0xffffffffu;
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < WM; i++)
#pragma unroll
        for (int j = 0; j < WN; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                low = min(low, (__float_as_uint(acc[i][j][v]) << 1) - 1u);   // zeros wrap to the top
                sum += fabsf(acc[i][j][v]);
            }
    return __any(low < TINY - 1u || !(sum < __builtin_inff()));
}

// a wavefront's sums by the fp32 matrix cores, operands read from memory value by value; ADD: to what acc holds
template <int WM, int WN, bool AK, bool BKC, bool ADD>
__device__ __forceinline__ void f32_sums(const GemmF32Args& g, const float* A, const float* B, int m, int n, int kBegin, int kEnd, int lane, floatx16 (&acc)[WM][WN])
{
    const int fr = lane & 31, half = lane >> 5;
    const float* a[WM];
    const float* b[WN];
#pragma unroll
    for (int t = 0; t < WM; t++) a[t] = A + (size_t)min(m + t * 32 + fr, g.M - 1) * (AK ? g.lda : 1);
#pragma unroll
    for (int t = 0; t < WN; t++) b[t] = B + (size_t)min(n + t * 32 + fr, g.N - 1) * (BKC ? g.ldb : 1);
#pragma unroll
    for (int i = 0; i < WM; i++)
#pragma unroll
        for (int j = 0; j < WN; j++)
#pragma unroll
            for (int v = 0; v < 16; v++)
                if (!ADD) acc[i][j][v] = 0.f;
    for (int k0 = kBegin; k0 < kEnd; k0 += 8) {
        float x[4][WM], y[4][WN];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int k = min(k0 + 2 * u + half, kEnd - 1);
#pragma unroll
            for (int t = 0; t < WM; t++) x[u][t] = a[t][(size_t)k * (AK ? 1 : g.lda)];
#pragma unroll
            for (int t = 0; t < WN; t++) y[u][t] = b[t][(size_t)k * (BKC ? 1 : g.ldb)];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const bool in = k0 + 2 * u + half < kEnd;
#pragma unroll
            for (int i = 0; i < WM; i++)
#pragma unroll
                for (int j = 0; j < WN; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(in ? y[u][j] : 0.f, in ? x[u][i] : 0.f, acc[i][j], 0, 0, 0);
        }
    }
}

// bytes of one plane of R rows by 16 KS k
template <int R, int KS, bool KFAST> constexpr int split_plane() { return KFAST ? 2 * KS * (R * 16 + 128 / KS) : 16 * KS * R * 2; }

// floats that the split kernel's stages, and then its results, take in LDS: behind them the row sums
template <int WVM, int WVN, int WM, int WN, int KS, bool AK, bool BKC> constexpr int split_lds()
{
    constexpr int stages = 2 * 3 * (split_plane<32 * WVM * WM, KS, AK>() + split_plane<32 * WVN * WN, KS, BKC>()), store = 4 * WVM * WVN * 32 * (32 * WN + 4);
    return (stages > store ? stages : store) / 4;
}
// where in bytes the flags lie, behind the row sums
template <int WVM, int WVN, int WM, int WN, int KS, bool AK, bool BKC, bool SUMS> constexpr int split_flags_at()
{
    return 4 * split_lds<WVM, WVN, WM, WN, KS, AK, BKC>() + (SUMS ? 64 * WVM * WVN * 16 : 0);
}
// sums of op(A)'s rows over some of the k, [part][tile column][M], behind the partial products
__device__ __forceinline__ float* f32_row_part(const GemmF32Args& g) { return g.part + (g.kChunk < g.K ? (size_t)g.parts * g.M * g.N : 0); }

// SUMS: the tiles of a row of tiles also add up the rows of op(A), each the stages that are its turn, from the chunks it fetches: the
// bias gradient beside a weight gradient (8192 rows, 768 to 2304: 169 us one after the other, 157 together).
template <int WVM, int WVN, int WM, int WN, int KS, int OCC, bool AK, bool BKC, bool VEC, bool HEADS, bool SUMS>
__global__ __launch_bounds__(64 * WVM * WVN, OCC) void gemm_f32_split_kernel(GemmF32Args g, HeadsArg<HEADS> hp)
{
    constexpr int NT = 64 * WVM * WVN, BK = 16 * KS, BM = 32 * WVM * WM, BN = 32 * WVN * WN;
    constexpr int PA = (BM * BK / 4 + NT - 1) / NT, PB = (BN * BK / 4 + NT - 1) / NT, P = PA + PB;   // chunks of four values per thread and stage
    constexpr int KGA = BM * 16 + 128 / KS, KGB = BN * 16 + 128 / KS;                                  // bytes between groups of eight k
    constexpr int PLA = split_plane<BM, KS, AK>(), PLB = split_plane<BN, KS, BKC>(), STAGE = 3 * (PLA + PLB);
    constexpr int NMF = WM * WN;
    static_assert(PA * NT == BM * BK / 4 && (KS == 1 || KS % 2 == 0), "whole chunks of A; fragments change registers from k-step to k-step");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int total = g.tilesM * g.tilesN * g.parts, item = xcd_item(total);
    if (item >= total) return;
    F32Item it;
    f32_item<BM, BN>(g, item, it);
    const int M = g.M, N = g.N, m0 = it.m0, n0 = it.n0, kBegin = it.kBegin;
    const int kEnd = !VEC && it.kEnd == g.K ? max(kBegin, it.kEnd - g.kTail) : it.kEnd;   // of what is fetched in chunks
    const float* __restrict__ A = g.A + (size_t)it.batch * g.sA;
    const float* __restrict__ B = g.B + (size_t)it.batch * g.sB;
    const int wm = (wave / WVN) * (32 * WM), wn = (wave % WVN) * (32 * WN);

    floatx16 acc[WM][WN];
#pragma unroll
    for (int i = 0; i < WM; i++)
#pragma unroll
        for (int j = 0; j < WN; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;

    // Chunk e of a stage, k at unit stride: row e / (BK / 4), k = 4 (e % (BK / 4)); row index at unit stride: k = e / (rows / 4),
    // rows 4 (e % (rows / 4)) .. + 3.  Where B's chunks do not divide by the threads, the last threads repeat earlier chunks.
    // Byte offsets from a buffer resource that begins at the tile, and where the row index is at unit stride at the stage, so that
    // operands of any size are reached with 32 bits; rows past the edge are clamped (valid memory) and never stored.  Not VEC, operands
    // that are not whole aligned chunks: a fetch of four values needs the alignment of one, a chunk across the last row goes on in the next
    // k, and the last k, where there is none, and what is left of four k are the tail (996 rows, 768 to 27230, forward, backward and
    // softmax: 1850 us on the fp32 matrix cores, value by value; 836).
    constexpr uint32_t OUTSIDE = 0x80000000u;
    constexpr int CK = BK / 4;
    const float* baseA = A + (AK ? (size_t)m0 * g.lda : (size_t)m0);
    const float* baseB = B + (BKC ? (size_t)n0 * g.ldb : (size_t)n0);
    uint32_t va[PA], vb[PB], wa[PA], wb[PB];   // where chunks come from, and where their h goes in a stage
    auto chunkB = [&](int p) { return (tid + NT * p) % (BN * CK); };
#pragma unroll
    for (int p = 0; p < PA; p++) {
        const int e = tid + NT * p;
        if (AK) {
            va[p] = 4 * ((uint32_t)min(e / CK, M - 1 - m0) * (uint32_t)g.lda + 4 * (e % CK));
            wa[p] = (e % CK / 2) * KGA + (e / CK) * 16 + (e & 1) * 8;
        } else {
            const int k = e / (BM / 4), row = 4 * (e % (BM / 4));
            va[p] = 4 * ((uint32_t)k * (uint32_t)g.lda + min(row, VEC ? M - 4 - m0 : (M - 1 - m0) & ~3));
            wa[p] = (k * BM + (row ^ (block_swizzle<BM * 2>(k) * 8))) * 2;
        }
    }
#pragma unroll
    for (int p = 0; p < PB; p++) {
        const int e = chunkB(p);
        if (BKC) {
            vb[p] = 4 * ((uint32_t)min(e / CK, N - 1 - n0) * (uint32_t)g.ldb + 4 * (e % CK));
            wb[p] = 3 * PLA + (e % CK / 2) * KGB + (e / CK) * 16 + (e & 1) * 8;
        } else {
            const int k = e / (BN / 4), row = 4 * (e % (BN / 4));
            vb[p] = 4 * ((uint32_t)k * (uint32_t)g.ldb + min(row, VEC ? N - 4 - n0 : (N - 1 - n0) & ~3));
            wb[p] = 3 * PLA + (k * BN + (row ^ (block_swizzle<BN * 2>(k) * 8))) * 2;
        }
    }
    auto resource = [](const void* base) { return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)(OUTSIDE - 16), 0x00020000); };
    const __amdgpu_buffer_rsrc_t rsA = resource(baseA), rsB = resource(baseB);
    // as in gemm_f32_kernel: the stage that is fetched next and the way to the one after it, where resources begin at stages
    const char *stageA = (const char*)(baseA + (size_t)kBegin * g.lda), *stageB = (const char*)(baseB + (size_t)kBegin * g.ldb);
    long long stepA = (long long)(BK * sizeof(float)) * g.lda, stepB = (long long)(BK * sizeof(float)) * g.ldb;
    auto advance = [&]() {
        if (!AK) stageA += stepA;
        if (!BKC) stageB += stepB;
    };
    // before the last stage is fetched, once: the chunks past the end of the contraction
    auto lastStage = [&](int k0) {
        asm volatile("" ::: "memory");   // a branch, not a select in every stage
        stepA = stepB = 0;
#pragma unroll
        for (int p = 0; p < PA; p++) {
            const int e = tid + NT * p;
            if (k0 + (AK ? 4 * (e % CK) : e / (BM / 4)) >= kEnd) va[p] = OUTSIDE;
        }
#pragma unroll
        for (int p = 0; p < PB; p++) {
            const int e = chunkB(p);
            if (k0 + (BKC ? 4 * (e % CK) : e / (BN / 4)) >= kEnd) vb[p] = OUTSIDE;
        }
    };
    const int nk = VEC ? (kEnd - kBegin + BK - 1) / BK : max(1, (kEnd - kBegin + BK - 1) / BK);
    int fetched = 0, kFetch = kBegin;   // the stage that is fetched and its first k
    auto nextStage = [&]() {
        if (fetched + 1 < nk) {         // past the end the last stage is fetched again, its products never made
            kFetch += BK;
            fetched++;
        }
        advance();
        if (fetched + 1 == nk) lastStage(kFetch);
    };
    u32x4 raw[P];
    auto fetch = [&](int c) {
        if (c < PA) {
            if (AK) raw[c] = __builtin_amdgcn_raw_buffer_load_b128(rsA, va[c], kFetch * 4, 0);
            else raw[c] = __builtin_amdgcn_raw_buffer_load_b128(resource(stageA), va[c], 0, 0);
        } else {
            if (BKC) raw[c] = __builtin_amdgcn_raw_buffer_load_b128(rsB, vb[c - PA], kFetch * 4, 0);
            else raw[c] = __builtin_amdgcn_raw_buffer_load_b128(resource(stageB), vb[c - PA], 0, 0);
        }
    };
    // SUMS: a thread's chunks of A are of the same four rows; without branches, between reads that are under way
    static_assert(!SUMS || (!AK && NT % (BM / 4) == 0), "");
    [[maybe_unused]] float sums[4] = {0.f, 0.f, 0.f, 0.f};
    [[maybe_unused]] int turn = n0 / BN, putting = 0;   // the stage that is put, and stages until this tile's next
    [[maybe_unused]] uint32_t mine = turn == 0 ? 0xffffffffu : 0u;
    uint32_t rest = 0;      // of all values, or-ed: what the last part is made of
    SplitFlags* flags = reinterpret_cast<SplitFlags*>(smem_raw + split_flags_at<WVM, WVN, WM, WN, KS, AK, BKC, SUMS>());
    if (tid == 0) *flags = SplitFlags{0, 0};
    // part s of chunk c to its plane of a stage
    auto put = [&](int c, int s, unsigned char* stage) {
        if constexpr (SUMS) {
            if (s == 0 && c < PA) {
                sums[0] += __uint_as_float(raw[c].x & mine); sums[1] += __uint_as_float(raw[c].y & mine);
                sums[2] += __uint_as_float(raw[c].z & mine); sums[3] += __uint_as_float(raw[c].w & mine);
            }
        }
        float v[4] = {__uint_as_float(raw[c].x), __uint_as_float(raw[c].y), __uint_as_float(raw[c].z), __uint_as_float(raw[c].w)};
        if (s == 2) {
            or3(rest, raw[c].x, raw[c].y);
            or3(rest, raw[c].z, raw[c].w);
        }
        const uint2 p = split_part(v, s == 2);
        raw[c].x = __float_as_uint(v[0]); raw[c].y = __float_as_uint(v[1]); raw[c].z = __float_as_uint(v[2]); raw[c].w = __float_as_uint(v[3]);
        *(uint2*)(stage + (c < PA ? wa[c] + s * PLA : wb[c - PA] + s * PLB)) = p;
    };

    // fragments: lane l holds row l % 32, k = 8 (l / 32) .. + 7 of a k-step of 16; transposing reads as in gemm_b16_kernel
    const int fr = lane & 31, half = lane >> 5;
    const int tk = 8 * half + ((lane & 15) >> 2), tcol = ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
    uint32_t ta[WM], tb[WN];
#pragma unroll
    for (int t = 0; t < WM; t++)
        ta[t] = AK ? half * KGA + (wm + t * 32 + fr) * 16 : (tk * BM + ((wm + t * 32) ^ (block_swizzle<BM * 2>(tk) * 8)) + tcol) * 2;
#pragma unroll
    for (int t = 0; t < WN; t++)
        tb[t] = 3 * PLA + (BKC ? half * KGB + (wn + t * 32 + fr) * 16 : (tk * BN + ((wn + t * 32) ^ (block_swizzle<BN * 2>(tk) * 8)) + tcol) * 2);
    const uint32_t smemAddr = (uint32_t)(uintptr_t)LDS3(smem_raw);
    // part s of k-step ks of the stage at `at`
    auto readA = [&](TrFragment (&f)[WM], int at, int ks, int s) {
#pragma unroll
        for (int t = 0; t < WM; t++) {
            if (AK) f[t].w = *(const u32x4*)(smem_raw + at + ta[t] + s * PLA + ks * 2 * KGA);
            else tr_read<BM * 2>(smemAddr + at + ta[t], s * PLA + ks * 16 * (BM * 2), f[t]);
        }
    };
    auto readB = [&](TrFragment (&f)[WN], int at, int ks, int s) {
#pragma unroll
        for (int t = 0; t < WN; t++) {
            if (BKC) f[t].w = *(const u32x4*)(smem_raw + at + tb[t] + s * PLB + ks * 2 * KGB);
            else tr_read<BN * 2>(smemAddr + at + tb[t], s * PLB + ks * 16 * (BN * 2), f[t]);
        }
    };
    auto arrived = [&](TrFragment (&a)[WM], TrFragment (&b)[WN]) {
#pragma unroll
        for (int t = 0; t < WM; t++)
            if (!AK) tr_wait(a[t]);
#pragma unroll
        for (int t = 0; t < WN; t++)
            if (!BKC) tr_wait(b[t]);
    };

    if (nk == 1) lastStage(kBegin);
#pragma unroll
    for (int c = 0; c < P; c++) fetch(c);
    nextStage();
#pragma unroll
    for (int c = 0; c < P; c++) {
#pragma unroll
        for (int s = 0; s < 3; s++) put(c, s, smem_raw);
        fetch(c);
    }
    __syncthreads();
    TrFragment ah[2][WM], bh[2][WN], am[WM], bm[WN], al[WM], bl[WN];
    readA(ah[0], 0, 0, 0);
    readB(bh[0], 0, 0, 0);
    arrived(ah[0], bh[0]);
    // stage u of two: in buffer u, its first h fragments in ah[KS u & 1], bh[KS u & 1]
    auto stage = [&](int u) {
        const int at = u * STAGE;
        unsigned char* next = smem_raw + STAGE - at;
        nextStage();
        if constexpr (SUMS) {
            putting++;
            turn = turn == 0 ? g.tilesN - 1 : turn - 1;
            mine = turn == 0 && putting < nk ? 0xffffffffu : 0u;   // past the end the last stage is put again
        }
        // what goes between the products: chunks of the next stage part by part to the other buffer, each then fetched anew
        constexpr int SLOTS = (6 * KS - 2) * NMF, STEPS = 3 * P;
        auto slot = [&](int q) {
#pragma unroll
            for (int st = STEPS * q / SLOTS; st < STEPS * (q + 1) / SLOTS; st++) {
                put(st / 3, st % 3, next);
                if (st % 3 == 2) fetch(st / 3);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int cur = (KS * u + ks) & 1, nxt = cur ^ 1;
            int q = ks * 6 * NMF;
            auto products = [&](TrFragment (&a)[WM], TrFragment (&b)[WN], bool fill) {
#pragma unroll
                for (int t = 0; t < NMF; t++) {
                    // the transposed tile (B as the row operand): a lane owns a row of C
                    acc[t / WN][t % WN] = BigTraits<bf16_t>::mma(b[t % WN].w, a[t / WN].w, acc[t / WN][t % WN]);
                    if (fill) slot(q + t);
                }
                q += NMF;
            };
            readA(am, at, ks, 1);
            readB(bm, at, ks, 1);
            products(ah[cur], bh[cur], true);
            arrived(am, bm);
            readA(al, at, ks, 2);
            readB(bl, at, ks, 2);
            products(ah[cur], bm, true);
            products(am, bh[cur], true);
            products(am, bm, true);
            arrived(al, bl);
            if (ks + 1 < KS) {
                readA(ah[nxt], at, ks + 1, 0);
                readB(bh[nxt], at, ks + 1, 0);
            } else {
                __syncthreads();
                readA(ah[nxt], STAGE - at, 0, 0);
                readB(bh[nxt], STAGE - at, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            products(ah[cur], bl, ks + 1 < KS);
            products(al, bh[cur], ks + 1 < KS);
            arrived(ah[nxt], bh[nxt]);
        }
    };
    for (int kt = 0; kt < nk; kt += 2) {
        stage(0);
        if (kt + 1 < nk) stage(1);
    }
    if constexpr (SUMS) {
        float* all = reinterpret_cast<float*>(smem_raw) + split_lds<WVM, WVN, WM, WN, KS, AK, BKC>();
        *(float4*)(all + 4 * tid) = make_float4(sums[0], sums[1], sums[2], sums[3]);
        __syncthreads();
        if (tid < BM && m0 + tid < M) {
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < NT / (BM / 4); w++) v += all[w * BM + tid];
            f32_row_part(g)[(size_t)(it.part * g.tilesN + n0 / BN) * M + m0 + tid] = v;
        }
    }
    if (rest & 0xffffu) flags->lost = 1;
    __syncthreads();
    if (flags->lost) {   // the same for the whole workgroup
        if (split_large<BM, 64 * WVM * WVN, AK>(baseA, g.lda, M - m0, kBegin, it.kEnd, tid) || split_large<BN, 64 * WVM * WVN, BKC>(baseB, g.ldb, N - n0, kBegin, it.kEnd, tid))
            flags->large = 1;
        __syncthreads();
    }
    if (split_lost(acc, *flags, it.kEnd - kBegin)) f32_sums<WM, WN, AK, BKC, false>(g, A, B, m0 + wm, n0 + wn, kBegin, it.kEnd, lane, acc);
    else if (!VEC && kEnd < it.kEnd) f32_sums<WM, WN, AK, BKC, true>(g, A, B, m0 + wm, n0 + wn, kEnd, it.kEnd, lane, acc);
    f32_store<WM, WN, HEADS>(g, hp, acc, reinterpret_cast<float*>(smem_raw) + wave * 32 * (32 * WN + 4), lane, m0 + wm, n0 + wn, it.part, it.batch);
}
// ---------------------------------------------------------------------------
// Products that do not fill the chip with the tiles above: 32 x 32 of C to a workgroup, every stage of the contraction dealt to its
// NW wavefronts, whose sums are added up through LDS at the end.
// With tiles of 64 x 64 such a product is a chain of short stages on a few CUs (1024 x 288 x 288: 80 workgroups, nine stages of 32 k,
// each longer than its 1024 cycles of MFMA by a trip through LDS and a barrier), and cutting the contraction over workgroups costs a
// second launch of 4 us.  Here there are four times the workgroups, a stage is 64 k that go from memory straight into LDS, two of
// them under way and three workgroups to a CU, and a wavefront's share of it is 16 k.  What bounds it is the fp32 matrix core of a
// CU, 0.21 us for a tile's stage of 0.36, and the latency of the first fetch and of the end, some 2.5 us.
// Fragments fetched from memory straight into registers take 1.5 - 2 times as long (1024 x 288 x 288: 8.5 us): 32 rows of 32 bytes to
// an instruction.  Stages of 128 k, two workgroups to a CU: 768 x 768 x 700 15.5 instead of 12.5 us, the same where every CU has
// one; eight wavefronts, five stages, fragments read a stage ahead: no better.
// Measured, before and now, us: 1024 x 288 x 288 8.7 -> 5.8, 1024 x 288 x 768 12.6 -> 9.9, 768 x 288 x 1024 (A^T B, beta 1) 13.3 -> 8.7,
// 768 x 768 x 700 (A^T B) 17.1 -> 12.6, 24 times 256 x 48 x 256 with a transposed operand 8.3 -> 5.7, 96 x 192 x 48 4.4 -> 2.9.
//
// LDS holds [row][k] for an operand with k at unit stride, the 16-byte piece c of row r at c ^ (r & 15), and [k][row] for the other,
// k and k + 4 of every eight next to each other: the two halves of a wavefront, four k apart, then read from the two halves of the banks.
//
// VEC: as above; otherwise 4 bytes per lane go into LDS, to the same places.
// rowSums: null, or a value for every row of C to which the sum of the row of A is added (by the tiles of the first columns).
constexpr int SMALL_STAGES = 3;
constexpr int SMALL_TILE_COST = 84;   // what a tile costs beside its contraction, in k (the last term of gemm_f32_small_time)
// LEVELS: sums of eight stages each, which are added up: the rounding of a long contraction like that of one cut into parts (130 x 768 x
// 2304: error against float64 4.3e-7 in one run, 2.1e-7 so).
template <int NW, int BK, bool AK, bool BKC, bool VEC, bool HEADS, bool LEVELS = false>
__device__ __forceinline__ void f32_small_tile(const GemmF32Args& g, const HeadsArg<HEADS>& hp, const F32Item& it, float* rowSums, float* smem)
{
    constexpr int NT = 64 * NW, W = VEC ? 4 : 1, P = 32 * BK / W / NT, STAGE = 2 * 32 * BK, S = SMALL_STAGES;   // values per lane and fetch; fetches per thread, operand and stage
    constexpr int LDC = 36;                                                                     // floats between rows of a wavefront's sums in LDS
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kBegin = it.kBegin, kEnd = it.kEnd;
    constexpr uint32_t OUTSIDE = 0x80000000u;
    auto resource = [](const void* base) { return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)(OUTSIDE - 16), 0x00020000); };
    const float* baseA = g.A + (size_t)it.batch * g.sA + (AK ? (size_t)it.m0 * g.lda : (size_t)it.m0);
    const float* baseB = g.B + (size_t)it.batch * g.sB + (BKC ? (size_t)it.n0 * g.ldb : (size_t)it.n0);
    const __amdgpu_buffer_rsrc_t rsA = resource(baseA), rsB = resource(baseB);
    const char *stageA = (const char*)(baseA + (size_t)kBegin * g.lda), *stageB = (const char*)(baseB + (size_t)kBegin * g.ldb);
    // value e of a stage, k at unit stride: piece e % BK / 4 of row e / BK holds k = 4 (piece ^ (row & 15)) .. + 3; row index at unit
    // stride: row e % 32 of the k at place e / 32, where k and k + 4 of every eight are next to each other
    auto valueK = [&](bool kFast, int e) { return kFast ? (4 * (e % BK / 4 ^ (e / BK & 15)) | (e & 3)) : ((e / 32) & ~7) | ((e / 32 & 1) << 2) | (e / 64 & 3); };
    auto valueRow = [&](bool kFast, int e, int left) { return min(kFast ? e / BK : e % 32, kFast || !VEC ? left - 1 : left - 4); };
    uint32_t va[P], vb[P];
#pragma unroll
    for (int p = 0; p < P; p++) {
        const int e = W * (tid + NT * p), ka = valueK(AK, e), kb = valueK(BKC, e), ra = valueRow(AK, e, g.M - it.m0), rb = valueRow(BKC, e, g.N - it.n0);
        va[p] = 4 * (AK ? (uint32_t)ra * (uint32_t)g.lda + ka : (uint32_t)ka * (uint32_t)g.lda + ra);
        vb[p] = 4 * (BKC ? (uint32_t)rb * (uint32_t)g.ldb + kb : (uint32_t)kb * (uint32_t)g.ldb + rb);
    }
    const int nk = (kEnd - kBegin + BK - 1) / BK;
    int fetched = 0;
    auto fetch = [&](float* stage) {
        const int k0 = kBegin + fetched * BK;
        if (fetched + 1 == nk) {   // what lies past the end of the contraction
#pragma unroll
            for (int p = 0; p < P; p++) {
                const int e = W * (tid + NT * p);
                if (k0 + valueK(AK, e) >= kEnd) va[p] = OUTSIDE;
                if (k0 + valueK(BKC, e) >= kEnd) vb[p] = OUTSIDE;
            }
        }
#pragma unroll
        for (int p = 0; p < P; p++) {
            float* to = stage + (p * NT + wave * 64) * W;
            if (AK) lds_fetch<4 * W>(rsA, to, va[p], k0 * 4);
            else lds_fetch<4 * W>(resource(stageA), to, va[p], 0);
        }
#pragma unroll
        for (int p = 0; p < P; p++) {
            float* to = stage + 32 * BK + (p * NT + wave * 64) * W;
            if (BKC) lds_fetch<4 * W>(rsB, to, vb[p], k0 * 4);
            else lds_fetch<4 * W>(resource(stageB), to, vb[p], 0);
        }
        stageA += (size_t)(BK * sizeof(float)) * g.lda;
        stageB += (size_t)(BK * sizeof(float)) * g.ldb;
        fetched++;
    };
    const int fr = lane & 31, half = lane >> 5;
    // unit of eight k: a lane's four k
    auto fragment = [&](bool kFast, const float* stage, int unit) {
        u32x4 v;
        if (kFast) return *(const u32x4*)(stage + fr * BK + 4 * ((2 * unit + half) ^ (fr & 15)));
        const uint32_t* q = (const uint32_t*)(stage + (8 * unit + half) * 32 + fr);
        v.x = q[0]; v.y = q[64]; v.z = q[128]; v.w = q[192];
        return v;
    };
    floatx16 acc;
    [[maybe_unused]] floatx16 all;
#pragma unroll
    for (int v = 0; v < 16; v++) { acc[v] = 0.f; all[v] = 0.f; }
    // a row's sum as two, with LEVELS also in levels (the bias gradient of 3667 rows: error against float64 2.1e-7 as one in one run, 1.2e-7 so)
    const bool sumRows = rowSums && it.n0 == 0;
    constexpr int J = BK / 8 / NW;
    float rowSum[J] = {}, rowAll = 0.f;
#pragma unroll
    for (int i = 0; i < S - 1; i++)
        if (i < nk) fetch(smem + i * STAGE);
    int buf = 0, free = S - 1;
    auto step = [&](int kt) {
        // the stage has landed, of this wavefront and then of all, while the stages after it are still on their way (__syncthreads
        // would wait for those too)
        if (kt + S - 2 < nk) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(2 * P * (S - 2)) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" : : : "memory");
        const float* stage = smem + buf * STAGE;
        buf = buf == S - 1 ? 0 : buf + 1;
        const int units = (min(BK, kEnd - kBegin - kt * BK) + 7) / 8;
        u32x4 a[J], b[J];
#pragma unroll
        for (int j = 0; j < J; j++) {
            a[j] = fragment(AK, stage, wave + NW * j);
            b[j] = fragment(BKC, stage + 32 * BK, wave + NW * j);
        }
        if (kt + S - 1 < nk) {   // into the buffer of stage kt - 1, whose fragments every wavefront has had since the barrier
            fetch(smem + free * STAGE);
            free = free == S - 1 ? 0 : free + 1;
        }
#pragma unroll
        for (int j = 0; j < J; j++)
            if (NW * j < units) acc = BigTraits<float>::mma(b[j], a[j], acc);   // the transposed tile (B as the row operand): a lane owns a row of C
        if (sumRows)
#pragma unroll
            for (int j = 0; j < J; j++)   // zeros past the end
                rowSum[j] += (__uint_as_float(a[j].x) + __uint_as_float(a[j].y)) + (__uint_as_float(a[j].z) + __uint_as_float(a[j].w));
    };
    if constexpr (LEVELS) {
        for (int kt = 0; kt < nk;) {
            const int end = min(nk, kt + 8);
            for (; kt < end; kt++) step(kt);
#pragma unroll
            for (int v = 0; v < 16; v++) { all[v] += acc[v]; acc[v] = 0.f; }
#pragma unroll
            for (int j = 0; j < J; j++) { rowAll += rowSum[j]; rowSum[j] = 0.f; }
        }
        acc = all;
    } else
        for (int kt = 0; kt < nk; kt++) step(kt);
    __syncthreads();
    float* slice = smem + wave * 32 * LDC;
#pragma unroll
    for (int q = 0; q < 4; q++) *(float4*)(slice + fr * LDC + 8 * q + 4 * half) = make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
    if (sumRows) {
#pragma unroll
        for (int j = 0; j < J; j++) rowAll += rowSum[j];
        smem[NW * 32 * LDC + tid] = rowAll;
    }
    __syncthreads();
    if (sumRows && tid < 32 && it.m0 + tid < g.M) {
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < 2 * NW; w++) t += smem[NW * 32 * LDC + 32 * w + tid];
        rowSums[it.m0 + tid] += t;
    }
    const int r = it.m0 + (tid >> 3), c = it.n0 + (tid & 7) * 4;   // four columns of a row each
    if (tid >= 256 || r >= g.M || c >= g.N) return;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; w++) {
        const float4 t = *(const float4*)(smem + (w * 32 + (tid >> 3)) * LDC + (tid & 7) * 4);
        v[0] += t.x; v[1] += t.y; v[2] += t.z; v[3] += t.w;
    }
    const float4 bias = f32_bias4(g.bias, c, g.N);
    v[0] = g.alpha * v[0] + bias.x; v[1] = g.alpha * v[1] + bias.y; v[2] = g.alpha * v[2] + bias.z; v[3] = g.alpha * v[3] + bias.w;
    if constexpr (HEADS) {
        heads_store4(hp.he, r, c, g.N, g.vecC, heads_col<float>(hp.he, c), v);
        return;
    }
    float* cp = g.C + (size_t)it.batch * g.sC + (size_t)r * g.ldc + c;
    if (g.vecC) {
        if (g.beta != 0.f) {
            const float4 o = *(const float4*)cp;
            v[0] += g.beta * o.x; v[1] += g.beta * o.y; v[2] += g.beta * o.z; v[3] += g.beta * o.w;
        }
        *(float4*)cp = make_float4(v[0], v[1], v[2], v[3]);
    } else {
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (c + q < g.N) cp[q] = v[q] + (g.beta != 0.f ? g.beta * cp[q] : 0.f);
    }
}

template <int NW, int BK, bool AK, bool BKC, bool VEC, bool HEADS>
__global__ __launch_bounds__(64 * NW) void gemm_f32_small_kernel(GemmF32Args g, HeadsArg<HEADS> hp)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int total = g.tilesM * g.tilesN * g.parts, item = xcd_item(total);
    if (item >= total) return;
    F32Item it;
    f32_item<32, 32>(g, item, it);
    f32_small_tile<NW, BK, AK, BKC, VEC, HEADS>(g, hp, it, nullptr, reinterpret_cast<float*>(smem_raw));
}

// The gradients of an inner product whose products do not fill the chip, as one launch: w is dW += dY^T X, its tiles of the first
// columns add the column sums of dY to db, and x is dX = dY W.  Apart they are three or four launches, each with its own first
// fetch and end, on half the CUs.  (The ones with the longer contraction come
// first, in runs of equal work, xcd_runs.h.)  Calls in a row, us, apart and together: 1024 rows, 288 to 768 23.9 and 15.1, 288 to 864 25.4 and
// 16.6, 768 to 288 21.2 and 15.5; 200 rows, 384 to 1536 21.6 and 13.4; 1500 rows, 768 to 768 53 and 40; 2800 rows, 768 to 768 65 and 69.
template <int NW, int BK, bool VEC, bool LEVELS>
__global__ __launch_bounds__(64 * NW) void linear_bwd_f32_small_kernel(GemmF32Args w, GemmF32Args x, float* db, XcdRuns runs)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    float* smem = reinterpret_cast<float*>(smem_raw);
    const int tilesW = w.tilesM * w.tilesN, tilesX = x.tilesM * x.tilesN, at = runs.first[blockIdx.x % 8] + (int)(blockIdx.x / 8), end = runs.first[blockIdx.x % 8 + 1];
    asm volatile("" : : "s"(w.K), "s"(x.K), "s"(tilesW), "s"(tilesX), "s"(at), "s"(end));   // one trip for the arguments, not one after the other
    if (at >= end) return;
    const int item = w.K >= x.K ? at : at < tilesX ? tilesW + at : at - tilesX;
    F32Item it;
    if (item < tilesW) {
        f32_item<32, 32>(w, item, it);
        f32_small_tile<NW, BK, false, false, VEC, false, LEVELS>(w, HeadsArg<false>(), it, db, smem);
    } else {
        f32_item<32, 32>(x, item - tilesW, it);
        f32_small_tile<NW, BK, true, false, VEC, false, LEVELS>(x, HeadsArg<false>(), it, nullptr, smem);
    }
}

// the row sums that gemm_f32_sum_kernel adds to `sum`: `count` partial ones for each of M rows, by its first `blocks` workgroups
struct F32RowSums { int blocks, count; const float* part; float* sum; };
// C = sum over the S partial products, in their order (alpha is in them already), + beta C; or through the heads epilogue
template <bool HEADS>
__global__ __launch_bounds__(256) void gemm_f32_sum_kernel(const float* __restrict__ part, int S, int M, int N, long long ldc, float beta, bool vecC,
                                                           float* __restrict__ C, const float* __restrict__ bias, HeadsArg<HEADS> hp, F32RowSums rows)
{
    const int block = (int)blockIdx.x - rows.blocks;
    if (block < 0) {   // the first workgroups: the partial row sums
        const int r = (int)blockIdx.x * 256 + threadIdx.x;
        if (r >= M) return;
        rows.sum[r] += sum_partials(rows.part + r, rows.count, M);
        return;
    }
    const int quads = (N + 3) / 4;
    const size_t mn = (size_t)M * N;
    for (size_t e = (size_t)block * blockDim.x + threadIdx.x; e < (size_t)M * quads; e += (size_t)blockDim.x * (gridDim.x - rows.blocks)) {
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
// How a product is cut: the tile and the number of parts of the contraction with the smallest estimated time.  A split contraction
// pays for a second launch and for the partial products' way through memory (of at most wsBytes).  Estimates in microseconds.
struct GemmF32Plan { int shape, splits, kChunk; };

template <typename TIME>
static GemmF32Plan best_plan(int m, int n, int k, int batch, bool causal, size_t wsBytes, int shapes, const int (*tile)[2], double* estimate, TIME time)
{
    GemmF32Plan best = {shapes - 1, 1, k};
    double bestT = 1e30;
    for (int sh = 0; sh < shapes; sh++) {
        const long long tiles = (long long)((m + tile[sh][0] - 1) / tile[sh][0]) * ((n + tile[sh][1] - 1) / tile[sh][1]) * batch;
        for (int S = 1; S <= 32; S++) {
            if (S > 1 && (batch > 1 || causal || k / S < 128 || (size_t)S * m * n * sizeof(float) > wsBytes)) break;
            const int chunk = S > 1 ? ((k + S - 1) / S + 31) / 32 * 32 : k;
            if ((k + chunk - 1) / chunk != S) continue;
            double t = time(sh, tiles * S, ((tiles * S + 7) / 8 + 31) / 32, chunk);
            if (S > 1) t += 4.5 + (double)(S + 1) * m * n * 4.0 / 4.0e6;
            if (t < bestT) { bestT = t; best = {sh, S, chunk}; }
        }
    }
    *estimate = bestT;
    return best;
}

// gemm_f32_kernel.  Cycles of a tile: its products at 256 flops per cycle and CU over the efficiency of a CU's two or more
// workgroups, and its first fetches and its stores; a workgroup alone on its CU shows every stage's latency.  Fitted to tiles of
// 768 and 2304 k: 128 x 192 (one workgroup per CU: nothing covers its ends) 176k / 500k cycles, 128 x 128 111k / 332k, 64 x 128
// 59k / 169k, 64 x 64 31k / 88k.
static GemmF32Plan gemm_f32_plan(int m, int n, int k, int batch, bool causal, size_t wsBytes, double* estimate)
{
    static const int tile[4][2] = {{128, 192}, {128, 128}, {64, 128}, {64, 64}};
    static const struct { double eff, ends, alone; } fit[4] = {{0.909, 14000, 1.10}, {0.89, 600, 1.30}, {0.895, 4000, 1.45}, {0.863, 2200, 1.60}};
    return best_plan(m, n, k, batch, causal, wsBytes, 4, tile, estimate, [](int sh, long long, long long perCu, int chunk) {
        const double body = 2.0 * tile[sh][0] * tile[sh][1] * ((chunk + 31) / 32 * 32) / 256.0;
        return (perCu == 1 ? body * fit[sh].alone + fit[sh].ends : perCu * (body / fit[sh].eff + fit[sh].ends)) / 2400.0;
    });
}

static const int g_splitTile[6][2] = {{256, 256}, {256, 192}, {128, 192}, {128, 128}, {64, 128}, {64, 64}};   // of gemm_f32_split_kernel

// gemm_f32_split_kernel.  Microseconds: what the workgroups of the busiest CU take for their stages and ends, and, because the
// clock follows the load, a share that grows with the workgroups in all.  Fitted by least squares to 700 measurements of 40 sizes
// in three layouts and up to 16 parts; the tile chosen is within 1 % of the best one on average, 8 % at most.
static GemmF32Plan gemm_f32_split_plan(int m, int n, int k, int batch, bool causal, size_t wsBytes, double* estimate)
{
    struct Fit { double stage, ends, loadStage, loadEnds, once; };
    static const struct { int k; Fit alone, shared; } fit[6] = {
        {16, {1.475, 9.5, 0.34, 0, 0}, {1.56, 4.9, 0.64, 0, 0}},      {16, {1.125, 9.55, 0.36, 0, 0}, {1.153, 5.7, 0.55, 0, 0}},
        {16, {0.817, 8.9, 0.156, 0.7, 0}, {0.546, 3.1, 0.39, 0, 0}},  {16, {0.669, 3.64, 0, 5.0, 0}, {0.383, 0.25, 0.286, 0, 2.4}},
        {32, {0.89, 1.3, 0.066, 2.1, 1.1}, {0.457, 0, 0.332, 0, 5.4}}, {32, {0.637, 1.1, 0.056, 1.07, 0}, {0.307, 0, 0.133, 0.38, 3.0}}};
    return best_plan(m, n, k, batch, causal, wsBytes, 6, g_splitTile, estimate, [](int sh, long long items, long long perCu, int chunk) {
        const Fit& f = perCu == 1 ? fit[sh].alone : fit[sh].shared;
        const double nk = (chunk + fit[sh].k - 1) / fit[sh].k, load = items / 256.0;
        return perCu * (nk * f.stage + f.ends) + load * (nk * f.loadStage + f.loadEnds) + f.once;
    });
}

// gemm_f32_small_kernel, microseconds: what the workgroups of the busiest CU take for their products, and what each three of them that
// run at once (by LDS) take for their stages' latencies.  Within 10 % of 34 sizes.
static double gemm_f32_small_time(long long tiles, int k)
{
    const long long perCu = ((tiles + 7) / 8 + 31) / 32;
    return 1.7 + (double)((perCu + 2) / 3) * (0.8 + 0.28 * k / 128) + (double)perCu * (0.3 + 0.46 * k / 128);
}

// Which kernel takes a product, and its plan.  (fp32Sums also for a result in an operand's memory: the other two kernels read
// operands while some of the result is written, the small tiles of one part of the rows and columns each, the split one once more
// for a wavefront whose parts lost something.)  The bf16 matrix cores from 64 k on (below, the split's error is larger than that of the
// fp32 matrix cores) and from 2^28 multiplications on (2048 x 512 x 384: 10.2 against 11.0 us; below, the chip is not full, and 16 x 288 x
// 32000 takes 51 against 44 us); 32 x 32 tiles where their estimate is the smallest, which is a tenth of a round of the larger ones.
enum { F32_TILES, F32_SPLIT, F32_SMALL };
struct GemmF32Choice { int kernel; GemmF32Plan plan; double time; };
static GemmF32Choice gemm_f32_choose(int m, int n, int k, int batch, bool causal, size_t wsBytes, bool fp32Sums, bool heads = false)
{
    GemmF32Choice c;
    c.kernel = F32_TILES;
    c.plan = gemm_f32_plan(m, n, k, batch, causal, wsBytes, &c.time);
    if (fp32Sums) return c;
    if (k >= 64 && (double)m * n * k * batch >= 268435456.0) {   // faster than the fp32 matrix cores at every size from there on
        c.kernel = F32_SPLIT;
        c.plan = gemm_f32_split_plan(m, n, k, batch, causal, wsBytes, &c.time);
    }
    c.time += 1.8;   // a launch, which the next estimate holds
    // the heads epilogue of 16 rows and more a lane, one after the other (1024 x 864 x 288: 13.3 us, 9.3 without it)
    if (heads) c.time += 3;
    const double t = gemm_f32_small_time((long long)((m + 31) / 32) * ((n + 31) / 32) * batch, k);
    if (t < c.time) c = {F32_SMALL, {0, 1, k}, t};
    return c;
}

int gemm_f32_route(int m, int n, int k, int batch, bool causal, bool fp32Sums, bool heads)
{
    const GemmF32Choice c = gemm_f32_choose(m, n, k, batch, causal, SIZE_MAX, fp32Sums, heads);
    return c.kernel + 4 * c.plan.shape + 64 * c.plan.splits;
}

// 31-bit byte offsets within a tile's rows of k (256 at most), or within the k rows of a stage (128)
static bool f32_near(bool kFast, int rows, int k, long long ld) { return (kFast ? (std::min(rows, 256) + 1) * ld : std::min(k, 128) * ld + 256) < (1ll << 29); }

size_t gemm_f32_workspace_bytes(int m, int n, int k, int batch, bool causal)
{
    if (m <= 0 || n <= 0 || k <= 0) return 0;
    // which kernel takes it depends on the caller too: enough for any
    const int splits = std::max(gemm_f32_choose(m, n, k, batch, causal, SIZE_MAX, false).plan.splits, gemm_f32_choose(m, n, k, batch, causal, SIZE_MAX, true).plan.splits);
    return splits > 1 ? (size_t)splits * m * n * sizeof(float) : 0;
}

// With the sums of op(A)'s rows: the partial products (none where the contraction is not cut), then the partial sums.  0: not together,
// because another kernel takes the product, because a sum would be longer than the column sums' own (128 values in each of eight
// accumulators and more a row and tile), or because one short launch (up to 1024 k) would only be another.
static int split_tile_columns(int shape, int n) { return (n + g_splitTile[shape][1] - 1) / g_splitTile[shape][1]; }
size_t gemm_f32_row_sums_workspace_bytes(int m, int n, int k, bool vec)
{
    if (m <= 0 || n <= 0 || k <= 0 || !vec || !f32_near(false, m, k, m) || !f32_near(false, n, k, n)) return 0;
    const GemmF32Choice c = gemm_f32_choose(m, n, k, 1, false, SIZE_MAX, false);
    if (c.kernel != F32_SPLIT || (k <= 1024 && c.plan.splits == 1)) return 0;
    const int columns = split_tile_columns(c.plan.shape, n);
    if (c.plan.kChunk / (8 * columns) > 128) return 0;
    return ((c.plan.splits > 1 ? (size_t)c.plan.splits * m * n : 0) + (size_t)c.plan.splits * columns * m) * sizeof(float);
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
    if (p.shape == 0) return launch_f32<2, 3, 1, AK, BKC, VEC, HEADS>(s, a, p.splits, batch, he);
    if (p.shape == 1) return launch_f32<2, 2, 2, AK, BKC, VEC, HEADS>(s, a, p.splits, batch, he);
    if (p.shape == 2) return launch_f32<1, 2, 2, AK, BKC, VEC, HEADS>(s, a, p.splits, batch, he);
    return launch_f32<1, 1, 3, AK, BKC, VEC, HEADS>(s, a, p.splits, batch, he);
}

// the shapes of gemm_f32_split_kernel, in the order of gemm_f32_split_plan: wavefronts, tiles of a wavefront, k-steps of a stage,
// wavefronts of a SIMD that the registers are to hold
#define SPLIT_SHAPES(X) X(0, 2, 4, 4, 2, 1, 2) X(1, 4, 2, 2, 3, 1, 2) X(2, 2, 2, 2, 3, 1, 2) X(3, 2, 2, 2, 2, 1, 2) X(4, 2, 2, 1, 2, 2, 2) X(5, 2, 2, 1, 1, 2, 2)

template <int WVM, int WVN, int WM, int WN, int KS, int OCC, bool AK, bool BKC, bool VEC, bool HEADS, bool SUMS>
static hipError_t launch_split(hipStream_t s, GemmF32Args& g, int splits, int batch, const HeadsEpilogue* he)
{
    constexpr int BM = 32 * WVM * WM, BN = 32 * WVN * WN;
    constexpr int lds = split_flags_at<WVM, WVN, WM, WN, KS, AK, BKC, SUMS>() + (int)sizeof(SplitFlags);
    static const hipError_t attr = hipFuncSetAttribute((const void*)gemm_f32_split_kernel<WVM, WVN, WM, WN, KS, OCC, AK, BKC, VEC, HEADS, SUMS>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (attr != hipSuccess) return attr;
    g.tilesM = (g.M + BM - 1) / BM;
    g.tilesN = (g.N + BN - 1) / BN;
    g.parts = splits > 1 ? splits : batch;
    const long long total = (long long)g.tilesM * g.tilesN * g.parts;
    if (total > (1ll << 27)) return hipErrorInvalidValue;
    const int per = (int)((total + 7) / 8);
    hipLaunchKernelGGL((gemm_f32_split_kernel<WVM, WVN, WM, WN, KS, OCC, AK, BKC, VEC, HEADS, SUMS>), dim3(per * 8), 64 * WVM * WVN, lds, s, g, heads_arg<HEADS>(he));
    return hipGetLastError();
}

template <bool AK, bool BKC, bool VEC, bool HEADS, bool SUMS = false>
static hipError_t launch_split_shape(hipStream_t s, GemmF32Args& a, const GemmF32Plan& p, int batch, const HeadsEpilogue* he = nullptr)
{
    switch (p.shape) {
#define X(I, WVM, WVN, WM, WN, KS, OCC) case I: return launch_split<WVM, WVN, WM, WN, KS, OCC, AK, BKC, VEC, HEADS, SUMS>(s, a, p.splits, batch, he);
        SPLIT_SHAPES(X)
#undef X
    }
    return hipErrorInvalidValue;
}

// LDS of gemm_f32_small_kernel: the stages, in which the sums find room at the end
template <int NW, int BK> constexpr int small_lds() { static_assert(SMALL_STAGES * 2 * 32 * BK >= NW * (32 * 36 + 64), ""); return SMALL_STAGES * 2 * 32 * BK * (int)sizeof(float); }

template <int NW, int BK, bool AK, bool BKC, bool VEC, bool HEADS>
static hipError_t launch_small(hipStream_t s, const GemmF32Args& a, int batch, const HeadsEpilogue* he)
{
    constexpr int lds = small_lds<NW, BK>();
    static const hipError_t attr = hipFuncSetAttribute((const void*)gemm_f32_small_kernel<NW, BK, AK, BKC, VEC, HEADS>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (attr != hipSuccess) return attr;
    GemmF32Args g = a;
    g.tilesM = (g.M + 31) / 32;
    g.tilesN = (g.N + 31) / 32;
    g.parts = batch;
    g.kChunk = g.K;
    const long long total = (long long)g.tilesM * g.tilesN * batch;
    if (total > (1ll << 27)) return hipErrorInvalidValue;
    const int per = (int)((total + 7) / 8);
    hipLaunchKernelGGL((gemm_f32_small_kernel<NW, BK, AK, BKC, VEC, HEADS>), dim3(per * 8), 64 * NW, lds, s, g, heads_arg<HEADS>(he));
    return hipGetLastError();
}

// VEC: operands in whole aligned 16-byte chunks
template <bool AK, bool BKC, bool VEC, bool HEADS>
static hipError_t launch_layout(hipStream_t s, GemmF32Args& a, const GemmF32Choice& c, int batch, const HeadsEpilogue* he)
{
    if (c.kernel == F32_SMALL) return launch_small<4, 64, AK, BKC, VEC, HEADS>(s, a, batch, he);
    if (c.kernel == F32_SPLIT) return launch_split_shape<AK, BKC, VEC, HEADS>(s, a, c.plan, batch, he);
    return launch_f32_tile<AK, BKC, VEC, HEADS>(s, a, c.plan, batch, he);
}

bool gemm_f32_shares(const GemmF32& q)
{
    auto values = [&](bool kFast, int rows, long long ld, long long stride) { return (q.batch - 1) * stride + (kFast ? (rows - 1) * ld + q.k : (q.k - 1) * ld + rows); };
    const long long out = (q.batch - 1) * q.sC + (q.m - 1) * q.ldc + q.n;
    return result_meets(q.C, out, q.heads, q.m, q.n, q.A, values(q.aK, q.m, q.lda, q.sA)) || result_meets(q.C, out, q.heads, q.m, q.n, q.B, values(q.bK, q.n, q.ldb, q.sB));
}

hipError_t gemm_f32(hipStream_t s, const GemmF32& q, void* ws, size_t wsBytes)
{
    if (q.m <= 0 || q.n <= 0 || q.batch <= 0) return hipSuccess;
    if (q.k <= 0 || (q.causal && ((q.causal >= CAUSAL_B_LOWER ? q.n : q.m) != q.k || !q.flag)) || (q.heads && (q.alpha != 1.f || q.beta != 0.f || q.batch != 1 || !q.aK || !q.bK)))
        return hipErrorInvalidValue;
    GemmF32Args a = {};
    a.M = q.m; a.N = q.n; a.K = q.k;
    a.A = q.A; a.B = q.B; a.C = q.C;
    a.lda = q.lda; a.ldb = q.ldb; a.ldc = q.ldc; a.sA = q.sA; a.sB = q.sB; a.sC = q.sC;
    a.alpha = q.alpha; a.beta = q.beta;
    a.causal = q.causal; a.flag = q.flag; a.epoch = q.epoch;
    a.part = (float*)ws;
    a.bias = q.heads ? (const float*)q.heads->bias : q.bias;
    if (q.heads) {
        const HeadsEpilogue& he = *q.heads;
        a.vecC = q.n % 4 == 0 && he.hs % 4 == 0 && (((uintptr_t)he.dst[0] | (uintptr_t)he.dst[1] | (uintptr_t)he.dst[2]) & 15) == 0;
    } else {
        a.vecC = q.n % 4 == 0 && q.ldc % 4 == 0 && (q.batch == 1 || q.sC % 4 == 0) && ((uintptr_t)q.C & 15) == 0;
    }
    const bool near = f32_near(q.aK, q.m, q.k, q.lda) && f32_near(q.bK, q.n, q.k, q.ldb);
    const bool vec = near && (((uintptr_t)q.A | (uintptr_t)q.B) & 15) == 0 && q.lda % 4 == 0 && q.ldb % 4 == 0 && (q.batch == 1 || (q.sA % 4 == 0 && q.sB % 4 == 0)) &&
                     (q.aK ? q.k % 4 == 0 : q.m % 4 == 0) && (q.bK ? q.k % 4 == 0 : q.n % 4 == 0);
    if (!ws || ((uintptr_t)ws & 15)) wsBytes = 0;
    const GemmF32Choice choice = gemm_f32_choose(q.m, q.n, q.k, q.batch, q.causal != 0, wsBytes, q.fp32Sums || !near || gemm_f32_shares(q), q.heads != nullptr);
    const GemmF32Plan& p = choice.plan;
    a.kChunk = p.kChunk;
    if (q.rowSum) {
        const size_t need = gemm_f32_row_sums_workspace_bytes(q.m, q.n, q.k, vec && !q.aK && !q.bK && q.lda == q.m && q.ldb == q.n && q.batch == 1 && !q.fp32Sums);
        if (need == 0 || wsBytes < need || choice.kernel != F32_SPLIT) return hipErrorInvalidValue;
    }
    // rows shorter than the three values that a chunk may read past one: so many more k
    auto past = [&](bool kFast, int rows, long long ld) { return kFast ? q.k % 4 : rows % 4 == 0 ? 0 : ld >= 3 ? 1 : 3; };
    a.kTail = std::max(past(q.aK, q.m, q.lda), past(q.bK, q.n, q.ldb));
    hipError_t e;
    if (q.rowSum) e = launch_split_shape<false, false, true, false, true>(s, a, p, 1);
    else if (q.heads) e = vec ? launch_layout<true, true, true, true>(s, a, choice, 1, q.heads) : launch_layout<true, true, false, true>(s, a, choice, 1, q.heads);
#define LAYOUT(AKV, BKV) (vec ? launch_layout<AKV, BKV, true, false>(s, a, choice, q.batch, nullptr) : launch_layout<AKV, BKV, false, false>(s, a, choice, q.batch, nullptr))
    else if (q.aK) e = q.bK ? LAYOUT(true, true) : LAYOUT(true, false);
    else e = q.bK ? LAYOUT(false, true) : LAYOUT(false, false);
#undef LAYOUT
    F32RowSums rows = {};
    if (q.rowSum) rows = {(q.m + 255) / 256, p.splits * a.tilesN, a.part + (p.splits > 1 ? (size_t)p.splits * q.m * q.n : 0), q.rowSum};
    const size_t quads = (size_t)q.m * ((q.n + 3) / 4);
    const int grid = rows.blocks + (p.splits > 1 ? (int)std::min<size_t>((quads + 255) / 256, 4096) : 0);
    if (e != hipSuccess || grid == 0) return e;
    if (q.heads) hipLaunchKernelGGL(gemm_f32_sum_kernel<true>, grid, 256, 0, s, (const float*)ws, p.splits, q.m, q.n, q.ldc, q.beta, a.vecC, q.C, a.bias, heads_arg<true>(q.heads), rows);
    else hipLaunchKernelGGL(gemm_f32_sum_kernel<false>, grid, 256, 0, s, (const float*)ws, p.splits, q.m, q.n, q.ldc, q.beta, a.vecC, q.C, a.bias, HeadsArg<false>(), rows);
    return hipGetLastError();
}

// Whether the gradients of an inner product (m rows, n outputs, k inputs) are one launch, and whether that adds in levels.
struct LinearBwdF32Plan { bool together, levels; };
static LinearBwdF32Plan linear_bwd_f32_plan(int m, int n, int k, bool bias, bool vec)
{
    if (!f32_near(false, n, m, n) || !f32_near(false, k, m, k) || !f32_near(true, m, n, n) || !f32_near(false, k, n, k)) return {false, false};
    const long long tilesK = (k + 31) / 32, tilesW = (n + 31) / 32 * tilesK, tilesX = (m + 31) / 32 * tilesK;
    if (tilesW + tilesX > (1ll << 20)) return {false, false};
    // against the launches apart: their estimates, that of the column sums (one launch, two from 1025 rows on), and 2.5 us for each
    // time that one launch waits for the last one's stores
    const bool sumsToo = bias && gemm_f32_row_sums_workspace_bytes(n, k, m, vec) > 0;   // the column sums with the weight gradient
    const GemmF32Choice dw = gemm_f32_choose(n, k, m, 1, false, SIZE_MAX, false), dx = gemm_f32_choose(m, k, n, 1, false, SIZE_MAX, false);
    const double apart = dw.time + dx.time + 2.5 +
                         (!bias ? 0.0 : sumsToo ? dw.plan.splits > 1 ? 0.5 : 4.5 : m <= 1024 ? 4.5 : 9.0);
    // the one launch, fitted to 43 sizes (0.8 .. 1.24 of what was measured, 4.4 to 199 us); a tenth on top of it, as both sides are estimates.  In
    // 4-byte pieces it takes a quarter longer, and so do the products apart, except in the split kernel: beside two of those an estimate of
    // its own, fitted to 179 sizes (971 rows, 1996 to 1045: 96 us together, 87 apart; 2385 rows, 2252 to 770 210 and 142)
    const double tiles = (double)(tilesW + tilesX), work = (double)tilesW * m + (double)tilesX * n, longer = std::max(m, n);
    const bool pieces = !vec && dw.kernel == F32_SPLIT && dx.kernel == F32_SPLIT;
    const double together = pieces ? 3.4 + (0.382 * tiles + 0.638 / 128 * work) / 256 + 0.83 * longer / 128 : 2.65 + (0.714 * tiles + 0.458 / 128 * work) / 256 + 0.64 * longer / 128;
    if (1.1 * together >= apart) return {false, false};
    // Long contractions that the calls apart would not give to 32 x 32 tiles: those cut them, or add fewer values in a row.  (With fewer
    // tiles than CUs nothing else is there while one adds up: 142 tiles of up to 2000 rows 16.0 -> 17.0 us.)
    return {true, tilesW + tilesX > 256 && ((dw.kernel != F32_SMALL && m > 512) || (dx.kernel != F32_SMALL && n > 512))};
}

int linear_bwd_f32_route(int m, int n, int k)
{
    const LinearBwdF32Plan p = linear_bwd_f32_plan(m, n, k, true, n % 4 == 0 && k % 4 == 0);
    return (p.together ? 1 : 0) + (p.levels ? 2 : 0);
}

// The gradients of an inner product as one launch, if that is what the sizes call for (*done): dW (n x k) += dY^T (n x m) X (m x k),
// db (n, or null) += column sums of dY, dX (m x k) = dY W (n x k) + beta dX.
hipError_t linear_bwd_f32_small(hipStream_t s, int m, int n, int k, const float* X, const float* W, const float* dY, float* dW, float* db, float* dX, float beta,
                                bool* done)
{
    *done = false;
    // what is written lies apart from everything else: the three calls, one after the other, may share memory
    const struct { const float* p; size_t n; bool out; } mem[] = {{dW, (size_t)n * k, true}, {dX, (size_t)m * k, true}, {db, db ? (size_t)n : 0, true},
                                                                 {X, (size_t)m * k, false}, {W, (size_t)n * k, false}, {dY, (size_t)m * n, false}};
    for (int i = 0; i < 3; i++)
        for (int j = i + 1; j < 6; j++)
            if (mem[i].n && mem[j].n && mem[i].p < mem[j].p + mem[j].n && mem[j].p < mem[i].p + mem[i].n) return hipSuccess;
    const bool vec = ((((uintptr_t)X | (uintptr_t)W | (uintptr_t)dY) & 15) == 0) && n % 4 == 0 && k % 4 == 0;
    const LinearBwdF32Plan plan = linear_bwd_f32_plan(m, n, k, db != nullptr, vec);
    if (!plan.together) return hipSuccess;
    const int tilesN = (k + 31) / 32, tilesW = (n + 31) / 32 * tilesN, tilesX = (m + 31) / 32 * tilesN;
    GemmF32Args w = {}, x = {};
    w.M = n; w.N = k; w.K = w.kChunk = m;
    w.A = dY; w.B = X; w.C = dW;
    w.lda = n; w.ldb = k; w.ldc = k;
    w.alpha = 1.f; w.beta = 1.f; w.parts = 1;
    w.vecC = k % 4 == 0 && ((uintptr_t)dW & 15) == 0;
    w.tilesM = (n + 31) / 32; w.tilesN = tilesN;
    x.M = m; x.N = k; x.K = x.kChunk = n;
    x.A = dY; x.B = W; x.C = dX;
    x.lda = n; x.ldb = k; x.ldc = k;
    x.alpha = 1.f; x.beta = beta; x.parts = 1;
    x.vecC = k % 4 == 0 && ((uintptr_t)dX & 15) == 0;
    x.tilesM = (m + 31) / 32; x.tilesN = tilesN;
    constexpr int lds = small_lds<4, 64>();
    typedef void (*Kernel)(GemmF32Args, GemmF32Args, float*, XcdRuns);
    static const Kernel kernels[2][2] = {{linear_bwd_f32_small_kernel<4, 64, false, false>, linear_bwd_f32_small_kernel<4, 64, true, false>},
                                         {linear_bwd_f32_small_kernel<4, 64, false, true>, linear_bwd_f32_small_kernel<4, 64, true, true>}};
    static const hipError_t attr = [] {
        hipError_t e = hipSuccess;
        for (int i = 0; i < 4 && e == hipSuccess; i++) e = hipFuncSetAttribute((const void*)kernels[i / 2][i % 2], hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        return e;
    }();
    if (attr != hipSuccess) return attr;
    int most;
    const bool wFirst = w.K >= x.K;
    const XcdRuns runs = xcd_runs(wFirst ? tilesW : tilesX, std::max(w.K, x.K), wFirst ? tilesX : tilesW, std::min(w.K, x.K), SMALL_TILE_COST, &most);
    const int grid = 8 * most;
    *done = true;
    hipLaunchKernelGGL(kernels[plan.levels][vec], grid, 256, lds, s, w, x, db, runs);
    return hipGetLastError();
}

}  // namespace mch
