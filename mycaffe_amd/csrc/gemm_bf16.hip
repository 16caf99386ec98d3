// 16-bit GEMM on the bf16 matrix cores (v_mfma_f32_16x16x32_bf16), any operand layout, fp32 accumulation, gfx950.
//
// WVM x WVN wavefronts of WM x WN MFMA tiles each cover (32 WVM WM) x (32 WVN WN) of C and walk K in stages of 64 that go
// from global memory straight into LDS (buffer loads to LDS: no staging registers, no writes to issue), two to four of them there,
// one barrier per stage.  At this matrix rate a tile is bound by what it moves: 128 x 128 needs 64 bytes per clock and CU from
// L2, all that L2 has; 256 x 256 half of that.  Large products therefore take 256 x 256 or 256 x 192 with eight
// wavefronts, one workgroup per CU, whichever leaves the shorter last round, small ones the tile that fills the chip.
//
// Large products run at the power limit (1.8 GHz at 8192 x 3072 x 6144), where what an instruction costs is time: products of 16 x 16 x 32
// alone, on normally distributed values, reach 2.0 PFLOP/s, those of 32 x 32 x 16 1.8 (2.4 and 2.5 on zeros), and a wavefront reads the same
// fragments for either (4096^3, A B^T 124 -> 119 us, A B 125.5 -> 123; 8000 x 3072 x 768 47.7 -> 46.5).  The sums are the same bits.  Where
// it is not power but the first product of a stage that is waited for, and operands are read transposed, the longer instruction stays, for
// which half as much has to arrive (time with the shorter one over time with the longer, means of ten sizes of 10^9 multiplications and
// more): four wavefronts alone on their CU (128 x 128 in three stages: A B 1.03, A^T B 1.09, A^T B^T 1.03), eight with 32 x 32 of C each (A^T B^T
// 1.03) and both operands read transposed by wavefronts with at most 32 x 64 (1.02).  All others are 0.95 - 1.01, and better where the
// contraction is short (4096 x 512 x 512 behind an attention launch: 0.8 us less).
//
//   * k at unit stride: LDS holds [row][64 k] without padding, the 16-byte piece c of row r at position c ^ ((r >> 1) & 7)
//     (sixteen consecutive rows read by a 128-bit access then fall on sixteen bank groups).
//   * row index at unit stride: LDS holds [k][row] as it is stored, the 32-row blocks of row k exchanged by a function of
//     k & 3 and their halves by k & 8, and the fragments are read with the transposing 64-bit access (ds_read_b64_tr_b16: lane i of a group of
//     sixteen receives column i of the 4 x 16 block whose rows four lanes each address).  Gradients need no operand turned
//     in memory first (57 of 570 us of an MLP's training step).
//   * The contraction may end anywhere a 16-byte chunk ends: chunks past the end get an offset outside the buffer, which
//     reads as zeros.
#include "gemm_common.h"

namespace mch {

struct GemmB16Args {
    int M, N, K;
    const bf16_t *A, *B;
    bf16_t* C;
    int lda, ldb;
    float alpha, beta;
    int tilesM, tilesN, parts, kChunk;
    float* part;              // kChunk < K: partial products, [part][M][N]
    bool vecC;
    const bf16_t* bias;
};

// sums of op(A)'s rows over some of the k, [part][tile column][M], behind the partial products
__device__ __forceinline__ float* b16_row_part(const GemmB16Args& g) { return g.part + (g.kChunk < g.K ? (size_t)g.parts * g.M * g.N : 0); }

// the bias of eight columns from c on (past the matrix the last one, never stored); all eight loads are under way at once
__device__ __forceinline__ void b16_bias8(const GemmB16Args& g, int c, float (&bias)[8])
{
    if (!g.bias) {
#pragma unroll
        for (int q = 0; q < 8; q++) bias[q] = 0.f;
        return;
    }
    bf16_t b[8];
#pragma unroll
    for (int q = 0; q < 8; q++) b[q] = g.bias[min(c + q, g.N - 1)];
#pragma unroll
    for (int q = 0; q < 8; q++) bias[q] = bf16_to_f32(b[q]);
}

// eight values of row r from column c on (inside the matrix up to N), alpha applied, and the bias, to C or through the heads
// epilogue, whose column c of row 0 is at col and row r rowAt further.  HEADS: 0 none, 1 without a rotation, 2 with (a rotation's code in the ends of a tile
// costs those that have none 1 us of 31: 3744 x 2880 x 960, 30.0 us, with a rotation 34.3, 42.1 with its tables read value by value and
// every row's place divided out)
template <int HEADS>
__device__ __forceinline__ void b16_store8(const GemmB16Args& g, const HeadsArg<(HEADS > 0)>& hp, int r, int c, const float (&bias)[8], bf16_t* col, size_t rowAt, float (&v)[8])
{
#pragma unroll
    for (int q = 0; q < 8; q++) v[q] += bias[q];
    if (g.vecC) {
        bf16_t* cp = g.C + (size_t)r * g.N + c;
        if constexpr (HEADS) cp = col + rowAt;
        if (!HEADS && g.beta != 0.f) {
            const u32x4 o = *(const u32x4*)cp;
            const uint32_t w[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
            for (int q = 0; q < 4; q++) {
                v[2 * q] += g.beta * __uint_as_float(w[q] << 16);
                v[2 * q + 1] += g.beta * __uint_as_float(w[q] & 0xffff0000u);
            }
        }
        u32x4 p;
        p.x = pack2_bf16(v[0], v[1]); p.y = pack2_bf16(v[2], v[3]); p.z = pack2_bf16(v[4], v[5]); p.w = pack2_bf16(v[6], v[7]);
        if constexpr (HEADS == 2) p = heads_rope_piece<bf16_t>(hp.he, r, c, p);
        *(u32x4*)cp = p;
        return;
    }
#pragma unroll
    for (int q = 0; q < 8; q += 2) {
        if (c + q >= g.N) continue;
        const bool two = c + q + 1 < g.N;
        if constexpr (HEADS) {
            float o0 = bf16_to_f32(f32_to_bf16(v[q])), o1 = bf16_to_f32(f32_to_bf16(v[q + 1]));   // as the storage type holds them
            if constexpr (HEADS == 2)
                if (hp.he.fcos && c + q < 2 * hp.he.H * hp.he.hs) {
                    const size_t ti = heads_rope_at(hp.he, r, c + q);
                    heads_rope_pair(hp.he.fcos[ti], hp.he.fsin[ti], o0, o1);
                }
            *heads_dst<bf16_t>(hp.he, r, c + q) = f32_to_bf16(o0);
            if (two) *heads_dst<bf16_t>(hp.he, r, c + q + 1) = f32_to_bf16(o1);
        } else {
            bf16_t* cp = g.C + (size_t)r * g.N + c + q;
            cp[0] = f32_to_bf16(v[q] + (g.beta != 0.f ? g.beta * bf16_to_f32(cp[0]) : 0.f));
            if (two) cp[1] = f32_to_bf16(v[q + 1] + (g.beta != 0.f ? g.beta * bf16_to_f32(cp[1]) : 0.f));
        }
    }
}

// Epilogues of the prompt pass of the Llama engine (fp32 results of 16-bit operands; llama2_ext.hip), which save the
// round trip of the product through memory and the kernel that would read it back:
//   1, SwiGLU of the stacked W1 | W3 product.  Tile column c multiplies weight row (c & 1) hid + c / 2, so that a
//     lane's register quad holds (w1 x, w3 x) of two consecutive hidden units j: out[j] = silu(w1 x) (w3 x), stored as
//     bf16 (rows of hid), or as the bf16 nearest to it followed, hid further on, by the bf16 nearest to the remainder
//     (rows of 2 hid: the operand form of k_gemm_bf16_f32's split product).
//   2, rotation and scatter of the stacked Wq | Wk | Wv product (row = sequence b, position p): q and k rotated at p
//     (adjacent pairs, the decode kernel's arithmetic), q / k / v written as (B, H, P, hs) head tensors - fp32 or bf16,
//     every key / value head repeated for the query heads that share it - and the rotated key and the value appended to
//     the caches [b][p][kvd] (fp32 or bf16; the head tensors then carry the values the cache holds).
struct PromptEpilogue {
    void* out; int hid; int split;                                   // 1
    void* q; void* k; void* v; void* kc; void* vc;                   // 2
    const float* fcos; const float* fsin;
    int P, H, kvH, hs, seqLen, heads16, cache16, kvMul;
    float invP, invHs;
    int kB;                                                          // all: of B, which is walked again from there on (K or K / 2)
};
// the argument behind a product's: nothing, the heads epilogue's (1, 2), the prompt pass's (3: none of its epilogues, 4, 5: 1, 2)
struct PromptArg { PromptEpilogue pe; };
template <int END> using B16Arg = std::conditional_t<(END >= 3), PromptArg, HeadsArg<(END > 0)>>;
__device__ __forceinline__ uint32_t pe_pack(float a, float b) { return pack2_bf16(a, b); }
__device__ __forceinline__ float pe_round(float a) { return bf16_to_f32(f32_to_bf16(a)); }
// four consecutive values to a tensor of fp32 or bf16
__device__ __forceinline__ void pe_store4(void* base, size_t idx, int is16, const float (&v)[4])
{
    if (is16) *(uint2*)((bf16_t*)base + idx) = make_uint2(pe_pack(v[0], v[1]), pe_pack(v[2], v[3]));
    else *(float4*)((float*)base + idx) = make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ void prompt_epilogue_swiglu(const PromptEpilogue& pe, int r, int c, const float (&a)[4])
{
    const int j = c >> 1;   // c is a multiple of 4: hidden units j, j + 1
    float o[2];
#pragma unroll
    for (int q = 0; q < 2; q++) o[q] = a[2 * q] * (1.0f / (1.0f + expf(-a[2 * q]))) * a[2 * q + 1];
    bf16_t* row = (bf16_t*)pe.out + (size_t)r * (pe.split ? 2 : 1) * pe.hid;
    *(uint32_t*)(row + j) = pe_pack(o[0], o[1]);
    if (pe.split) *(uint32_t*)(row + pe.hid + j) = pe_pack(o[0] - pe_round(o[0]), o[1] - pe_round(o[1]));
}
// x / d for 0 <= x < 2^24, d > 0, through the reciprocal (an integer division is some forty instructions)
__device__ __forceinline__ int pe_div(int x, int d, float inv)
{
    int q = (int)((float)x * inv);
    if ((q + 1) * d <= x) q++;
    if (q * d > x) q--;
    return q;
}
__device__ __forceinline__ void prompt_epilogue_rope(const PromptEpilogue& pe, int r, int c, const float (&a)[4])
{
    const int dim = pe.H * pe.hs, kvd = pe.kvH * pe.hs, kvMul = pe.kvMul, half = pe.hs >> 1;
    const int b = pe_div(r, pe.P, pe.invP), p = r - b * pe.P;
    float o[4] = {a[0], a[1], a[2], a[3]};
    const int which = c < dim ? 0 : c < dim + kvd ? 1 : 2;
    const int cc = which == 0 ? c : which == 1 ? c - dim : c - dim - kvd;
    const int h = pe_div(cc, pe.hs, pe.invHs), d = cc - h * pe.hs;
    if (which < 2) {
        const float2 cs = *(const float2*)(pe.fcos + (size_t)p * half + (d >> 1)), sn = *(const float2*)(pe.fsin + (size_t)p * half + (d >> 1));
        o[0] = a[0] * cs.x - a[1] * sn.x; o[1] = a[0] * sn.x + a[1] * cs.x;
        o[2] = a[2] * cs.y - a[3] * sn.y; o[3] = a[2] * sn.y + a[3] * cs.y;
    }
    if (which == 0) {
        pe_store4(pe.q, (((size_t)b * pe.H + h) * pe.P + p) * pe.hs + d, pe.heads16, o);
        return;
    }
    if (pe.cache16) {
#pragma unroll
        for (int q = 0; q < 4; q++) o[q] = pe_round(o[q]);   // the pass attends over the values the cache holds
    }
    pe_store4(which == 1 ? pe.kc : pe.vc, ((size_t)b * pe.seqLen + p) * kvd + cc, pe.cache16, o);
    for (int g = 0; g < kvMul; g++)
        pe_store4(which == 1 ? pe.k : pe.v, (((size_t)b * pe.H + h * kvMul + g) * pe.P + p) * pe.hs + d, pe.heads16, o);
}

// eight values of row r from column c on to an fp32 matrix, beta C added
__device__ __forceinline__ void prompt_store8(const GemmB16Args& g, int r, int c, const float (&v)[8])
{
    float* cp = (float*)g.C + (size_t)r * g.N + c;
#pragma unroll
    for (int q = 0; q < 8; q += 4) {
        if (g.vecC && c + q < g.N) {
            float4 o = make_float4(v[q], v[q + 1], v[q + 2], v[q + 3]);
            if (g.beta != 0.f) {
                const float4 old = *(const float4*)(cp + q);
                o.x += g.beta * old.x; o.y += g.beta * old.y; o.z += g.beta * old.z; o.w += g.beta * old.w;
            }
            *(float4*)(cp + q) = o;
        } else {
#pragma unroll
            for (int e = q; e < q + 4; e++)
                if (c + e < g.N) cp[e] = v[e] + (g.beta != 0.f ? g.beta * cp[e] : 0.f);
        }
    }
}

// tile `item` of a product.  SUMS: the tiles of a row of tiles also add up the rows of op(A), each the stages that are its turn, from
// the fragments it multiplies: the bias gradient beside a weight gradient (8000 x 3072, 6.2 to 12.8 us and a launch of 5 on their own).
template <int WVM, int WVN, int WM, int WN, int S, bool AK, bool BKC, int HEADS, bool SUMS = false>
__device__ __forceinline__ void b16_tile(const GemmB16Args& g, const B16Arg<HEADS>& hp, int item)
{
    constexpr int NT = 64 * WVM * WVN, BM = 32 * WVM * WM, BN = 32 * WVN * WN, BK = 64;
    constexpr bool PROMPT = HEADS >= 3;
    constexpr bool WAITS = (WVM * WVN == 4 && WM * WN == 4 && S == 3 && !(AK && BKC)) || (WVM * WVN == 8 && WM * WN == 1 && !AK) || (!AK && !BKC && WM * WN <= 2);
    constexpr int F = WAITS ? 32 : 16, KM = 512 / F, KS = BK / KM, TM = 32 * WM / F, TN = 32 * WN / F;   // rows and k of a product; products' tiles of a wavefront
    constexpr int PA = BM * 8 / NT, PB = BN * 8 / NT;               // 16-byte chunks per thread and stage
    constexpr int STAGE = (BM + BN) * BK;                           // elements of one stage: A's part, then B's
    constexpr int NMF = TM * TN;
    static_assert(PA * NT == BM * 8 && PB * NT == BN * 8, "whole chunks per thread");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    bf16_t* smem = reinterpret_cast<bf16_t*>(smem_raw);
    constexpr bool ENDS_IN_HEADS = HEADS == 1 || HEADS == 2;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tiles = g.tilesM * g.tilesN;
    const int part = item / tiles, tile = item - part * tiles;
    constexpr int GROUP = 4;   // tile rows per group, walked down first: few rows of A and columns of B in flight per XCD
    const int group = tile / (GROUP * g.tilesN), inGroup = tile - group * GROUP * g.tilesN;
    const int groupRows = min(GROUP, g.tilesM - group * GROUP);
    const int M = g.M, N = g.N;
    const int m0 = (group * GROUP + inGroup % groupRows) * BM, n0 = (inGroup / groupRows) * BN;
    const bool split = g.kChunk < g.K;
    const int kBegin = split ? part * g.kChunk : 0, kEnd = min(g.K, kBegin + g.kChunk);
    const int wm = (wave / WVN) * (32 * WM), wn = (wave % WVN) * (32 * WN);

    // The buffer resource of an operand begins at the tile, and where the row index is at unit stride at the stage, so that
    // operands of any size are reached with 32-bit byte offsets (gemm_b16_takes).  Offsets of this thread's chunks from there;
    // rows past the edge are clamped and never stored.
    constexpr uint32_t OUTSIDE = 0x80000000u;
    const bf16_t* baseA = g.A + (AK ? (size_t)m0 * g.lda : (size_t)m0);
    const bf16_t* baseB = g.B + (BKC ? (size_t)n0 * g.ldb : (size_t)n0);
    // (16 x 16: groups of lanes eight k apart read the same sixteen rows, from the other half of their 32)
    auto place = [](auto rowb, int k) { return block_swizzle<decltype(rowb)::value>(k) + (F == 16 ? ((k >> 3) & 1) * 2 : 0); };
    uint32_t va[PA], vb[PB];
#pragma unroll
    for (int p = 0; p < PA; p++) {
        const int e = p * NT + tid;
        if (AK) va[p] = ((uint32_t)min(e / 8, M - 1 - m0) * (uint32_t)g.lda + ((e & 7) ^ ((e >> 4) & 7)) * 8) * 2;
        else va[p] = ((uint32_t)(e / (BM / 8)) * (uint32_t)g.lda + min(((e % (BM / 8)) ^ place(std::integral_constant<int, BM * 2>(), e / (BM / 8))) * 8, M - 8 - m0)) * 2;
    }
#pragma unroll
    for (int p = 0; p < PB; p++) {
        const int e = p * NT + tid;
        if (BKC) vb[p] = ((uint32_t)min(e / 8, N - 1 - n0) * (uint32_t)g.ldb + ((e & 7) ^ ((e >> 4) & 7)) * 8) * 2;
        else vb[p] = ((uint32_t)(e / (BN / 8)) * (uint32_t)g.ldb + min(((e % (BN / 8)) ^ place(std::integral_constant<int, BN * 2>(), e / (BN / 8))) * 8, N - 8 - n0)) * 2;
    }
    // a prompt product's B by its addresses: pairs of rows of a stacked matrix lie far apart
    [[maybe_unused]] const bf16_t* pb64[PB];
    if constexpr (PROMPT) {
#pragma unroll
        for (int p = 0; p < PB; p++) {
            const int e = p * NT + tid, c = min(n0 + e / 8, N - 1);
            pb64[p] = g.B + (size_t)(HEADS == 4 ? (c & 1) * hp.pe.hid + (c >> 1) : c) * g.ldb + ((e & 7) ^ ((e >> 4) & 7)) * 8;
        }
    }
    auto resource = [](const void* base) { return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)(OUTSIDE - 16), 0x00020000); };
    const __amdgpu_buffer_rsrc_t rsA = resource(baseA), rsB = resource(baseB);
    // where resources begin at stages: the stage that is fetched next, and the way to the one after it (0 from the last on).
    // Added up and not multiplied out: the scalar instructions of a stage show (gradients at 1000 x 32000 x 768: 0.5 %).
    const char *stageA = (const char*)(baseA + (size_t)kBegin * g.lda), *stageB = (const char*)(baseB + (size_t)kBegin * g.ldb);
    long long stepA = (long long)(BK * sizeof(bf16_t)) * g.lda, stepB = (long long)(BK * sizeof(bf16_t)) * g.ldb;
    auto advance = [&]() {
        if (!AK) stageA += stepA;
        if (!BKC) stageB += stepB;
    };
    // before a stage is fetched that ends the contraction or lies past it: the chunks past the end
    auto lastStage = [&](int k0) {
        asm volatile("" ::: "memory");   // a branch, not a select in every stage
        stepA = stepB = 0;
#pragma unroll
        for (int p = 0; p < PA; p++) {
            const int e = p * NT + tid;
            if (k0 + (AK ? ((e & 7) ^ ((e >> 4) & 7)) * 8 : e / (BM / 8)) >= kEnd) va[p] = OUTSIDE;
        }
#pragma unroll
        for (int p = 0; p < PB; p++) {
            const int e = p * NT + tid;
            if (k0 + (BKC ? ((e & 7) ^ ((e >> 4) & 7)) * 8 : e / (BN / 8)) >= kEnd) vb[p] = OUTSIDE;
        }
    };
    // fetch p of a stage: this wavefront fills the 1 KB from chunk p NT + 64 wave on, lane i its i-th chunk
    auto fetch = [&](int p, int k0, bf16_t* stage) {
        if (p < PA) {
            bf16_t* to = stage + (p * NT + wave * 64) * 8;
            if (AK) lds_fetch<16>(rsA, to, va[p], k0 * 2);
            else lds_fetch<16>(resource(stageA), to, va[p], 0);
        } else {
            bf16_t* to = stage + BM * BK + ((p - PA) * NT + wave * 64) * 8;
            if constexpr (PROMPT) __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(pb64[p - PA] + (k0 >= hp.pe.kB ? k0 - hp.pe.kB : k0)), LDS3(to), 16, 0, 0);
            else if (BKC) lds_fetch<16>(rsB, to, vb[p - PA], k0 * 2);
            else lds_fetch<16>(resource(stageB), to, vb[p - PA], 0);
        }
    };

    typedef std::conditional_t<F == 32, floatx16, floatx4> Sums;
    Sums acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int v = 0; v < F * F / 64; v++) acc[i][j][v] = 0.f;

    // fragments: lane l holds row l % F, k = 8 (l / F) .. + 7 of a k-step of KM
    const int fr = lane & (F - 1), kp = lane / F;
    int koff[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) koff[ks] = ((KM / 8 * ks + kp) ^ ((fr >> 1) & 7)) * 8;
    // transposing reads: lane i of a group of sixteen addresses row k = 8 kp + i / 4 (and + 4) of the k-step, columns
    // 16 (group & 1) (F = 32) + 4 (i % 4) .. + 3; k % 4 is the same for both reads, so the exchange of the 32-row blocks is one
    // constant per lane.  Byte offsets of this lane's first element of every block of rows:
    const int tk = 8 * kp + ((lane & 15) >> 2), tcol = (F == 32 ? ((lane >> 4) & 1) * 16 : 0) + (lane & 3) * 4;
    uint32_t ta[TM], tb[TN];
#pragma unroll
    for (int t = 0; t < TM; t++) ta[t] = (uint32_t)(tk * BM + ((wm + t * F) ^ (place(std::integral_constant<int, BM * 2>(), tk) * 8)) + tcol) * 2;
#pragma unroll
    for (int t = 0; t < TN; t++) tb[t] = (uint32_t)(BM * BK + tk * BN + ((wn + t * F) ^ (place(std::integral_constant<int, BN * 2>(), tk) * 8)) + tcol) * 2;
    auto fragA = [&](const bf16_t* pa, uint32_t stageAddr, int t, int ks, TrFragment& o) {
        if (AK) o.w = *(const u32x4*)(pa + (wm + t * F + fr) * BK + koff[ks]);
        else tr_read<BM * 2>(stageAddr + ta[t], ks * KM * (BM * 2), o);
    };
    auto fragB = [&](const bf16_t* pb, uint32_t stageAddr, int t, int ks, TrFragment& o) {
        if (BKC) o.w = *(const u32x4*)(pb + (wn + t * F + fr) * BK + koff[ks]);
        else tr_read<BN * 2>(stageAddr + tb[t], ks * KM * (BN * 2), o);
    };
    auto multiply = [&](const TrFragment& x, const TrFragment& y, Sums& o) {
        if constexpr (F == 32) o = BigTraits<bf16_t>::mma(x.w, y.w, o);
        else o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)&x.w, *(const bf16x8*)&y.w, o, 0, 0, 0);
    };

    // S stages in LDS: one is read, the S - 1 after it are fetched
    const int nk = (kEnd - kBegin + BK - 1) / BK;
#pragma unroll
    for (int u = 0; u < S - 1; u++) {
        if (u > 0) advance();
        if (u + 1 >= nk) lastStage(kBegin + u * BK);
#pragma unroll
        for (int p = 0; p < PA + PB; p++) fetch(p, PROMPT ? kBegin + min(u, nk - 1) * BK : kBegin + u * BK, smem + u * STAGE);
        asm volatile("" ::: "memory");
    }
    // the oldest of S - 1 stages under way has landed, of this wavefront and then of all
    auto landed = [&]() {
        if constexpr (S == 2) {
            __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
            __syncthreads();
        } else {
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((S - 2) * (PA + PB)) : "memory");
        }
    };
    landed();
    const uint32_t smemAddr = (uint32_t)(uintptr_t)LDS3(smem);
    TrFragment a[2][TM], b[2][TN];
    [[maybe_unused]] float sums[TM][8];
    [[maybe_unused]] int turn = n0 / BN;   // stages until this tile's next
    if constexpr (SUMS) {
#pragma unroll
        for (int t = 0; t < TM; t++)
#pragma unroll
            for (int e = 0; e < 8; e++) sums[t][e] = 0.f;
    }
    int slot = 0;
    for (int kt = 0; kt < nk; kt++) {
        const bf16_t* pa = smem + slot * STAGE;
        const bf16_t* pb = pa + BM * BK;
        bf16_t* next = smem + (slot == 0 ? S - 1 : slot - 1) * STAGE;   // read during stage kt - 1; free since the barrier that ended it
        // past the end two stages fetch the last one again, never read, and more of them nothing
        const int k1 = kBegin + (S == 2 || PROMPT ? min(kt + S - 1, nk - 1) : kt + S - 1) * BK;
        advance();
        if (S == 2 ? kt + 2 == nk : kt + S >= nk) lastStage(k1);
        const uint32_t stageAddr = smemAddr + slot * STAGE * 2;
#pragma unroll
        for (int t = 0; t < TM; t++) fragA(pa, stageAddr, t, 0, a[0][t]);
#pragma unroll
        for (int t = 0; t < TN; t++) fragB(pb, stageAddr, t, 0, b[0][t]);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int cur = ks & 1, nxt = cur ^ 1;
            // what the transposing reads of this k-step's fragments brought, by now long issued
#pragma unroll
            for (int t = 0; t < TM; t++)
                if (!AK) tr_wait(a[cur][t]);
#pragma unroll
            for (int t = 0; t < TN; t++)
                if (!BKC) tr_wait(b[cur][t]);
            if constexpr (SUMS) {
                if (wn == 0 && turn == 0) {
#pragma unroll
                    for (int t = 0; t < TM; t++)
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            sums[t][2 * e] += __uint_as_float(a[cur][t].w[e] << 16);
                            sums[t][2 * e + 1] += __uint_as_float(a[cur][t].w[e] & 0xffff0000u);
                        }
                }
            }
            // in issue order: a product, the fragments of the next k-step spread over the products, and from the first
            // product on one fetch of the next stage each
            constexpr int RF = (TM + TN + NMF - 1) / NMF * (AK && BKC ? 1 : 2);
            constexpr int FE = (PA + PB + (KS - 1) * NMF - 1) / ((KS - 1) * NMF);   // fetches per product
#pragma unroll
            for (int q = 0; q < NMF; q++) {
                const int i = q / TN, j = q % TN;
                multiply(b[cur][j], a[cur][i], acc[i][j]);
                if (ks + 1 < KS) {
#pragma unroll
                    for (int r = q * RF; r < (q + 1) * RF; r++) {
                        if (r < TM) fragA(pa, stageAddr, r, ks + 1, a[nxt][r]);
                        else if (r < TM + TN) fragB(pb, stageAddr, r - TM, ks + 1, b[nxt][r - TM]);
                    }
                }
#pragma unroll
                for (int f = (ks * NMF + q) * FE; f < (ks * NMF + q + 1) * FE; f++)
                    if (f < PA + PB) fetch(f, k1, next);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if constexpr (SUMS) turn = turn == 0 ? g.tilesN - 1 : turn - 1;
        slot = slot == S - 1 ? 0 : slot + 1;
        landed();
    }
    if constexpr (S > 2) {   // what was fetched past the end
        __builtin_amdgcn_s_waitcnt(0x0f70);
        __syncthreads();
    }
    if constexpr (SUMS) {
        if (wn == 0) {
#pragma unroll
            for (int t = 0; t < TM; t++) {
                float v = ((sums[t][0] + sums[t][1]) + (sums[t][2] + sums[t][3])) + ((sums[t][4] + sums[t][5]) + (sums[t][6] + sums[t][7]));
                v += __shfl_xor(v, 32);
                if (F == 16) v += __shfl_xor(v, 16);
                const int r = m0 + wm + t * F + fr;
                if (kp == 0 && r < M) b16_row_part(g)[(size_t)(part * g.tilesN + n0 / BN) * M + r] = v;
            }
        }
    }

    // The products are the transposed tiles: a lane owns row lane % F, register v is column 4 (lane / F) + v (F = 32:
    // 8 (v / 4) + 4 (lane / 32) + v % 4).
    // Each wavefront passes 32 rows by CH tiles of columns at a time through its own slice of LDS (free after the last
    // barrier; operations of one wavefront complete in order) and the lanes walk the rows eight columns each.
    constexpr int CH = WN % 2 == 0 ? 2 : WN, CW = 32 * CH, LDC = CW + 4, LPR = CW / 8, RPI = 64 / LPR, NIT = (32 + RPI - 1) / RPI;
    float* cs = reinterpret_cast<float*>(smem_raw) + wave * 32 * LDC;
    const int rr = lane / LPR, cc = (lane % LPR) * 8, fg = kp * 4;
#pragma unroll
    for (int i = 0; i < WM; i++)
#pragma unroll
        for (int c0 = 0; c0 < WN; c0 += CH) {
            // 32 rows of CH tiles of 32 columns: the products' tiles in them, four columns of a row at a time
#pragma unroll
            for (int x = 0; x < 32 / F; x++)
#pragma unroll
                for (int j = 0; j < CW / F; j++)
#pragma unroll
                    for (int q = 0; q < F * F / 256; q++) {
                        const Sums& o = acc[32 / F * i + x][32 / F * c0 + j];
                        *(float4*)(cs + (x * F + fr) * LDC + j * F + 8 * q + fg) = make_float4(g.alpha * o[4 * q], g.alpha * o[4 * q + 1], g.alpha * o[4 * q + 2], g.alpha * o[4 * q + 3]);
                    }
            // a lane keeps its columns while it walks the rows
            const int c = n0 + wn + c0 * 32 + cc;
            float bias[8];
            bf16_t* col = nullptr;
            if (!PROMPT && !split && c < N) {
                b16_bias8(g, c, bias);
                if constexpr (ENDS_IN_HEADS) col = heads_col<bf16_t>(hp.he, c);
            }
            // the rows' places: added up, not divided out for each
            size_t nextAt = 0;
            int t = 0;
            if constexpr (ENDS_IN_HEADS) nextAt = heads_row(hp.he, m0 + wm + i * 32 + rr, t);
#pragma unroll 2
            for (int it = 0; it < NIT; it++) {
                const int row = it * RPI + rr, r = m0 + wm + i * 32 + row;
                const size_t rowAt = nextAt;
                if constexpr (ENDS_IN_HEADS) {
                    nextAt += (size_t)(RPI * hp.he.hs);
                    for (t += RPI; t >= hp.he.T; t -= hp.he.T) nextAt += hp.he.perBatch - (unsigned long long)(uint32_t)hp.he.T * (uint32_t)hp.he.hs;
                }
                if (rr >= RPI || row >= 32 || r >= M || c >= N) continue;
                const float4 t0 = *(const float4*)(cs + row * LDC + cc), t1 = *(const float4*)(cs + row * LDC + cc + 4);
                float v[8] = {t0.x, t0.y, t0.z, t0.w, t1.x, t1.y, t1.z, t1.w};
                if constexpr (PROMPT) {
                    const float lo[4] = {v[0], v[1], v[2], v[3]}, hi[4] = {v[4], v[5], v[6], v[7]};   // of a multiple of four columns
                    if constexpr (HEADS == 3) prompt_store8(g, r, c, v);
                    else if constexpr (HEADS == 4) {
                        prompt_epilogue_swiglu(hp.pe, r, c, lo);
                        if (c + 4 < N) prompt_epilogue_swiglu(hp.pe, r, c + 4, hi);
                    } else {
                        prompt_epilogue_rope(hp.pe, r, c, lo);
                        if (c + 4 < N) prompt_epilogue_rope(hp.pe, r, c + 4, hi);
                    }
                } else if (split) {
                    float* cp = g.part + ((size_t)part * M + r) * N + c;
                    if (g.vecC) {
                        *(float4*)cp = t0;
                        *(float4*)(cp + 4) = t1;
                    } else {
#pragma unroll
                        for (int q = 0; q < 8; q++)
                            if (c + q < N) cp[q] = v[q];
                    }
                } else {
                    if constexpr (!PROMPT) b16_store8<HEADS>(g, hp, r, c, bias, col, rowAt, v);
                }
            }
        }
}

// each XCD (workgroup index mod 8) takes a contiguous run of the tiles
__device__ __forceinline__ int b16_xcd_item(int total) { return (int)(blockIdx.x % 8) * ((total + 7) / 8) + (int)(blockIdx.x / 8); }

template <int WVM, int WVN, int WM, int WN, int S, int OCC, bool AK, bool BKC, int HEADS, bool SUMS>
__global__ __launch_bounds__(64 * WVM * WVN, OCC) void gemm_b16_kernel(GemmB16Args g, B16Arg<HEADS> hp)
{
    const int total = g.tilesM * g.tilesN * g.parts, item = b16_xcd_item(total);
    if (item >= total) return;
    b16_tile<WVM, WVN, WM, WN, S, AK, BKC, HEADS, SUMS>(g, hp, item);
}

// Up to three products with heads epilogues as one launch: the projections of a multi-head attention layer.  One by one each is less
// than two rounds of the chip with its own first fetches and last stores (4096 and twice 8192 rows, 512 to 512: 9.4 + 12.3 + 11.9 us, as one launch 21.6).
struct GemmB16Group { GemmB16Args g[3]; HeadsArg<true> h[3]; int first[4]; };   // first: of the tiles of all, of each; then their number
template <int WVM, int WVN, int WM, int WN, int S, int OCC>
__global__ __launch_bounds__(64 * WVM * WVN, OCC) void gemm_b16_group_kernel(GemmB16Group grp)
{
    const int item = b16_xcd_item(grp.first[3]);
    if (item >= grp.first[3]) return;
    const int p = item >= grp.first[2] ? 2 : item >= grp.first[1] ? 1 : 0;
    b16_tile<WVM, WVN, WM, WN, S, true, true, 1>(grp.g[p], grp.h[p], item - grp.first[p]);
}

// ---------------------------------------------------------------------------
// Up to 32 rows against the rows of B (a decode step's projections).  Such a product reads B once and does little else.  The lanes of
// a wavefront take the fragments of 16 rows of B straight to registers, a stage of k at a time with the next one on its way; the
// rows of A, which every workgroup reads, come through LDS, because as fragments from memory they cost what the same bytes of B do.
// The k are dealt to NW wavefronts, each with stages of its own (nothing but its own fetches to wait for), whose sums meet in LDS.
// Microseconds with B not in any cache, before (tiles in parts of the contraction, and a launch that adds them up) and now:
// 8 x 12288 x 4096 24.2, 20.6 (4.9 TB/s); 8 x 4096 x 4096 15.4, 8.8; 32 x 12288 x 4096 25.2, 23.5; 32 x 4096 x 4096 15.6, 11.7;
// 8 x 2304 x 768 8.3, 3.7; 8 x 512 x 512 6.2, 3.3.  What is left over the reading of B is the launch's beginning and end.
template <int MT, int NT, int NW, int S, int HEADS>
__global__ __launch_bounds__(64 * NW) void gemm_b16_rows_kernel(GemmB16Args g, HeadsArg<(HEADS > 0)> hp)
{
    constexpr int KW = 128 / MT, KS = KW / 32, P = KW / 8;   // k, products and 16-byte pieces of a row, of a stage
    constexpr int STAGE = 16 * MT * KW, DA = STAGE / 512;    // elements of A in a stage, fetches
    constexpr int LDC = 16 * NT + 4;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    bf16_t* ring = reinterpret_cast<bf16_t*>(smem_raw) + wave * S * STAGE;
    const int r = lane & 15, kq = lane >> 4, n0 = (int)blockIdx.x * 16 * NT;
    const int row = tid / (2 * NT), c = n0 + (tid % (2 * NT)) * 8;   // of the eight results this thread adds up
    float bias[8];
    b16_bias8(g, c, bias);   // on its way before the operands
    // [row][k] in LDS, piece c of row r at c ^ swap(r): sixteen rows read at one piece fall on sixteen bank groups
    auto swap = [](int row) { return P == 16 ? row & 15 : (row >> 1) & 7; };
    constexpr uint32_t OUTSIDE = 0x80000000u;   // fetched from there: zeros
    const __amdgpu_buffer_rsrc_t rsA = __builtin_amdgcn_make_buffer_rsrc((void*)g.A, 0, (int)(OUTSIDE - 16), 0x00020000);
    uint32_t va[DA];
    int ka[DA];
#pragma unroll
    for (int p = 0; p < DA; p++) {
        const int ra = (p * 64 + lane) / P;
        ka[p] = ((lane % P) ^ swap(ra)) * 8;
        va[p] = ra < g.M ? ((uint32_t)ra * (uint32_t)g.lda + ka[p]) * 2 : OUTSIDE;
    }
    // lane l holds row l % 16, k = 8 (l / 16) .. + 7 of a product's 32; rows of B past the edge are clamped and never stored
    const bf16_t* pb[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) pb[j] = g.B + (size_t)min(n0 + j * 16 + r, g.N - 1) * g.ldb + kq * 8;
    struct Stage { u32x4 b[NT][KS]; };
    auto fetch = [&](Stage& st, int k, int slot) {
#pragma unroll
        for (int p = 0; p < DA; p++) lds_fetch<16>(rsA, ring + slot * STAGE + p * 512, va[p], k * 2);
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int i = 0; i < KS; i++) st.b[j][i] = *(const u32x4*)(pb[j] + k + i * 32);
        asm volatile("" ::: "memory");   // stage after stage
    };
    floatx4 acc[MT][NT];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[t][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const Stage& st, int slot) {
        const bf16_t* pa = ring + slot * STAGE;
#pragma unroll
        for (int i = 0; i < KS; i++)
#pragma unroll
            for (int t = 0; t < MT; t++) {
                const u32x4 a = *(const u32x4*)(pa + (t * 16 + r) * KW + ((4 * i + kq) ^ swap(t * 16 + r)) * 8);
#pragma unroll
                for (int j = 0; j < NT; j++)
                    acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)&st.b[j][i], *(const bf16x8*)&a, acc[t][j], 0, 0, 0);
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the slot has been read: it may be fetched into
    };
    // all but the latest S - 1 stages' fetches have landed; and all of them
    auto waitBefore = [&]() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"((S - 1) * (DA + NT * KS)) : "memory"); };
    auto waitAll = [&]() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
    // stages wave, wave + NW, .. are this wavefront's
    const int whole = g.K / KW;
    int left = (whole - wave + NW - 1) / NW, k = wave * KW;
    Stage st[S];
#pragma unroll
    for (int u = 0; u < S - 1; u++)
        if (left > u) fetch(st[u], k + u * NW * KW, u);
    for (; left >= 2 * S - 1; left -= S, k += S * NW * KW)
#pragma unroll
        for (int u = 0; u < S; u++) {
            fetch(st[(u + S - 1) % S], k + (u + S - 1) * NW * KW, (u + S - 1) % S);
            waitBefore();
            multiply(st[u], u);
        }
#pragma unroll
    for (int u = 0; u < 2 * S - 2; u++)
        if (left > u) {
            if (left > u + S - 1) {
                fetch(st[(u + S - 1) % S], k + (u + S - 1) * NW * KW, (u + S - 1) % S);
                waitBefore();
            } else waitAll();
            multiply(st[u % S], u % S);
        }
    if (whole * KW < g.K && whole % NW == wave) {   // the rest, whole 16-byte pieces
        k = whole * KW;
#pragma unroll
        for (int p = 0; p < DA; p++) lds_fetch<16>(rsA, ring + p * 512, k + ka[p] < g.K ? va[p] : OUTSIDE, k * 2);
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int i = 0; i < KS; i++) st[0].b[j][i] = k + i * 32 + kq * 8 < g.K ? *(const u32x4*)(pb[j] + k + i * 32) : u32x4{0, 0, 0, 0};
        waitAll();
        multiply(st[0], 0);
    }
    // the products are the transposed tiles: a lane owns row l % 16, columns 4 (l / 16) .. + 3
    constexpr int SLICE = S * STAGE / 2;   // floats from one wavefront's stages to the next's
    float* red = reinterpret_cast<float*>(smem_raw);
    static_assert(16 * MT * LDC <= SLICE, "the sums fit in place of the stages");
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int j = 0; j < NT; j++) *(floatx4*)(red + wave * SLICE + (t * 16 + r) * LDC + j * 16 + kq * 4) = acc[t][j];
    __syncthreads();
    if (row >= min(16 * MT, g.M) || c >= g.N) return;
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; w++) {
        const float* p = red + w * SLICE + row * LDC + c - n0;
        const floatx4 x = *(const floatx4*)p, y = *(const floatx4*)(p + 4);
#pragma unroll
        for (int q = 0; q < 4; q++) { v[q] += x[q]; v[4 + q] += y[q]; }
    }
#pragma unroll
    for (int q = 0; q < 8; q++) v[q] *= g.alpha;
    bf16_t* col = nullptr;
    size_t rowAt = 0;
    if constexpr (HEADS) { col = heads_col<bf16_t>(hp.he, c); rowAt = heads_row(hp.he, row); }
    b16_store8<HEADS>(g, hp, row, c, bias, col, rowAt, v);
}

// sum over the S partial products in their order, then as b16_store8; the first rowBlocks workgroups add the partial row sums to rowSum
template <int HEADS>
__global__ __launch_bounds__(256) void gemm_b16_sum_kernel(GemmB16Args g, HeadsArg<(HEADS > 0)> hp, int S, int rowBlocks, bf16_t* rowSum)
{
    const int block = (int)blockIdx.x - rowBlocks;
    if (block < 0) {
        const int r = (int)blockIdx.x * 256 + threadIdx.x;
        if (r >= g.M) return;
        rowSum[r] = f32_to_bf16(bf16_to_f32(rowSum[r]) + sum_partials(b16_row_part(g) + r, g.parts * g.tilesN, g.M));
        return;
    }
    const int oct = (g.N + 7) / 8;
    const size_t mn = (size_t)g.M * g.N;
    for (size_t e = (size_t)block * 256 + threadIdx.x; e < (size_t)g.M * oct; e += (size_t)256 * (gridDim.x - rowBlocks)) {
        const int r = (int)(e / oct), c = (int)(e % oct) * 8;
        const float* p = g.part + (size_t)r * g.N + c;
        float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        for (int z = 0; z < S; z++) {
            if (g.vecC) {
                const float4 a = *(const float4*)(p + z * mn), b = *(const float4*)(p + z * mn + 4);
                v[0] += a.x; v[1] += a.y; v[2] += a.z; v[3] += a.w; v[4] += b.x; v[5] += b.y; v[6] += b.z; v[7] += b.w;
            } else {
#pragma unroll
                for (int q = 0; q < 8; q++)
                    if (c + q < g.N) v[q] += p[z * mn + q];
            }
        }
        float bias[8];
        b16_bias8(g, c, bias);
        bf16_t* col = nullptr;
        size_t rowAt = 0;
        if constexpr (HEADS) { col = heads_col<bf16_t>(hp.he, c); rowAt = heads_row(hp.he, r); }
        b16_store8<HEADS>(g, hp, r, c, bias, col, rowAt, v);
    }
}

// ---------------------------------------------------------------------------
// How a product is cut: the tile and the number of parts of the contraction with the smallest estimated time.
struct GemmB16Plan { int shape, splits, kChunk; };
// The tiles: 256 x 256 and 256 x 192 for large products; the others with as many stages in LDS as leave room for the workgroups that
// share a CU.  With two stages a small tile waits for every one of them (2048 x 768 x 4096 in 64 x 64 tiles: 33.8 us; 128 x 64 on eight
// wavefronts with four stages 19.9; 1024^3 10.3, 6.7; 8192 x 768 x 768 in 128 x 192 on eight wavefronts 14.7, with three 13.0).
// Wavefronts, MFMA tiles of one, stages, workgroups a CU is to hold:
#define B16_SHAPES(X) X(0, 4, 2, 2, 4, 2, 2) X(1, 4, 2, 2, 3, 2, 2) X(2, 2, 2, 2, 3, 2, 2) X(3, 4, 2, 1, 3, 3, 2) X(4, 2, 2, 2, 2, 2, 2) \
                      X(5, 2, 2, 2, 2, 3, 1) X(6, 2, 2, 1, 2, 3, 2) X(7, 4, 2, 1, 1, 4, 2) X(8, 2, 2, 1, 1, 4, 2) X(9, 2, 2, 1, 2, 2, 3)
// Microseconds of one tile per 768 k and for its ends, with two and more on the CU (and once besides) and alone on it.  Fitted to 250
// sizes (M 64 .. 32000, N 256 .. 32000, K 256 .. 8192) in three layouts with up to eight parts, 60 launches in a row: the choice is
// 0.4 % slower than the fastest on average and 10 % at worst.  (64 x 128 with two stages has short contractions with two or three tiles
// on a CU, 8192 x 512 x 512 7.9 us against 8.5 in 128 x 128 with three.)
struct GemmB16Shape { int bm, bn; double perK, ends, once, perKAlone, endsAlone; };
static const GemmB16Shape g_b16Shapes[] = {{256, 256, 12.56, 9.20, 0, 12.64, 9.12},  {256, 192, 14.34, 5.68, 0.29, 10.62, 8.68},
                                           {128, 192, 5.33, 4.68, 0.29, 9.01, 5.00}, {128, 192, 6.54, 4.85, 0.12, 6.94, 6.06},
                                           {128, 128, 4.01, 2.78, 0.77, 7.00, 3.85}, {128, 128, 4.73, 3.27, 1.60, 4.79, 5.71},
                                           {64, 128, 2.78, 1.05, 2.42, 3.74, 4.62},  {128, 64, 3.24, 1.71, 2.90, 3.50, 3.60},
                                           {64, 64, 2.03, 0.47, 3.25, 2.21, 3.31},   {64, 128, 2.99, 0.69, 2.72, 6.12, 3.18}};
static constexpr int B16_NSHAPES = sizeof(g_b16Shapes) / sizeof(g_b16Shapes[0]);

static double b16_time(const GemmB16Shape& s, long long tiles, int k)
{
    const double len = ((k + 63) / 64 * 64) / 768.0;
    const long long perCu = ((tiles + 7) / 8 + 31) / 32;
    return perCu == 1 ? len * s.perKAlone + s.endsAlone : perCu * (len * s.perK + s.ends) + s.once;
}

// A result in the memory of an operand is right where everything has been read before any of it is written: where the contraction is
// cut into parts, or where one workgroup reads all that it overwrites - a single tile; with C in the rows of A (B16_ROWS) one tile in
// width, with C in the columns of B (B16_COLUMNS) one in height.  Such a cut is taken if there is one.
enum { B16_APART, B16_ROWS, B16_COLUMNS, B16_MEETS };
static int b16_shares(const GemmB16& q)
{
    const bool a = result_meets(q.C, (long long)q.m * q.n, q.heads, q.m, q.n, q.A, (long long)q.m * q.k);
    const bool b = result_meets(q.C, (long long)q.m * q.n, q.heads, q.m, q.n, q.B, (long long)q.n * q.k);
    if (!a && !b) return B16_APART;
    if (!b && q.C == q.A && q.aK && q.n == q.k) return B16_ROWS;
    if (!a && q.C == q.B && !q.bK && q.m == q.k) return B16_COLUMNS;
    return B16_MEETS;
}
static GemmB16Plan gemm_b16_plan(int m, int n, int k, int shares = B16_APART, int maxParts = 16)
{
    GemmB16Plan best = {0, 0, k};
    double bestT = 1e30;
    for (int sh = 0; sh < B16_NSHAPES; sh++) {
        const GemmB16Shape& s = g_b16Shapes[sh];
        const long long high = (m + s.bm - 1) / s.bm, wide = (n + s.bn - 1) / s.bn, tiles = high * wide;
        for (int S = 1; S <= maxParts; S++) {
            if (S > 1 && k / S < 256) break;
            if (S == 1 && ((shares != B16_APART && shares != B16_ROWS && high > 1) || (shares != B16_APART && shares != B16_COLUMNS && wide > 1))) continue;
            const int chunk = ((k + S - 1) / S + 63) / 64 * 64;
            if ((k + chunk - 1) / chunk != S) continue;
            double t = b16_time(s, tiles * S, chunk);
            if (S > 1) t += 2.0 + (double)(S + 1) * m * n * 4.0 / 3.4e6;
            if (t < bestT) { bestT = t; best = {sh, S, S > 1 ? chunk : k}; }
        }
    }
    return best.splits ? best : gemm_b16_plan(m, n, k, B16_APART, maxParts);
}
int gemm_b16_route(int m, int n, int k)
{
    const GemmB16Plan p = gemm_b16_plan(m, n, k);
    return 4 * p.shape + 64 * p.splits;
}

bool gemm_b16_takes(const GemmB16& q)
{
    if (q.k < 8 || q.m < 1 || q.n < 1) return false;
    if ((((uintptr_t)q.A | (uintptr_t)q.B) & 15) != 0) return false;
    if (q.aK ? q.k % 8 != 0 : (q.m % 8 != 0 || q.m < 8)) return false;
    if (q.bK ? q.k % 8 != 0 : (q.n % 8 != 0 || q.n < 8)) return false;
    // 31-bit byte offsets within a tile's rows of k (256 at most), or within the k rows of a stage
    auto near = [&](bool kFast, int rows) {
        return kFast ? ((long long)std::min(rows, 256) + 1) * q.k < (1ll << 30) : (long long)std::min(q.k, 64) * rows + 256 < (1ll << 30);
    };
    return near(q.aK, q.m) && near(q.bK, q.n);
}
size_t gemm_b16_workspace_bytes(const GemmB16& q)
{
    if (q.m <= 0 || q.n <= 0 || q.k <= 0) return 0;
    const GemmB16Plan p = gemm_b16_plan(q.m, q.n, q.k, b16_shares(q));
    return p.splits > 1 ? (size_t)p.splits * q.m * q.n * sizeof(float) : 0;
}
static int b16_tile_columns(int shape, int n) { return (n + g_b16Shapes[shape].bn - 1) / g_b16Shapes[shape].bn; }
// With the sums of op(A)'s rows: the partial products (none where the contraction is not cut), then the partial sums.  0: not together.
// A partial sum is one of sixteen accumulators per row and tile: up to 128 values each they are no longer than the column sums' own.
size_t gemm_b16_row_sums_workspace_bytes(int m, int n, int k)
{
    if (m <= 0 || n <= 0 || k <= 0) return 0;
    const GemmB16Plan p = gemm_b16_plan(m, n, k);
    const long long columns = b16_tile_columns(p.shape, n);
    if (p.kChunk / (16 * columns) > 128 || (k <= 1024 && p.splits == 1)) return 0;   // one short launch would only be another
    return ((p.splits > 1 ? (size_t)p.splits * m * n : 0) + (size_t)p.splits * columns * m) * sizeof(float);
}

template <int WVM, int WVN, int WM, int WN, int S, int OCC, bool AK, bool BKC, int HEADS, bool SUMS>
static hipError_t launch_b16(hipStream_t s, GemmB16Args& g, const B16Arg<HEADS>& end)
{
    constexpr int BM = 32 * WVM * WM, BN = 32 * WVN * WN, CH = WN % 2 == 0 ? 2 : WN;
    constexpr int stages = S * (BM + BN) * 64 * 2, slices = WVM * WVN * 32 * (32 * CH + 4) * 4, lds = stages > slices ? stages : slices;
    static const hipError_t attr = hipFuncSetAttribute((const void*)gemm_b16_kernel<WVM, WVN, WM, WN, S, OCC, AK, BKC, HEADS, SUMS>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (attr != hipSuccess) return attr;
    g.tilesM = (g.M + BM - 1) / BM;
    g.tilesN = (g.N + BN - 1) / BN;
    const long long total = (long long)g.tilesM * g.tilesN * g.parts;
    if (total > (1ll << 27)) return hipErrorInvalidValue;
    hipLaunchKernelGGL((gemm_b16_kernel<WVM, WVN, WM, WN, S, OCC, AK, BKC, HEADS, SUMS>), dim3((unsigned)((total + 7) / 8 * 8)), 64 * WVM * WVN, lds, s, g, end);
    return hipGetLastError();
}
template <bool AK, bool BKC, int HEADS, bool SUMS = false>
static hipError_t launch_b16_shape(hipStream_t s, GemmB16Args& a, int shape, const B16Arg<HEADS>& end = B16Arg<HEADS>{})
{
    switch (shape) {
#define X(I, WVM, WVN, WM, WN, S, OCC) case I: return launch_b16<WVM, WVN, WM, WN, S, OCC, AK, BKC, HEADS, SUMS>(s, a, end);
        B16_SHAPES(X)
#undef X
    }
    return hipErrorInvalidValue;
}

static GemmB16Args b16_args(const GemmB16& q)
{
    GemmB16Args a = {};
    a.M = q.m; a.N = q.n; a.K = a.kChunk = q.k;
    a.A = q.A; a.B = q.B; a.C = q.C;
    a.lda = q.aK ? q.k : q.m; a.ldb = q.bK ? q.k : q.n;
    a.alpha = q.alpha; a.beta = q.beta;
    a.parts = 1;
    a.bias = q.heads ? (const bf16_t*)q.heads->bias : q.bias;
    if (q.heads) {
        const HeadsEpilogue& he = *q.heads;
        a.vecC = q.n % 8 == 0 && he.hs % 8 == 0 && (((uintptr_t)he.dst[0] | (uintptr_t)he.dst[1] | (uintptr_t)he.dst[2]) & 15) == 0;
    } else {
        a.vecC = q.n % 8 == 0 && ((uintptr_t)q.C & 15) == 0;
    }
    return a;
}

// Whether gemm_b16_rows_kernel takes a product (microseconds with B not in any cache, against the tiles and their sum).  Not where a few
// workgroups would each walk a very long contraction (8 x 64 x 16384: 20.0 against 16.2; 8 x 64 x 8192: 11.3 against 12.1), and not
// where more than 16 rows meet more columns than one workgroup a CU holds (32 x 14336 x 4096: 36 against 27.6).  Its workgroups read
// all rows of A while others write, so a result that shares memory with an operand stays with the tiles.
static bool b16_rows_takes(const GemmB16& q)
{
    if (!q.aK || !q.bK || q.m > 32 || (q.k > 8192 && q.n < 4096) || (q.m > 16 && q.n > 768 * 16)) return false;
    return b16_shares(q) == B16_APART &&
           !result_meets(q.C, (long long)q.m * q.n, q.heads, q.m, q.n, q.heads ? (const bf16_t*)q.heads->bias : q.bias, (long long)q.n);
}
template <int MT, int NT, int NW, int S, int HEADS>
static hipError_t launch_b16_rows_shape(hipStream_t s, const GemmB16Args& g, const HeadsArg<(HEADS > 0)>& ha)
{
    constexpr int lds = NW * S * 16 * 128 * 2;
    static const hipError_t attr = hipFuncSetAttribute((const void*)gemm_b16_rows_kernel<MT, NT, NW, S, HEADS>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (attr != hipSuccess) return attr;
    hipLaunchKernelGGL((gemm_b16_rows_kernel<MT, NT, NW, S, HEADS>), (unsigned)((g.N + 16 * NT - 1) / (16 * NT)), 64 * NW, lds, s, g, ha);
    return hipGetLastError();
}
// One workgroup a CU of 16, 32 or 48 columns as long as that holds all of them: the wider ones read A as often less, and eight
// wavefronts with four stages, or more columns and two, keep 100 KB and more of B on their way.  Past that workgroups of four
// wavefronts, three of them on a CU, so that one's end is another's middle.
template <int MT, int HEADS>
static hipError_t launch_b16_rows(hipStream_t s, const GemmB16Args& g, const HeadsArg<(HEADS > 0)>& ha)
{
    if (g.N <= 256 * 16) return launch_b16_rows_shape<MT, 1, 8, 4, HEADS>(s, g, ha);
    if (g.N <= 512 * 16) return launch_b16_rows_shape<MT, 2, 8, 2, HEADS>(s, g, ha);
    if (g.N <= 768 * 16) return launch_b16_rows_shape<MT, 3, 8, 2, HEADS>(s, g, ha);
    if constexpr (MT == 1) return launch_b16_rows_shape<MT, 1, 4, 3, HEADS>(s, g, ha);
    return hipErrorInvalidValue;   // b16_rows_takes
}

hipError_t gemm_b16(hipStream_t s, const GemmB16& q, void* ws, size_t wsBytes)
{
    if (!gemm_b16_takes(q) || (q.heads && (q.alpha != 1.f || q.beta != 0.f || !q.aK || !q.bK))) return hipErrorInvalidValue;
    if (b16_rows_takes(q)) {
        const GemmB16Args a = b16_args(q);
        if (q.heads && q.heads->fcos) return q.m > 16 ? launch_b16_rows<2, 2>(s, a, heads_arg<true>(q.heads)) : launch_b16_rows<1, 2>(s, a, heads_arg<true>(q.heads));
        if (q.heads) return q.m > 16 ? launch_b16_rows<2, 1>(s, a, heads_arg<true>(q.heads)) : launch_b16_rows<1, 1>(s, a, heads_arg<true>(q.heads));
        return q.m > 16 ? launch_b16_rows<2, 0>(s, a, HeadsArg<false>()) : launch_b16_rows<1, 0>(s, a, HeadsArg<false>());
    }
    const int shares = b16_shares(q);
    GemmB16Plan p = gemm_b16_plan(q.m, q.n, q.k, shares);
    if (q.rowSum) {
        const size_t need = gemm_b16_row_sums_workspace_bytes(q.m, q.n, q.k);
        if (need == 0 || !ws || wsBytes < need || ((uintptr_t)ws & 15) || q.heads || q.aK || q.bK || shares != B16_APART) return hipErrorInvalidValue;
    }
    if (p.splits > 1 && (!ws || wsBytes < (size_t)p.splits * q.m * q.n * sizeof(float) || ((uintptr_t)ws & 15))) {
        if (shares == B16_APART) { p.splits = 1; p.kChunk = q.k; }
        else p = gemm_b16_plan(q.m, q.n, q.k, shares, 1);
    }
    GemmB16Args a = b16_args(q);
    a.parts = p.splits; a.kChunk = p.kChunk;
    a.part = (float*)ws;
    hipError_t e;
    if (q.heads && q.heads->fcos) e = launch_b16_shape<true, true, 2>(s, a, p.shape, heads_arg<true>(q.heads));
    else if (q.heads) e = launch_b16_shape<true, true, 1>(s, a, p.shape, heads_arg<true>(q.heads));
    else if (q.rowSum) e = launch_b16_shape<false, false, 0, true>(s, a, p.shape);
    else if (q.aK) e = q.bK ? launch_b16_shape<true, true, 0>(s, a, p.shape) : launch_b16_shape<true, false, 0>(s, a, p.shape);
    else e = q.bK ? launch_b16_shape<false, true, 0>(s, a, p.shape) : launch_b16_shape<false, false, 0>(s, a, p.shape);
    const int rowBlocks = q.rowSum ? (q.m + 255) / 256 : 0;
    const int grid = rowBlocks + (p.splits > 1 ? (int)std::min<size_t>(((size_t)q.m * ((q.n + 7) / 8) + 255) / 256, 4096) : 0);
    if (e != hipSuccess || grid == 0) return e;
    if (q.heads) hipLaunchKernelGGL(gemm_b16_sum_kernel<2>, grid, 256, 0, s, a, heads_arg<true>(q.heads), p.splits, 0, (bf16_t*)nullptr);
    else hipLaunchKernelGGL(gemm_b16_sum_kernel<0>, grid, 256, 0, s, a, HeadsArg<false>(), p.splits, rowBlocks, q.rowSum);
    return hipGetLastError();
}

template <int WVM, int WVN, int WM, int WN, int S, int OCC>
static hipError_t launch_b16_group(hipStream_t s, GemmB16Group& grp, int count)
{
    constexpr int BM = 32 * WVM * WM, BN = 32 * WVN * WN, CH = WN % 2 == 0 ? 2 : WN;
    constexpr int stages = S * (BM + BN) * 64 * 2, slices = WVM * WVN * 32 * (32 * CH + 4) * 4, lds = stages > slices ? stages : slices;
    static const hipError_t attr = hipFuncSetAttribute((const void*)gemm_b16_group_kernel<WVM, WVN, WM, WN, S, OCC>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (attr != hipSuccess) return attr;
    long long total = 0;
    for (int p = 0; p < 3; p++) {
        GemmB16Args& g = grp.g[p];
        grp.first[p] = (int)total;
        if (p >= count) continue;
        g.tilesM = (g.M + BM - 1) / BM;
        g.tilesN = (g.N + BN - 1) / BN;
        total += (long long)g.tilesM * g.tilesN;
        if (total > (1ll << 27)) return hipErrorInvalidValue;
    }
    grp.first[3] = (int)total;
    for (int p = count; p < 3; p++) grp.first[p] = (int)total;
    hipLaunchKernelGGL((gemm_b16_group_kernel<WVM, WVN, WM, WN, S, OCC>), dim3((unsigned)((total + 7) / 8 * 8)), 64 * WVM * WVN, lds, s, grp);
    return hipGetLastError();
}

// `count` (2 or 3) products A B^T through their heads epilogues, all of one n and k, as one launch.  False: a product is none that
// gemm_b16 takes, or one that gemm_b16_rows_kernel may take.
bool gemm_b16_group(hipStream_t s, const GemmB16* q, int count, hipError_t* e)
{
    GemmB16Group grp = {};
    for (int p = 0; p < count; p++) {
        if (!gemm_b16_takes(q[p]) || !q[p].heads || !q[p].aK || !q[p].bK || q[p].n != q[0].n || q[p].k != q[0].k || q[p].m <= 32) return false;
        grp.g[p] = b16_args(q[p]);
        grp.h[p].he = *q[p].heads;
    }
    int best = 0;
    double bestT = 1e30;
    for (int sh = 0; sh < B16_NSHAPES; sh++) {
        const GemmB16Shape& c = g_b16Shapes[sh];
        long long tiles = 0;
        for (int p = 0; p < count; p++) tiles += (long long)((q[p].m + c.bm - 1) / c.bm) * ((q[p].n + c.bn - 1) / c.bn);
        const double t = b16_time(c, tiles, q[0].k);
        if (t < bestT) { bestT = t; best = sh; }
    }
    switch (best) {
#define X(I, WVM, WVN, WM, WN, S, OCC) case I: *e = launch_b16_group<WVM, WVN, WM, WN, S, OCC>(s, grp, count); break;
        B16_SHAPES(X)
#undef X
    }
    return true;
}

// ---------------------------------------------------------------------------
// C (m x n, fp32) = alpha X W^T + beta C for a 16-bit weight matrix W (n x k), on the bf16 matrix cores, C in fp32.
// split = false: A is X rounded to bf16, m rows of k.  split = true keeps the activations' precision: A holds every row of
// an fp32 X as two bf16 rows back to back, the bf16 nearest to each of its k values and then the bf16 nearest to what
// those leave over, and the kernel walks W once for each.  The products are exact and accumulate in fp32, so what is lost
// is the part of X below its leading sixteen bits: 2^-17 relative, against 2^-9 for activations rounded to bf16.
// k a multiple of 64, 16-byte aligned operands.
// The tile with the smallest estimate for the whole contraction; a row of A that is split is 2 k long, and B is walked twice.  us at 2048
// rows of 768, split, before (a kernel that staged through registers) and now: with the rotation, to 2304 columns, 40.6, 30.9; with
// SwiGLU, to 4096, 40.5, 35.5; to 768, and from 2048 to 768, 26.9, 21.9 on average; to 32000 254, 249.
template <int END>
static hipError_t gemm_b16_prompt(hipStream_t s, int m, int n, int k, float alpha, const void* A, bool split, const void* W, float beta, float* C,
                                  const PromptEpilogue* pe)
{
    GemmB16Args a = {};
    a.M = m; a.N = n; a.K = a.kChunk = split ? 2 * k : k;
    a.A = (const bf16_t*)A; a.B = (const bf16_t*)W; a.C = (bf16_t*)C;
    a.lda = a.K; a.ldb = k;
    a.alpha = alpha; a.beta = beta;
    a.parts = 1;
    a.vecC = n % 4 == 0 && ((uintptr_t)C & 15) == 0;
    PromptArg end = {};
    if (pe) end.pe = *pe;
    end.pe.kB = k;
    int best = 0;
    double bestT = 1e30;
    for (int sh = 0; sh < B16_NSHAPES; sh++) {
        const GemmB16Shape& c = g_b16Shapes[sh];
        const long long tiles = (long long)((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn);
        const double t = b16_time(c, tiles, a.K);
        if (t < bestT) { bestT = t; best = sh; }
    }
    return launch_b16_shape<true, true, END>(s, a, best, end);
}
static bool bf16_f32_operands_ok(int k, const void* A, const void* W) { return k > 0 && k % 64 == 0 && (((uintptr_t)A | (uintptr_t)W) & 15) == 0; }
hipError_t k_gemm_bf16_f32(hipStream_t s, int m, int n, int k, float alpha, const void* A, bool split, const void* W, float beta, float* C)
{
    if (m <= 0 || n <= 0) return hipSuccess;
    if (!bf16_f32_operands_ok(k, A, W)) return hipErrorInvalidValue;
    return gemm_b16_prompt<3>(s, m, n, k, alpha, A, split, W, beta, C, nullptr);
}
// out (m x hid) = silu(X W1^T) (X W3^T) for the stacked 16-bit W13 (2 hid x k), as bf16 rows (outSplit: hi | lo rows)
hipError_t k_gemm_bf16_swiglu(hipStream_t s, int m, int hid, int k, const void* A, bool split, const void* W13, void* out, bool outSplit)
{
    if (m <= 0 || hid <= 0) return hipSuccess;
    if (!bf16_f32_operands_ok(k, A, W13) || (hid & 1) || (((uintptr_t)out) & 3)) return hipErrorInvalidValue;
    PromptEpilogue pe = {};
    pe.out = out; pe.hid = hid; pe.split = outSplit ? 1 : 0;
    return gemm_b16_prompt<4>(s, m, 2 * hid, k, 1.f, A, split, W13, 0.f, nullptr, &pe);
}
// the stacked 16-bit Wqkv ((H + 2 kvH) hs x k) product of B x P rows, rotated and scattered (PromptEpilogue, 2)
hipError_t k_gemm_bf16_qkv_rope(hipStream_t s, int B, int P, int H, int kvH, int hs, int k, const void* A, bool split, const void* Wqkv,
                                void* q, void* kh, void* vh, bool heads16, void* kc, void* vc, bool cache16, int seqLen,
                                const float* fcos, const float* fsin)
{
    const int m = B * P, n = (H + 2 * kvH) * hs;
    if (m <= 0 || n <= 0) return hipSuccess;
    if (!bf16_f32_operands_ok(k, A, Wqkv) || (hs & 3) || kvH <= 0 || H % kvH != 0) return hipErrorInvalidValue;
    if ((((uintptr_t)q | (uintptr_t)kh | (uintptr_t)vh | (uintptr_t)kc | (uintptr_t)vc) & 15) != 0) return hipErrorInvalidValue;
    PromptEpilogue pe = {};
    pe.q = q; pe.k = kh; pe.v = vh; pe.kc = kc; pe.vc = vc; pe.fcos = fcos; pe.fsin = fsin;
    pe.P = P; pe.H = H; pe.kvH = kvH; pe.hs = hs; pe.seqLen = seqLen; pe.heads16 = heads16 ? 1 : 0; pe.cache16 = cache16 ? 1 : 0;
    pe.kvMul = H / kvH; pe.invP = 1.0f / (float)P; pe.invHs = 1.0f / (float)hs;
    if (m >= (1 << 24) || n >= (1 << 24)) return hipErrorInvalidValue;
    return gemm_b16_prompt<5>(s, m, n, k, 1.f, A, split, Wqkv, 0.f, nullptr, &pe);
}

}  // namespace mch
