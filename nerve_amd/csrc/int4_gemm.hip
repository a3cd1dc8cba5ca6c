// INT4 linears, mostly for more than 16 rows: a tiled, split-K form of the kernels
// in int4.hip, for bf16 and for INT8-prequantized activations.
//
// A block (4 waves) owns 16 MT rows and 256 columns over a range of 128-column
// stages of K; wave w owns columns 64 w .. 64 w + 63.  Weights go from memory
// straight into each wave's registers as MFMA operands, one or two stages ahead,
// and are expanded once per 16 MT rows (code -> bf16 128 + q, one and-or per two
// codes).  Activations are staged once per block through registers into a
// double-buffered LDS tile: bf16 rows are put into the pair order of the
// expansion and summed per scale segment; int8 rows become bf16 (exact) and are
// summed per 32 columns.  A 16-byte piece p of row t sits in slot
// p ^ (t % 16), so the 16 rows of an operand read hit distinct banks.
//
//   sum_k x (q - z) = sum_k x (128 + q) - (128 + z) sum_k x
//
// Without zero points (z = 8) the MFMA chain's accumulator starts at
// -136 sum_k x, which the staging has stored.  For int8 rows every term is an
// integer below 2^24, so the 32-column block dots are exact in f32, as the
// shader's integer dots are.
//
// K is split over gridDim so that the launch fills the chip; partial sums go to
// the context's split-K scratch (f32 [split][row][column]) and a second launch
// adds them in split order.
//
// Bound: vector-ALU issue (a stage of four row tiles is 64 MFMAs, about 1024
// cycles, beside some 300 vector instructions of 4 cycles: 112 to expand the
// codes, 64 to fold the segment, 60 to stage the rows); leaving out the loads
// changes it by under 10%.  64 columns a wave halve the LDS operand reads of 32
// columns (512 rows of 4096 x 14336: 70 against 119 us).  Five row tiles spill
// throughout; four spill 3 to 10 registers in the CT and int8 forms, which the
// estimate below does not count.  Against the 16-row kernels in int4.hip: 301 rows of 14336 x 4096 (CT)
// 397 -> 65 us, 512 rows of 4096 x 14336 (GPTQ) 150 -> 69 us, 64 rows of
// 14336 x 4096 25.9 -> 20.0 us.
#include <algorithm>

#include "int4_dev.h"

namespace {

constexpr uint32_t GT_COLS = 256;           // columns per block
constexpr uint32_t GT_K = 128;              // K columns per stage
constexpr int GJ = 4;                       // 16-column MFMA tiles per wave
constexpr uint32_t GT_WAVES = GT_COLS / (16 * GJ);
constexpr uint32_t GT_THREADS = 64 * GT_WAVES;

struct GemmArgs {
    Int4Args L;
    const uint8_t* q;                       // int8 rows [B, K], or null
    const float* sx;                        // their scales [B, K/32]
    float* part;                            // [splits][B][N], or null (one split: finalize)
    uint32_t tiles, tgroups, splits, work, per_xcd;
};

__device__ __forceinline__ uint32_t bf16_hi_pair(float lo, float hi) {   // exact bf16 values
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}

__device__ __forceinline__ float byte_f32(uint32_t w, int b) { return (float)(int8_t)(w >> (8 * b)); }

// I8: 0 bf16 rows, 1 pair-packed int8, 2 int8 in column order.  SEG: 32-column
// blocks per scale segment (1, 2 or 4; it divides the group).
template <int MT, int SEG, int I8, bool CT, bool ZP>
__global__ __launch_bounds__(GT_THREADS, 2) void int4_gemm_kernel(GemmArgs P) {
    constexpr int NSEG = 4 / SEG;
    constexpr int NSUM = I8 ? 4 : NSEG;     // row sums per stage
    constexpr uint32_t ROWS = 16 * MT;
    constexpr float SUM = ZP ? 1.0f : -136.0f;   // what the row sums are stored times
    __shared__ __attribute__((aligned(16))) uint8_t at[2][ROWS][256];
    __shared__ __attribute__((aligned(16))) float rsum[2][NSUM][ROWS];
    __shared__ __attribute__((aligned(16))) float rsx[I8 ? 2 : 1][I8 ? 4 : 1][I8 ? ROWS : 4];
    const Int4Args& A = P.L;
    const uint32_t w = (blockIdx.x % 8) * P.per_xcd + blockIdx.x / 8;
    if (w >= P.work) return;
    // Row groups fastest, then column tiles: neighbours on an XCD share the
    // weights, then the activations, through its L2.
    const uint32_t tg = w % P.tgroups, tile = w / P.tgroups % P.tiles, split = w / P.tgroups / P.tiles;
    const uint32_t K = A.K, N = A.N, M = A.B, nst = (K + GT_K - 1) / GT_K;
    const uint32_t s0 = (uint32_t)((uint64_t)nst * split / P.splits), s1 = (uint32_t)((uint64_t)nst * (split + 1) / P.splits);
    const uint32_t tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const uint32_t g = lane >> 4, rr = lane & 15;
    const uint32_t m0 = tg * ROWS, n0 = tile * GT_COLS + wave * 16 * GJ;
    // Columns of MFMA tile j: GPTQ n0 + 4 rr + j (one 16-byte load feeds the
    // four tiles), CT n0 + 16 j + rr (a load feeds four steps).  Columns past
    // N are clamped and not stored.
    const uint32_t c4 = min(n0 + GJ * rr, N - GJ);
    uint32_t cj[GJ];
#pragma unroll
    for (int j = 0; j < GJ; j++) cj[j] = CT ? min(n0 + 16 * j + rr, N - 1) : c4 + j;
    const uint32_t ngroups = K / A.G;
    const uint32_t zshift = 4 * (c4 % 8);   // GJ codes of one word

    struct WSet {
        uint32_t w[4][GJ];                  // word of step u, tile j (CT before its transposition: word u of tile j)
        uint16_t s[NSEG][GJ];
        uint32_t z[NSEG];
    };
    auto load_step = [&](WSet& W, uint32_t st, int u) __attribute__((always_inline)) {
        const uint32_t k8 = st * (GT_K / 8);
        if constexpr (!CT) load_words<GJ>(A.qw + (uint64_t)min(k8 + 4 * u + g, K / 8 - 1) * N + c4, W.w[u]);
    };
    auto load_rest = [&](WSet& W, uint32_t st) __attribute__((always_inline)) {
        const uint32_t k0 = st * GT_K;
        if constexpr (CT) {
#pragma unroll
            for (int j = 0; j < GJ; j++) {
                const v4i v = *reinterpret_cast<const v4i*>(A.qw + (uint64_t)cj[j] * (K / 8) + k0 / 8 + 4 * g);
#pragma unroll
                for (int u = 0; u < 4; u++) W.w[u][j] = (uint32_t)v[u];
            }
        }
#pragma unroll
        for (int sg = 0; sg < NSEG; sg++) {
            const uint32_t grp = min(k0 + 32 * SEG * sg, K - 1) / A.G;
            if (CT) {
#pragma unroll
                for (int j = 0; j < GJ; j++) W.s[sg][j] = A.scales[(uint64_t)cj[j] * ngroups + grp];
            } else {
                uint32_t v[GJ / 2];
                load_words<GJ / 2>(reinterpret_cast<const uint32_t*>(A.scales + (uint64_t)grp * N + c4), v);
#pragma unroll
                for (int j = 0; j < GJ; j++) W.s[sg][j] = (uint16_t)(v[j / 2] >> (16 * (j % 2)));
            }
            W.z[sg] = ZP ? A.qzeros[(uint64_t)grp * (N / 8) + c4 / 8] >> zshift : 0x8888u;
        }
    };
    // Staging: 8 lanes read 128 contiguous bytes of a row (whole lines).  bf16:
    // the threads cover GT_THREADS / 8 rows of one 64-column half per pass,
    // lane p8 of 8 holding columns 8 p8 .. 8 p8 + 7; int8: the 128 bytes are
    // the row's stage, lane p8 holding columns 16 p8 .. 16 p8 + 15.
    constexpr uint32_t RPP = GT_THREADS / 8;                                // rows per pass
    constexpr int NP = (I8 ? 1 : 2) * (int)((ROWS + RPP - 1) / RPP);        // passes
    const uint32_t p8 = tid & 7, r8 = tid >> 3;
    // Row and half of pass i (both halves of a row block in turn).
    auto pass_row = [&](int i) { return I8 ? r8 + i * RPP : r8 + (i / 2) * RPP; };
    struct ASet {
        v4i a[NP];
        float sx[I8 ? NP : 1];
    };
    auto load_a = [&](ASet& S, uint32_t st) __attribute__((always_inline)) {
        const uint32_t k0 = st * GT_K;
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const uint32_t row = min(m0 + min(pass_row(i), ROWS - 1), M - 1);
            if (I8) {
                S.a[i] = *reinterpret_cast<const v4i*>(P.q + (uint64_t)row * K + min(k0 + 16 * p8, K - 16));
                S.sx[i] = P.sx[(uint64_t)row * (K / 32) + min(k0 / 32 + p8 / 2, K / 32 - 1)];
            } else {
                S.a[i] = *reinterpret_cast<const v4i*>(A.x + (uint64_t)row * K + min(k0 + 64 * (i % 2) + 8 * p8, K - 8));
            }
        }
    };
    auto put_a = [&](const ASet& S, uint32_t buf) __attribute__((always_inline)) {
        float half = 0.0f;
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const uint32_t t = pass_row(i), sw = t & 15;
            if (ROWS % RPP != 0 && t >= ROWS) break;
            uint8_t* row = &at[buf][t][0];
            if constexpr (I8 == 0) {
                float v = 0.0f;
#pragma unroll
                for (int d = 0; d < 4; d++) v = dot2_bf16((uint32_t)S.a[i][d], ONES_BF16, v);
                *reinterpret_cast<v4i*>(row + (((8 * (i % 2) + p8) ^ sw) << 4)) = permute_act(S.a[i]);
                // Segment sums: 4 lanes hold a 32-column block.
                v = lanes_sum_up<SEG == 1 ? 4 : 8>(v);
                if (SEG == 4) {
                    if (i % 2 == 0) half = v;
                    else if (p8 == 0) rsum[buf][0][t] = SUM * (half + v);
                } else if (SEG == 2) {
                    if (p8 == 0) rsum[buf][(i % 2) % NSUM][t] = SUM * v;
                } else if ((p8 & 3) == 0) {
                    rsum[buf][(2 * (i % 2) + (p8 >> 2)) % NSUM][t] = SUM * v;
                }
            } else {
                int sum = 0;
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const uint32_t a = (uint32_t)S.a[i][2 * h], b = (uint32_t)S.a[i][2 * h + 1];
                    sum = __builtin_amdgcn_sdot4((int)a, 0x01010101, sum, false);
                    sum = __builtin_amdgcn_sdot4((int)b, 0x01010101, sum, false);
                    // Columns (0,4), (1,5), (2,6), (3,7) of the octet.
                    v4i p;
                    if (I8 == 1)
                        p = v4i{(int)bf16_hi_pair(byte_f32(a, 0), byte_f32(a, 2)), (int)bf16_hi_pair(byte_f32(b, 0), byte_f32(b, 2)),
                                (int)bf16_hi_pair(byte_f32(a, 1), byte_f32(a, 3)), (int)bf16_hi_pair(byte_f32(b, 1), byte_f32(b, 3))};
                    else
                        p = v4i{(int)bf16_hi_pair(byte_f32(a, 0), byte_f32(b, 0)), (int)bf16_hi_pair(byte_f32(a, 1), byte_f32(b, 1)),
                                (int)bf16_hi_pair(byte_f32(a, 2), byte_f32(b, 2)), (int)bf16_hi_pair(byte_f32(a, 3), byte_f32(b, 3))};
                    *reinterpret_cast<v4i*>(row + (((2 * p8 + h) ^ sw) << 4)) = p;
                }
                sum += __builtin_amdgcn_update_dpp(0, sum, 0xB1, 0xF, 0xF, false);   // lanes 2 b, 2 b + 1: block b
                if ((p8 & 1) == 0) {
                    rsum[buf][(p8 >> 1) % NSUM][t] = (float)(-136 * sum);
                    rsx[buf][p8 >> 1][t] = S.sx[i] * I8_SCALE_DOWN;
                }
            }
        }
    };
    const uint32_t exponent = pair_exponent();
    v4f acc[MT][GJ];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int j = 0; j < GJ; j++) acc[m][j] = v4f{0.f, 0.f, 0.f, 0.f};
    // Contracts stage st from LDS buffer buf; each step's words are refilled
    // for stage `next` once expanded.
    auto contract = [&](WSet& W, uint32_t st, uint32_t buf, uint32_t next) __attribute__((always_inline)) {
        const uint32_t nu = min(4u, K / 32 - st * 4);        // blocks of this stage (a K tail has fewer)
        if constexpr (CT && I8 != 0) {
            // Lane group g holds block g's four words of each column tile:
            // transposed so that it holds word g of block u in element u.
#pragma unroll
            for (int j = 0; j < GJ; j++) {
                const auto a = __builtin_amdgcn_permlane32_swap(W.w[0][j], W.w[2][j], false, false);
                const auto b = __builtin_amdgcn_permlane32_swap(W.w[1][j], W.w[3][j], false, false);
                const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
                const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
                W.w[0][j] = c[0]; W.w[1][j] = c[1]; W.w[2][j] = d[0]; W.w[3][j] = d[1];
            }
        }
        v4f ag[MT][GJ];
        // Row operands one step ahead of their MFMAs (where the registers allow).
        constexpr int AVN = MT == 4 && (CT || I8) ? 1 : 2;
        v4i av[AVN][MT];
        auto read_rows = [&](int u) __attribute__((always_inline)) {
            const uint32_t piece = (CT && I8 == 0 ? 4 * g + u : 4 * u + g) ^ rr;
#pragma unroll
            for (int m = 0; m < MT; m++) av[u % AVN][m] = *reinterpret_cast<const v4i*>(&at[buf][16 * m + rr][piece << 4]);
        };
        v4f d[2][GJ];
        auto fold = [&](int u, int m) __attribute__((always_inline)) {
            const v4f sx = *reinterpret_cast<const v4f*>(&rsx[buf][I8 ? u : 0][I8 ? 16 * m + 4 * g : 0]);
#pragma unroll
            for (int j = 0; j < GJ; j++) {
                if (u % SEG == 0) ag[m][j] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < 4; i++) ag[m][j][i] = fmaf(d[m & 1][j][i], sx[i], ag[m][j][i]);
            }
        };
        if (AVN == 2) read_rows(0);
#pragma unroll
        for (int u = 0; u < 4; u++) {
            if (u % SEG == 0 && (uint32_t)u >= nu) break;    // the tail is whole segments
            v4i bw[GJ];
#pragma unroll
            for (int j = 0; j < GJ; j++) bw[j] = dequant_word(W.w[u][j], exponent);
            load_step(W, next, u);
            if (AVN == 1) read_rows(u);
            else if (u < 3) read_rows(u + 1);
#pragma unroll
            for (int m = 0; m < MT; m++) {
                if constexpr (I8 != 0) {
                    // The previous row tile's dots are folded while this one's
                    // are in the matrix unit.
                    const v4f c = *reinterpret_cast<const v4f*>(&rsum[buf][u][16 * m + 4 * g]);
#pragma unroll
                    for (int j = 0; j < GJ; j++) d[m & 1][j] = mfma_bf16(av[u % AVN][m], bw[j], c);
                    if (m > 0) fold(u, m - 1);
                    if (m == MT - 1) fold(u, m);
                } else {
                    if (u % SEG == 0) {
                        v4f c = v4f{0.f, 0.f, 0.f, 0.f};
                        if (!ZP) c = *reinterpret_cast<const v4f*>(&rsum[buf][u / SEG][16 * m + 4 * g]);
#pragma unroll
                        for (int j = 0; j < GJ; j++) ag[m][j] = c;
                    }
#pragma unroll
                    for (int j = 0; j < GJ; j++) ag[m][j] = mfma_bf16(av[u % AVN][m], bw[j], ag[m][j]);
                }
            }
            if (u % SEG == SEG - 1) {
                const int sg = u / SEG;
                float sc[GJ];
#pragma unroll
                for (int j = 0; j < GJ; j++) sc[j] = decode_scale(W.s[sg][j], A.scale_bf16);
                if constexpr (ZP) {
                    float zc[GJ];
#pragma unroll
                    for (int j = 0; j < GJ; j++) zc[j] = -128.0f - (float)((W.z[sg] >> (4 * j)) & 15u);
#pragma unroll
                    for (int m = 0; m < MT; m++) {
                        const v4f rs = *reinterpret_cast<const v4f*>(&rsum[buf][sg][16 * m + 4 * g]);
#pragma unroll
                        for (int j = 0; j < GJ; j++)
#pragma unroll
                            for (int i = 0; i < 4; i++) ag[m][j][i] = fmaf(zc[j], rs[i], ag[m][j][i]);
                    }
                }
#pragma unroll
                for (int m = 0; m < MT; m++)
#pragma unroll
                    for (int j = 0; j < GJ; j++)
#pragma unroll
                        for (int i = 0; i < 4; i++) acc[m][j][i] = fmaf(ag[m][j][i], sc[j], acc[m][j][i]);
            }
        }
        load_rest(W, next);
    };
    // Stage st's LDS tile is complete at its barrier, which every wave reaches
    // after its reads of the other buffer: the next stage's tile is written
    // there at once, and its registers reloaded for the stage after.
    const uint32_t last = s1 - 1;
    constexpr uint32_t WD = MT < (CT || ZP ? 3 : 4) ? 2 : 1;     // stages a weight set is loaded ahead
    ASet as;
    WSet wa, wb;
    WSet& w1 = WD == 2 ? wb : wa;
    load_a(as, s0);
#pragma unroll
    for (int u = 0; u < 4; u++) load_step(wa, s0, u);
    load_rest(wa, s0);
    put_a(as, 0);
    load_a(as, min(s0 + 1, last));
    if (WD == 2) {
#pragma unroll
        for (int u = 0; u < 4; u++) load_step(wb, min(s0 + 1, last), u);
        load_rest(wb, min(s0 + 1, last));
    }
    for (uint32_t st = s0; st < s1; st += 2) {
        __syncthreads();
        put_a(as, 1);
        load_a(as, min(st + 2, last));
        contract(wa, st, 0, min(st + WD, last));
        if (st + 1 >= s1) break;
        __syncthreads();
        put_a(as, 0);
        load_a(as, min(st + 3, last));
        contract(w1, st + 1, 1, min(st + 1 + WD, last));
    }
#pragma unroll
    for (int m = 0; m < MT; m++) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t t = m0 + 16 * m + 4 * g + i;
            if (t >= M) continue;
            if (I8) {
#pragma unroll
                for (int j = 0; j < GJ; j++) acc[m][j][i] *= I8_SCALE_UP;
            }
            if (P.part) {
                float* p = P.part + ((uint64_t)split * M + t) * N;
                if (CT) {
#pragma unroll
                    for (int j = 0; j < GJ; j++)
                        if (n0 + 16 * j + rr < N) p[n0 + 16 * j + rr] = acc[m][j][i];
                } else if (n0 + GJ * rr < N) {
                    *reinterpret_cast<v4f*>(p + c4) = v4f{acc[m][0][i], acc[m][1][i], acc[m][2][i], acc[m][3][i]};
                }
            } else {
#pragma unroll
                for (int j = 0; j < GJ; j++)
                    if ((CT ? n0 + 16 * j + rr : n0 + GJ * rr) < N) finalize_store(A, t, cj[j], acc[m][j][i]);
            }
        }
    }
}

// Partial sums in split order, then bias or residual and the bf16 store: four
// columns per thread, eight splits' loads in flight.
__global__ __launch_bounds__(256) void int4_split_sum_kernel(Int4Args A, const float* part, uint32_t splits) {
    const uint64_t i = ((uint64_t)blockIdx.x * 256 + threadIdx.x) * 4, total = (uint64_t)A.B * A.N;
    if (i >= total) return;
    const float* p = part + i;
    v4f v = v4f{0.f, 0.f, 0.f, 0.f};
    for (uint32_t s = 0; s < splits; s += 8) {
        v4f t[8];
#pragma unroll
        for (uint32_t e = 0; e < 8; e++) t[e] = *reinterpret_cast<const v4f*>(p + min(s + e, splits - 1) * total);
#pragma unroll
        for (uint32_t e = 0; e < 8; e++)
            if (s + e < splits) v += t[e];
    }
    const uint32_t t = (uint32_t)(i / A.N), n = (uint32_t)(i % A.N);
#pragma unroll
    for (int j = 0; j < 4; j++) finalize_store(A, t, n + j, v[j]);
}

template <int MT, int SEG, int I8, bool CT, bool ZP>
void launch_form(const GemmArgs& P, hipStream_t st) {
    int4_gemm_kernel<MT, SEG, I8, CT, ZP><<<P.per_xcd * 8, GT_THREADS, 0, st>>>(P);
}

template <int SEG, int I8, bool CT, bool ZP>
void launch_rows(const GemmArgs& P, uint32_t mt, hipStream_t st) {
    if (mt == 1) launch_form<1, SEG, I8, CT, ZP>(P, st);
    else if (mt == 2) launch_form<2, SEG, I8, CT, ZP>(P, st);
    else if (mt == 3) launch_form<3, SEG, I8, CT, ZP>(P, st);
    else launch_form<4, SEG, I8, CT, ZP>(P, st);
}

template <int I8, bool CT, bool ZP = false>
void launch_seg(const GemmArgs& P, uint32_t mt, hipStream_t st) {
    if constexpr (CT && I8 == 0) {
        launch_rows<4, I8, CT, ZP>(P, mt, st);       // the entry point needs groups of 128
    } else {
        if (P.L.G % 128 == 0) launch_rows<4, I8, CT, ZP>(P, mt, st);
        else if (P.L.G % 64 == 0) launch_rows<2, I8, CT, ZP>(P, mt, st);
        else launch_rows<1, I8, CT, ZP>(P, mt, st);
    }
}

// Row tiles per block and splits of K, by an estimate in units of one stage of
// a four-row-tile block alone on its CU (about 1.2 us): a block's stage costs
// its row tiles and two more for the weights' expansion; two blocks share a CU
// at 1.2 times the time of one; the second launch costs 2.5 units and a quarter
// more for every MiB of partial sums.  Measured (us, this choice / the other):
// 64 rows of 14336 x 4096, 16 splits / 28: 20.6 / 22.5; 301 rows of the same,
// 6 / 3: 65.9 / 81; 300 rows of 4096 x 14336, 3 row tiles / 4: 59.6 / 66; 512
// rows, 4 / 3: 70 / 92.  Two blocks on a CU that hold fewer than six
// stages times row tiles each cost more than the estimate's 1.2 (CT, two such a CU
// / one: 33 rows of 8192 x 1024 15.8 / 12.8, 64 of 4096 x 4096 21.0 / 17.9, 128 of
// 3072 x 3072 19.1 / 17.3; but 17 of 8192 x 8192 with two row tiles 23.6 / 28.8)
// and are not taken, except where one row group reads the weights (8 rows of 8192 x
// 8192, g32, 16.8 / 19.2).
struct Plan {
    uint32_t mt, tgroups, splits;
};

Plan plan_gemm(uint32_t M, uint32_t N, uint32_t K, uint32_t tiles, uint32_t cus) {
    const uint32_t rt = (M + 15) / 16, nst = (K + GT_K - 1) / GT_K;
    const uint64_t bytes = (uint64_t)M * N * 4;
    const uint32_t most = (uint32_t)std::min<uint64_t>(std::max(1u, nst / 2), std::max<uint64_t>(1, nh::kSplitBytes / bytes));
    Plan best{};
    double least = 1e30;
    for (uint32_t mt = 1; mt <= 4; mt++) {
        const uint32_t tgroups = (rt + mt - 1) / mt;
        for (uint32_t splits = 1; splits <= most; splits++) {
            const uint64_t nb = (uint64_t)tiles * tgroups * splits, full = nb / (2 * cus), rem = nb % (2 * cus);
            if (splits > 1 && nb > 2 * cus) break;
            if (splits > 1 && tgroups > 1 && nb > cus && mt * ((nst + splits - 1) / splits) < 6) continue;
            const double rounds = 1.2 * (double)full + (rem == 0 ? 0.0 : rem <= cus ? 1.0 : 1.2);
            double cost = rounds * ((nst + splits - 1) / splits + 2) * (mt + 2) / 6.0;
            if (splits > 1) cost += 2.5 + 0.25 * splits * (double)bytes / (1 << 20);
            if (cost < least) least = cost, best = Plan{mt, tgroups, splits};
        }
    }
    return best;
}

}  // namespace

namespace nh {

bool int4_gemm(const nerve_hip_ctx* ctx, const Int4Args& A, const PpArgs* i8, bool paired, bool ct, hipStream_t st) {
    // 16-byte loads of weights and rows, 8-byte ones of GPTQ scales; K / 32
    // blocks come in whole stages for CT rows.
    if (A.N % 16 || A.K % 32 || ((uintptr_t)A.qw & 15) || ((uintptr_t)(i8 ? (const void*)i8->q : A.x) & 15)) return false;
    if (ct ? A.K % GT_K != 0 : ((uintptr_t)A.scales & 7) != 0) return false;
    GemmArgs P{};
    P.L = A;
    if (i8) {
        P.q = reinterpret_cast<const uint8_t*>(i8->q);
        P.sx = i8->s;
        if (A.K % 16) return false;
    }
    P.tiles = (A.N + GT_COLS - 1) / GT_COLS;
    const Plan plan = plan_gemm(A.B, A.N, A.K, P.tiles, (uint32_t)ctx->cu_count);
    const uint32_t mt = plan.mt;
    P.tgroups = plan.tgroups;
    P.splits = plan.splits;
    P.part = P.splits > 1 ? static_cast<float*>(ctx->split) : nullptr;
    P.work = P.tiles * P.tgroups * P.splits;
    P.per_xcd = (P.work + 7) / 8;
    if (!i8) {
        if (ct) launch_seg<0, true>(P, mt, st);
        else if (A.qzeros) launch_seg<0, false, true>(P, mt, st);
        else launch_seg<0, false>(P, mt, st);
    } else if (paired) {
        launch_seg<1, false>(P, mt, st);
    } else {
        if (ct) launch_seg<2, true>(P, mt, st);
        else launch_seg<2, false>(P, mt, st);
    }
    if (P.splits > 1) int4_split_sum(A, P.part, P.splits, st);
    return true;
}

void int4_split_sum(const Int4Args& A, const float* part, uint32_t splits, hipStream_t st) {
    int4_split_sum_kernel<<<(uint32_t)(((uint64_t)A.B * A.N / 4 + 255) / 256), 256, 0, st>>>(A, part, splits);
}

}  // namespace nh
