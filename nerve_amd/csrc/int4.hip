// Group-scaled INT4 linear (a9) on gfx950 bf16 MFMA.
//
// Reference: linear_int4_gptq.comp.template:95-119 / linear_int4_ct.comp.
// template:95-124 compute y[n] = sum over packed words of
// fma(dot8(x, q - 8), scale[group, n], sum) in f32 and round to bf16.
//
// Here each 4-bit code is turned into the bf16 value 128 + q with one and-or
// per two codes (bf16 0x4300 | q), the MFMA contracts x against those values,
// and a second MFMA against bf16 ones yields sum(x) over the same k, so that
//   sum_k x (q - z) = sum_k x (128 + q) - (128 + z) sum_k x
// per group, which is then scaled by the group scale.  Products are exact in
// f32; only the accumulation order differs from the shader.
//
// MFMA v_mfma_f32_16x16x32_bf16: lane (g = l/16, r = l%16) supplies 8 bf16 of
// A row r and of B column r for its k-slice; both operands are loaded in the
// same per-lane k order, so A/B pairing is the identity.  Result lane (g, r)
// holds D[4g+i][r].
#include <algorithm>

#include "int4_dev.h"

namespace {

// GPTQ layout: qweight [K/8, N].  A wave owns 16 J columns (J MFMA column
// tiles; lane r takes columns n0 + J r .. n0 + J r + J - 1 so one load feeds
// all J) and 16 tokens; the block's KS waves split the groups.
template <int KS, int J, uint32_t GQ_BATCH>
__global__ __launch_bounds__(64 * KS) void int4_gptq_kernel(Int4Args A) {
    __shared__ v4f part[KS][J][64];
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t g = lane >> 4, rr = lane & 15;
    // XCD-aware order: the hardware deals consecutive workgroups to the 8
    // XCDs in turn; remapping gives each XCD a contiguous run of column tiles
    // so partial cache lines shared by neighbouring tiles hit its L2.  The
    // grid is padded to a multiple of 8; padding blocks exit.
    const uint32_t per_xcd = gridDim.x / 8;
    const uint32_t tile = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    const uint32_t n0 = tile * (16 * J);
    if (n0 >= A.N) return;
    const uint32_t m0 = blockIdx.y * 16;
    const uint32_t tok = m0 + rr;
    const uint32_t ngroups = A.K / A.G, steps = A.G / 32;
    const uint32_t per = (ngroups + KS - 1) / KS;
    const uint32_t g0 = min(ngroups, wave * per), g1 = min(ngroups, g0 + per);
    const uint32_t col = n0 + J * rr;
    const bool tv = tok < A.B;
    const uint16_t* xrow = A.x + (uint64_t)(tv ? tok : 0) * A.K;
    v4f acc[J], ag[J];
#pragma unroll
    for (int j = 0; j < J; j++) acc[j] = ag[j] = v4f{0.f, 0.f, 0.f, 0.f};
    v4f as = v4f{0.f, 0.f, 0.f, 0.f};
    // The wave's 32-k steps run in batches of GQ_BATCH: every weight and
    // activation load of a batch is issued before its first MFMA, so the wave
    // waits for memory once per batch.  A group's partial sums are scaled and
    // folded into acc when its last step has been contracted.
    const uint32_t first = g0 * steps, last = g1 * steps;
    for (uint32_t base = first; base < last; base += GQ_BATCH) {
        uint32_t wbuf[GQ_BATCH][J], zbuf[GQ_BATCH];
        uint16_t sbuf[GQ_BATCH][J];
        v4i abuf[GQ_BATCH];
#pragma clang loop unroll(full)
        for (uint32_t u = 0; u < GQ_BATCH; u++) {
            const uint32_t i = min(base + u, last - 1);
            const uint32_t kb = i * 32;
            const uint32_t p = kb / 8 + g;
            load_words<J>(A.qw + (uint64_t)p * A.N + col, wbuf[u]);
            abuf[u] = tv ? *reinterpret_cast<const v4i*>(xrow + kb + 8 * g) : v4i{0, 0, 0, 0};
            // The group's scales and zero codes ride with its last step, so
            // the fold below does not wait on a dependent load.
            if ((i + 1) % steps == 0) {
                const uint32_t grp = i / steps;
                const uint16_t* sp = A.scales + (uint64_t)grp * A.N + col;
#pragma unroll
                for (int j = 0; j < J; j++) sbuf[u][j] = sp[j];
                zbuf[u] = A.qzeros ? A.qzeros[(uint64_t)grp * (A.N / 8) + col / 8] >> (4 * (col % 8)) : 0x8888u;
            }
        }
#pragma clang loop unroll(full)
        for (uint32_t u = 0; u < GQ_BATCH; u++) {
            const uint32_t i = base + u;
            if (i >= last) continue;
            v4i ap = permute_act(abuf[u]);
#pragma unroll
            for (int j = 0; j < J; j++) ag[j] = mfma_bf16(ap, dequant_word(wbuf[u][j]), ag[j]);
            as = mfma_bf16(ap, v4i{(int)ONES_BF16, (int)ONES_BF16, (int)ONES_BF16, (int)ONES_BF16}, as);
            if ((i + 1) % steps == 0) {
                const uint32_t zw = zbuf[u];
#pragma unroll
                for (int j = 0; j < J; j++) {
                    float sc = decode_scale(sbuf[u][j], A.scale_bf16);
                    float off = 128.0f + (float)((zw >> (4 * j)) & 15u);
#pragma unroll
                    for (int q = 0; q < 4; q++) acc[j][q] = fmaf(sc, ag[j][q] - off * as[q], acc[j][q]);
                    ag[j] = v4f{0.f, 0.f, 0.f, 0.f};
                }
                as = v4f{0.f, 0.f, 0.f, 0.f};
            }
        }
    }
#pragma unroll
    for (int j = 0; j < J; j++) part[wave][j][lane] = acc[j];
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int j = 0; j < J; j++) {
        v4f t = part[0][j][lane];
#pragma unroll
        for (int w = 1; w < KS; w++) t += part[w][j][lane];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t tt = m0 + 4 * g + i;
            if (tt < A.B) finalize_store(A, tt, col + j, t[i]);
        }
    }
}

// GPTQ layout with the group length fixed at compile time (STEPS = G / 32).
// Same tile and lane mapping as int4_gptq_kernel; a load batch holds GPB whole
// groups (GPB * STEPS 32-k steps), so the per-group fold needs no per-step
// test, and the wave's group range is derived from a scalar wave index so
// that all step and group addressing stays on the scalar unit.
template <int KS, int J, int STEPS>
__global__ __launch_bounds__(64 * KS) void int4_gptq_fixed_kernel(Int4Args A) {
    constexpr int GPB = STEPS >= 8 ? 1 : 8 / STEPS;
    __shared__ v4f part[KS][J][64];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t g = lane >> 4, rr = lane & 15;
    const uint32_t per_xcd = gridDim.x / 8;
    const uint32_t tile = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    const uint32_t n0 = tile * (16 * J);
    if (n0 >= A.N) return;
    const uint32_t m0 = blockIdx.y * 16;
    const uint32_t tok = m0 + rr;
    const uint32_t N = A.N;
    const uint32_t ngroups = A.K / (32 * STEPS);
    const uint32_t per = (ngroups + KS - 1) / KS;
    const uint32_t g0 = min(ngroups, wave * per), g1 = min(ngroups, g0 + per);
    const uint32_t col = n0 + J * rr;
    const bool tv = tok < A.B;
    // Lane bases: packed row 4 i + g of step i is wq + i * 4 N; activations
    // of step i start at xq + 32 i.
    const uint32_t* wq = A.qw + (uint64_t)g * N + col;
    const uint16_t* xq = A.x + (uint64_t)(tv ? tok : 0) * A.K + 8 * g;
    const uint16_t* sq = A.scales + col;
    const uint32_t* zq = A.qzeros ? A.qzeros + col / 8 : nullptr;
    const uint32_t zshift = 4 * (col % 8);
    v4f acc[J];
#pragma unroll
    for (int j = 0; j < J; j++) acc[j] = v4f{0.f, 0.f, 0.f, 0.f};
    const v4i ones = v4i{(int)ONES_BF16, (int)ONES_BF16, (int)ONES_BF16, (int)ONES_BF16};
    for (uint32_t grp = g0; grp < g1; grp += GPB) {
        uint32_t wbuf[GPB][STEPS][J], zbuf[GPB];
        uint16_t sbuf[GPB][J];
        v4i abuf[GPB][STEPS];
#pragma unroll
        for (int gb = 0; gb < GPB; gb++) {
            const uint32_t gi = min(grp + gb, g1 - 1);
#pragma unroll
            for (int st = 0; st < STEPS; st++) {
                const uint32_t i = gi * STEPS + st;
                load_words<J>(wq + (uint64_t)i * 4 * N, wbuf[gb][st]);
                abuf[gb][st] = tv ? *reinterpret_cast<const v4i*>(xq + 32 * i) : v4i{0, 0, 0, 0};
            }
#pragma unroll
            for (int j = 0; j < J; j++) sbuf[gb][j] = sq[(uint64_t)gi * N + j];
            zbuf[gb] = zq ? zq[(uint64_t)gi * (N / 8)] >> zshift : 0x8888u;
        }
#pragma unroll
        for (int gb = 0; gb < GPB; gb++) {
            if (grp + gb >= g1) continue;
            v4f ag[J], as = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < J; j++) ag[j] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int st = 0; st < STEPS; st++) {
                v4i ap = permute_act(abuf[gb][st]);
#pragma unroll
                for (int j = 0; j < J; j++) ag[j] = mfma_bf16(ap, dequant_word(wbuf[gb][st][j]), ag[j]);
                as = mfma_bf16(ap, ones, as);
            }
#pragma unroll
            for (int j = 0; j < J; j++) {
                const float sc = decode_scale(sbuf[gb][j], A.scale_bf16);
                const float off = 128.0f + (float)((zbuf[gb] >> (4 * j)) & 15u);
#pragma unroll
                for (int q = 0; q < 4; q++) acc[j][q] = fmaf(sc, ag[j][q] - off * as[q], acc[j][q]);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < J; j++) part[wave][j][lane] = acc[j];
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int j = 0; j < J; j++) {
        v4f t = part[0][j][lane];
#pragma unroll
        for (int w = 1; w < KS; w++) t += part[w][j][lane];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t tt = m0 + 4 * g + i;
            if (tt < A.B) finalize_store(A, tt, col + j, t[i]);
        }
    }
}

// Decode-sized GPTQ linear (M <= GEMV_MAX_M tokens).  The kernel is shaped
// for the weight stream: a block owns 64 columns and its 16 waves split the
// packed rows in batches of 32, each wave issuing every load of its batch up
// front.  Weights are read 16 bytes per lane: lane (q = l / 16, c = l % 16)
// loads columns 4c..4c+3 of packed rows 4i + q (i = 0..7) of the batch, so one
// load instruction covers four whole 256-byte row segments (a dword per lane
// would take four times the instructions and memory requests for the bytes).
//
// The loaded words are exactly the B operand of v_mfma_f32_16x16x32_bf16
// (lane (q, c) = k-slice q of column c) once each 4-bit code is turned into
// the bf16 value 128 + q (one and-or per two codes), so MFMA j of step i
// contracts columns 4c + j; A row c is token min(c, M - 1), and only result
// rows t < M are read.  The matrix core does the multiply-adds that would
// otherwise cost four v_dot2 per word per token; the vector ALU is left with
// the code expansion.  As in the other kernels
//   sum_k x (q - z) = sum_k x (128 + q) - (128 + z) sum_k x
// per group, with sum_k x from shuffles over the activation slice.
//
// Loads go oldest first in the order they are needed (the wave's activation
// slice, group scales and zero codes, then the packed words), so the wave
// waits for the slice alone and then contracts each load as it lands.  The
// slice is permuted into pair order and parked in the wave's own LDS region;
// the 16 waves' partial sums meet in LDS.
constexpr uint32_t GEMV_MAX_M = 4;
constexpr uint32_t GEMV_ROWS = 32;       // packed rows per wave batch (256 k)

__device__ __forceinline__ float sum8_bf16(v4i v) {
    float s = 0.f;
#pragma unroll
    for (int q = 0; q < 4; q++)
        s += bf16_to_f32((uint16_t)((uint32_t)v[q] & 0xFFFFu)) + bf16_to_f32((uint16_t)((uint32_t)v[q] >> 16));
    return s;
}

template <int KS, int G, bool ZP, uint32_t MT, bool SPLIT>
__global__ __launch_bounds__(64 * KS) void int4_gptq_gemv_kernel(Int4Args A, float* split_part, uint32_t span) {
    constexpr uint32_t GR = G / 8;                 // packed rows per group
    constexpr uint32_t GPB = GEMV_ROWS / GR;       // groups per batch
    constexpr uint32_t LR = GEMV_ROWS / 4;         // packed rows per lane per batch
    static_assert(GR % 4 == 0 && GR <= GEMV_ROWS && GEMV_ROWS % GR == 0, "group length must divide the batch");
    __shared__ v4i xw[KS][MT][GEMV_ROWS];
    __shared__ v4f part[KS][MT][16];
    const uint32_t K = A.K, N = A.N, M = A.B, prow = K / 8;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63, lr = lane & (GEMV_ROWS - 1);
    const uint32_t q = lane >> 4, c = lane & 15;
    const uint32_t per_xcd = gridDim.x / 8;
    const uint32_t tile = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    const uint32_t n0 = tile * 64;
    if (n0 >= N) return;
    const uint32_t col = n0 + 4 * c;               // first of the lane's 4 columns
    const uint32_t ngroups = K / G;
    // The batches of K, or this split's `span` of them, dealt to the waves.
    const uint32_t batches = (ngroups + GPB - 1) / GPB;
    const uint32_t s0 = SPLIT ? blockIdx.y * span : 0u, nbatch = SPLIT ? min(batches, s0 + span) : batches;
    const uint32_t per = (nbatch - s0 + KS - 1) / KS;
    const uint32_t b0 = min(nbatch, s0 + wave * per), b1 = min(nbatch, b0 + per);
    const uint32_t zshift = 4 * (col % 8);
    v4f acc[MT];
#pragma unroll
    for (uint32_t t = 0; t < MT; t++) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
    for (uint32_t b = b0; b < b1; b++) {
        const uint32_t grp0 = b * GPB, row0 = grp0 * GR;
        // Loads, oldest first.
        v4i xl[MT];
#pragma unroll
        for (uint32_t t = 0; t < MT; t++)
            xl[t] = *reinterpret_cast<const v4i*>(A.x + (uint64_t)min(t, M - 1) * K + 8 * min(row0 + lr, prow - 1));
        v2i sb[GPB];
        uint32_t zb[GPB];
#pragma unroll
        for (uint32_t gb = 0; gb < GPB; gb++) {
            const uint32_t gi = min(grp0 + gb, ngroups - 1);
            sb[gb] = *reinterpret_cast<const v2i*>(A.scales + (uint64_t)gi * N + col);
            zb[gb] = ZP ? A.qzeros[(uint64_t)gi * (N / 8) + col / 8] >> zshift : 0x8888u;
        }
        // Scheduling fences keep the issue order (the compiler would otherwise
        // hoist the packed-word loads ahead and then drain them all for the
        // slice).
        __builtin_amdgcn_sched_barrier(0);
        v4i w[LR];
#pragma unroll
        for (uint32_t i = 0; i < LR; i++)
            w[i] = *reinterpret_cast<const v4i*>(A.qw + (uint64_t)min(row0 + 4 * i + q, prow - 1) * N + col);
        __builtin_amdgcn_sched_barrier(0);
        // Activation slice: pair order into LDS (lane lr holds row row0 + lr;
        // lanes 32..63 mirror lanes 0..31), and per-group sums of the slice.
        float gsum[MT][GPB];
#pragma unroll
        for (uint32_t t = 0; t < MT; t++) {
            if (lane < GEMV_ROWS) xw[wave][t][lr] = permute_act(xl[t]);
            float v = sum8_bf16(xl[t]);
            v = lanes_sum_up<GR>(v);   // the __shfl_xor butterfly 1, 2, ..., GR / 2
#pragma unroll
            for (uint32_t gb = 0; gb < GPB; gb++) gsum[t][gb] = lane_bcast(v, gb * GR);
        }
        __builtin_amdgcn_wave_barrier();
        // MFMA j of step i contracts packed rows 4 i .. 4 i + 3 (k-slice q)
        // of columns 4 c + j against the activations: A row c is token
        // min(c, M - 1), so result rows t < M are the tokens and the rest are
        // never read.  Result lane (0, c) holds D[t][4 c + j] in element t.
        const uint32_t tsel = min(c, M - 1);
#pragma unroll
        for (uint32_t gb = 0; gb < GPB; gb++) {
            if (grp0 + gb >= ngroups) continue;
            v4f ag[4];
#pragma unroll
            for (uint32_t j = 0; j < 4; j++) ag[j] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (uint32_t i = gb * (GR / 4); i < (gb + 1) * (GR / 4); i++) {
                const v4i xv = xw[wave][tsel][4 * i + q];
#pragma unroll
                for (uint32_t j = 0; j < 4; j++) ag[j] = mfma_bf16(xv, dequant_word((uint32_t)w[i][j]), ag[j]);
            }
#pragma unroll
            for (uint32_t j = 0; j < 4; j++) {
                const uint32_t sbits = (uint32_t)sb[gb][j / 2] >> (16 * (j % 2));
                const float sc = decode_scale((uint16_t)(sbits & 0xFFFFu), A.scale_bf16);
                const float off = 128.0f + (float)((zb[gb] >> (4 * j)) & 15u);
#pragma unroll
                for (uint32_t t = 0; t < MT; t++) acc[t][j] = fmaf(sc, ag[j][t] - off * gsum[t][gb], acc[t][j]);
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (uint32_t t = 0; t < MT; t++)
        if (lane < 16) part[wave][t][lane] = acc[t];
    __syncthreads();
    if (wave != 0) return;
    const float* pf = reinterpret_cast<const float*>(&part[0][0][0]);
    for (uint32_t t = 0; t < M; t++) {
        float v = pf[t * 64 + lane];
#pragma unroll
        for (int w2 = 1; w2 < KS; w2++) v += pf[(w2 * MT + t) * 64 + lane];
        if (SPLIT) split_part[((uint64_t)blockIdx.y * M + t) * N + n0 + lane] = v;
        else finalize_store(A, t, n0 + lane, v);
    }
}

// CT layout: qweight [N, K/8], scales [N, K/G], G % 128 == 0.  A block owns 16 J
// rows of weights (output columns) and 16 tokens; its KS waves split the 128-k
// steps of K in batches of four (512 columns).  A batch's weights are read 256
// contiguous bytes per row (lane l: 16-byte piece l % 16 of rows l / 16 + 4 i),
// nontemporal when one token tile reads them, pass through a wave-private LDS
// slot (rows padded by 16 bytes: operand reads of 16 rows hit distinct banks)
// and come back as lane (g, r)'s 4 consecutive words of row r (k-slices 4g..4g+3
// of a step); MFMA j contracts slice 4g+j of every lane group.
//
// Bound: the weight stream; from about 8 tokens on the activation rows each
// block re-reads (J = 2 halves them).  One register set and 16 waves a CU
// (<= 128 registers) stream better than two sets and 8: 4096 x 14336, one token
// 12.6 us against 15.5; 16.1 when the weights were read in the operand layout
// (64 bytes per row and instruction) and the scales at the fold.  J = 2 needs 144
// registers (held to 128 it spills: 16 tokens 21.0 us against 17.7; 25.6 before).
// 14336 x 4096, one token: 17.1 -> 11.5.
constexpr uint32_t CT_BATCH = 4;
constexpr uint32_t CT_STRIDE = CT_BATCH * 64 + 16;

template <int KS, int J>
__global__ __launch_bounds__(64 * KS, J == 1 ? 4 : 2) void int4_ct_kernel(Int4Args A) {
    __shared__ __attribute__((aligned(16))) uint8_t slots[KS][J * 16 * CT_STRIDE];   // then the wave's partial sums
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t g = lane >> 4, rr = lane & 15;
    const uint32_t n0 = blockIdx.x * 16 * J, m0 = blockIdx.y * 16;
    const uint32_t tok = m0 + rr;
    const uint32_t ngroups = A.K / A.G, steps = A.G / 128, nstep = A.K / 128;
    const uint32_t per = (nstep + KS - 1) / KS;
    const uint32_t first = min(nstep, wave * per), last = min(nstep, first + per);
    const bool tv = tok < A.B;
    const uint16_t* xrow = A.x + (uint64_t)(tv ? tok : 0) * A.K + 32 * g;
    const uint32_t* wrow = A.qw + (uint64_t)(n0 + g) * (A.K / 8);          // row l / 16 of the load pattern
    const uint16_t* srow = A.scales + (uint64_t)(n0 + rr) * ngroups;
    const uint32_t exponent = pair_exponent();
    uint8_t* slot = slots[wave];
    struct Batch {
        v4i w[J][4], a[CT_BATCH][4];
        uint16_t s[J][CT_BATCH];
    };
    auto load = [&](Batch& B, uint32_t base) __attribute__((always_inline)) {
        const uint32_t pc = min(base * 4 + rr, last * 4 - 1);
#pragma unroll
        for (int j = 0; j < J; j++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const v4i* p = reinterpret_cast<const v4i*>(wrow + (uint64_t)(16 * j + 4 * i) * (A.K / 8) + pc * 4);
                B.w[j][i] = gridDim.y == 1 ? __builtin_nontemporal_load(p) : *p;
            }
#pragma unroll
        for (uint32_t u = 0; u < CT_BATCH; u++) {
            const uint32_t i = min(base + u, last - 1);
#pragma unroll
            for (int j = 0; j < 4; j++) B.a[u][j] = tv ? *reinterpret_cast<const v4i*>(xrow + i * 128 + 8 * j) : v4i{0, 0, 0, 0};
#pragma unroll
            for (int j = 0; j < J; j++) B.s[j][u] = srow[(uint64_t)(16 * j) * ngroups + i / steps];
        }
    };
    v4f acc[J];
#pragma unroll
    for (int j = 0; j < J; j++) acc[j] = v4f{0.f, 0.f, 0.f, 0.f};
    const v4i ones = v4i{(int)ONES_BF16, (int)ONES_BF16, (int)ONES_BF16, (int)ONES_BF16};
    auto contract = [&](Batch& B, uint32_t base) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < J; j++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                *reinterpret_cast<v4i*>(slot + (16 * j + 4 * i + g) * CT_STRIDE + rr * 16) = B.w[j][i];
        __builtin_amdgcn_wave_barrier();
        // A step's sums are folded by its own scale (a group's steps share one).
#pragma unroll
        for (uint32_t u = 0; u < CT_BATCH; u++) {
            if (base + u >= last) break;
            v4i ap[4];
            v4f as = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < 4; q++) {
                ap[q] = permute_act(B.a[u][q]);
                as = mfma_bf16(ap[q], ones, as);
            }
#pragma unroll
            for (int j = 0; j < J; j++) {
                const v4i w = *reinterpret_cast<const v4i*>(slot + (16 * j + rr) * CT_STRIDE + (4 * u + g) * 16);
                v4f ag = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int q = 0; q < 4; q++) ag = mfma_bf16(ap[q], dequant_word((uint32_t)w[q], exponent), ag);
                const float sc = decode_scale(B.s[j][u], A.scale_bf16);
#pragma unroll
                for (int i = 0; i < 4; i++) acc[j][i] = fmaf(sc, ag[i] - 136.0f * as[i], acc[j][i]);
            }
        }
        __builtin_amdgcn_wave_barrier();
    };
    Batch p;
    for (uint32_t base = first; base < last; base += CT_BATCH) {
        load(p, base);
        contract(p, base);
    }
#pragma unroll
    for (int j = 0; j < J; j++) reinterpret_cast<v4f*>(slot)[j * 64 + lane] = acc[j];
    __syncthreads();
    if (wave >= J) return;
    v4f t = reinterpret_cast<const v4f*>(slots[0])[wave * 64 + lane];
#pragma unroll
    for (int w = 1; w < KS; w++) t += reinterpret_cast<const v4f*>(slots[w])[wave * 64 + lane];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t tt = m0 + 4 * g + i;
        if (tt < A.B) finalize_store(A, tt, n0 + 16 * wave + rr, t[i]);
    }
}

// ---------------------------------------------------------------------------
// Pair-packed INT8 activations (quantize_int8_symmetric_pairpacked.comp.
// template:22-72): per 32 columns s = amax > 0 ? amax / 127 : 1,
// q = round-half-even(clamp(x / s, -127, 127)) and the block sum of q.  A
// thread owns 8 columns c..c+7 and writes the words (q[c], q[c+2], q[c+4],
// q[c+6]) and (q[c+1], q[c+3], q[c+5], q[c+7]); the 4 threads of a block are
// consecutive lanes.
// ---------------------------------------------------------------------------
// SILU: silu_multiply_quantize_int8_pairpacked.comp.template: the values are
// y = bf16(bf16(g / (1 + exp(-g))) * u) of the gate (x) and up rows, and y is
// written out as well.
template <bool SILU, bool PAIRED = true>
__global__ __launch_bounds__(256) void quant_i8pp_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ up,
                                                         uint16_t* __restrict__ y, uint32_t rows, uint32_t cols,
                                                         uint32_t* __restrict__ q, float* __restrict__ s,
                                                         int32_t* __restrict__ sums) {
    const uint32_t oct = blockIdx.x * 256 + threadIdx.x, per_row = cols / 8;
    const bool ok = oct < rows * per_row;
    const uint32_t o = ok ? oct : 0u;
    const v4i v = *reinterpret_cast<const v4i*>(x + (uint64_t)o * 8);
    float f[8];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        f[2 * e] = bf16_to_f32((uint32_t)v[e]);
        f[2 * e + 1] = bf16_to_f32((uint32_t)v[e] >> 16);
    }
    if (SILU) {
        const v4i uv = *reinterpret_cast<const v4i*>(up + (uint64_t)o * 8);
        uint32_t yb[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float act = round_bf16(f[e] / (1.0f + expf(-f[e])));
            yb[e] = f32_to_bf16(act * bf16_to_f32((uint32_t)uv[e / 2] >> (16 * (e & 1)))) & 0xffffu;
            f[e] = bf16_to_f32(yb[e]);
        }
        if (ok)
            *reinterpret_cast<v4i*>(y + (uint64_t)o * 8) = v4i{(int)(yb[0] | (yb[1] << 16)), (int)(yb[2] | (yb[3] << 16)),
                                                               (int)(yb[4] | (yb[5] << 16)), (int)(yb[6] | (yb[7] << 16))};
    }
    float m = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; e++) m = fmaxf(m, fabsf(f[e]));
    m = fmaxf(m, __shfl_xor(m, 1));
    m = fmaxf(m, __shfl_xor(m, 2));
    const float sc = m > 0.0f ? m / 127.0f : 1.0f;
    int iv[8], sum = 0;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        iv[e] = (int)__builtin_rintf(fminf(fmaxf(f[e] / sc, -127.0f), 127.0f));
        sum += iv[e];
    }
    sum += __shfl_xor(sum, 1);
    sum += __shfl_xor(sum, 2);
    if (!ok) return;
    // pair-packed: (q[c], q[c+2], q[c+4], q[c+6]), (q[c+1], ...); unpaired:
    // the 8 codes in column order
    const int a0 = PAIRED ? 0 : 0, a1 = PAIRED ? 2 : 1, a2 = PAIRED ? 4 : 2, a3 = PAIRED ? 6 : 3;
    const int b0 = PAIRED ? 1 : 4, b1 = PAIRED ? 3 : 5, b2 = PAIRED ? 5 : 6, b3 = PAIRED ? 7 : 7;
    const uint32_t w0 = (uint32_t)(iv[a0] & 255) | ((uint32_t)(iv[a1] & 255) << 8) | ((uint32_t)(iv[a2] & 255) << 16) |
                        ((uint32_t)(iv[a3] & 255) << 24);
    const uint32_t w1 = (uint32_t)(iv[b0] & 255) | ((uint32_t)(iv[b1] & 255) << 8) | ((uint32_t)(iv[b2] & 255) << 16) |
                        ((uint32_t)(iv[b3] & 255) << 24);
    *reinterpret_cast<uint2*>(q + (uint64_t)o * 2) = uint2{w0, w1};
    if ((o & 3u) == 0) {
        s[o / 4] = sc;
        if (sums) sums[o / 4] = sum;
    }
}

// ---------------------------------------------------------------------------
// Pair-packed INT8 x GPTQ INT4 linear (linear_prequant_pairpacked_int4_gptq.
// comp.template:56-95).  Lane = output column (64 per block), the 4 waves
// split the weight groups; per 32-column block the integer dot is exact
// (v_dot4_i32_i8 on the bytes (q - 0) of the packed word's low and high
// nibbles against the even and odd activation words, minus 8 times the block
// sum), then acc = fma(dot, s_x * s_w, acc).  Only the f32 accumulation order
// differs from the shader (per-wave partials added in wave order).
// ---------------------------------------------------------------------------
// Unpaired input (linear_prequant_int4_{gptq,ct}.comp.template): the int8
// words hold columns in order, so each packed weight word becomes the signed
// bytes (code - 8) of nibbles 0..3 and 4..7 for two v_dot4_i32_i8.
__device__ __forceinline__ int nibbles_to_i8x4(uint32_t t16) {
    uint32_t b = (t16 & 0xFu) | ((t16 & 0xF0u) << 4) | ((t16 & 0xF00u) << 8) | ((t16 & 0xF000u) << 12);
    b ^= 0x08080808u;                       // code - 8 as a 4-bit two's complement value
    return (int)(b | ((b & 0x08080808u) * 0x1Eu));   // sign-extend each byte
}

template <bool PAIRED, bool CT>
__global__ __launch_bounds__(256) void int4_pp_kernel(PpArgs P) {
    __shared__ float red[4][64];
    const Int4Args& A = P.L;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t K = A.K, N = A.N, G = A.G, ngroups = K / G, bpg = G / 32, nblk = K / 32;
    const uint32_t n = blockIdx.x * 64 + lane;
    const uint32_t nc = n < N ? n : N - 1;
    const uint32_t per = (ngroups + 3) / 4, g0 = min(ngroups, wave * per), g1 = min(ngroups, g0 + per);
    for (uint32_t t = 0; t < A.B; t++) {
        const uint32_t* qt = P.q + (uint64_t)t * (K / 4);
        float acc = 0.0f;
        for (uint32_t g = g0; g < g1; g++) {
            const float sw = decode_scale(CT ? A.scales[(uint64_t)nc * ngroups + g] : A.scales[(uint64_t)g * N + nc],
                                          A.scale_bf16);
            for (uint32_t b = g * bpg; b < (g + 1) * bpg; b++) {
                int dot = PAIRED ? -8 * P.sums[(uint64_t)t * nblk + b] : 0;
#pragma unroll
                for (uint32_t p = 0; p < 4; p++) {
                    const uint32_t word = CT ? A.qw[(uint64_t)nc * (K / 8) + b * 4 + p] : A.qw[(uint64_t)(b * 4 + p) * N + nc];
                    if (PAIRED) {
                        dot = __builtin_amdgcn_sdot4((int)qt[(b * 4 + p) * 2], (int)(word & 0x0f0f0f0fu), dot, false);
                        dot = __builtin_amdgcn_sdot4((int)qt[(b * 4 + p) * 2 + 1], (int)((word >> 4) & 0x0f0f0f0fu), dot,
                                                     false);
                    } else {
                        dot = __builtin_amdgcn_sdot4((int)qt[(b * 4 + p) * 2], nibbles_to_i8x4(word & 0xffffu), dot, false);
                        dot = __builtin_amdgcn_sdot4((int)qt[(b * 4 + p) * 2 + 1], nibbles_to_i8x4(word >> 16), dot, false);
                    }
                }
                acc = fmaf((float)dot, P.s[(uint64_t)t * nblk + b] * sw, acc);
            }
        }
        red[wave][lane] = acc;
        __syncthreads();
        if (wave == 0 && n < N) finalize_store(A, t, n, ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane]);
        __syncthreads();
    }
}


// ---------------------------------------------------------------------------
// The same linears on the integer matrix cores: v_mfma_i32_16x16x32_i8
// contracts exactly one 32-column activation block, so its int32 result is
// the block's exact dot and each block is folded as acc_g = fma(dot, s_x,
// acc_g), a segment of blocks that share a weight scale as acc = fma(acc_g,
// s_w, acc), s_x times I8_SCALE_DOWN.
//
// A wave owns 16 J columns and 16 MT tokens and the block's KS waves split the
// blocks of K.  Operands: lane (g = l / 16, r = l % 16) supplies 8 bytes of
// token r and of column r; the k order inside a block is free as long as both
// agree.  Activations are read 16 bytes per lane (octets 2g, 2g+1 of 64
// columns) and one v_permlane32_swap per dword deals them to the two blocks,
// which leaves octet pi(g) = (0, 2, 1, 3)[g] on lane group g; the packed words
// are read from row 4 b + pi(g) (GPTQ: J columns per load).  A word's nibbles
// 0, 2, 4, 6 and 1, 3, 5, 7 are already the byte order of pair-packed
// activations (column-order ones are brought into it with two v_perm); code - 8
// per byte is ((w & 0x0f0f0f0f) + 0x78787878) ^ 0x80808080, so the block sums
// are not needed.  The activation scales of a load batch pass through a
// wave-private LDS slice that transposes them to result rows.
//
// Bound: the weight stream and, from about 32 tokens on, the activation rows
// every column tile re-reads from L2.  One token of 4096 x 14336: 11.0 us a
// launch (31.3 with a lane per column), of 14336 x 4096 13.4 us; a feed-forward
// of 30 tokens 1782 -> 62 us.  Up to four tokens the conversion and fold of all
// 16 result rows is the larger part: RT = 1 gives each lane group one token
// (operand rows 4 t .. 4 t + 3 repeat token t) and folds one row in four: 9.3
// and 12.0 us.
// ---------------------------------------------------------------------------
template <int MT, int J, int KS, int U, int BPG, bool PAIRED, bool CT, int RT>
__global__ __launch_bounds__(64 * KS) void int4_i8_kernel(PpArgs P, uint32_t tgroups, float* split_part, uint32_t per) {
    static_assert(U % 2 == 0 && U % BPG == 0, "a batch holds whole 64-column pairs and scale segments");
    static_assert(!CT || (J == 1 && U % 4 == 0), "CT rows are read 128 columns at a time");
    static_assert(RT == 4 || MT == 1, "one token per lane group: at most four tokens");
    constexpr int TOK = 4 * RT * MT;                  // tokens of the block
    constexpr int NV = (TOK * U + 63) / 64;           // activation scales per lane and batch
    __shared__ __attribute__((aligned(16))) float xs[KS][U][TOK];
    __shared__ __attribute__((aligned(16))) float part[KS][J][64][RT];
    const Int4Args& A = P.L;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t g = lane >> 4, rr = lane & 15, pg = ((g & 1) << 1) | (g >> 1);
    const uint32_t K = A.K, N = A.N, M = A.B, nblk = K / 32;
    // Token groups fastest within an XCD's run of column tiles, so the groups
    // of a tile read its weights through one L2.
    const uint32_t per_xcd = gridDim.x / 8 / tgroups, seq = blockIdx.x / 8;
    const uint32_t tile = (blockIdx.x % 8) * per_xcd + seq / tgroups;
    const uint32_t n0 = tile * (16 * J), m0 = (seq % tgroups) * TOK;
    if (n0 >= N) return;
    // `per` blocks of K a wave: whole units of a load (CT), an activation pair or a
    // scale segment.
    const uint32_t b0 = min(nblk, (blockIdx.y * KS + wave) * per), b1 = min(nblk, b0 + per);
    const uint32_t col = n0 + J * rr;
    const uint32_t ngroups = K / A.G;

    struct Batch {
        v4i a[MT][U / 2];
        uint32_t w[U][J];
        uint16_t sw[U / BPG][J];
        float sx[NV];
    };
    const uint8_t* arow[MT];
#pragma unroll
    for (int m = 0; m < MT; m++)
        arow[m] = reinterpret_cast<const uint8_t*>(P.q) + (uint64_t)min(m0 + 4 * RT * m + rr * RT / 4, M - 1) * K + 16 * g;
    // Loads past the wave's range repeat its last pair; their scales are zero.
    auto load = [&](Batch& B, uint32_t b) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            if constexpr (CT) {
                if (u % 4 == 0) {
                    // 4 words of one block per lane, clamped into the row (K % 128 may be 64).
                    const uint32_t bb = min(b + u + g, nblk - 1);
                    const v4i v = *reinterpret_cast<const v4i*>(A.qw + (uint64_t)col * (K / 8) + bb * 4);
                    B.w[u][0] = (uint32_t)v.x; B.w[u + 1][0] = (uint32_t)v.y;
                    B.w[u + 2][0] = (uint32_t)v.z; B.w[u + 3][0] = (uint32_t)v.w;
                }
            } else {
                const uint32_t bb = min(b + u, b1 - 1);
                load_words<J>(A.qw + (uint64_t)(bb * 4 + pg) * N + col, B.w[u]);
            }
        }
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int c = 0; c < U / 2; c++)
                B.a[m][c] = *reinterpret_cast<const v4i*>(arow[m] + min(b + 2 * c, b1 - 2) * 32);
#pragma unroll
        for (int s = 0; s < U / BPG; s++) {
            const uint32_t grp = min(b + s * BPG, b1 - 1) * 32 / A.G;
#pragma unroll
            for (int j = 0; j < J; j++)
                B.sw[s][j] = CT ? A.scales[(uint64_t)(col + j) * ngroups + grp] : A.scales[(uint64_t)grp * N + col + j];
        }
#pragma unroll
        for (int v = 0; v < NV; v++) {
            const uint32_t i = v * 64 + lane, t = min(m0 + i / U, M - 1), bb = b + i % U;
            const float s = P.s[(uint64_t)t * nblk + min(bb, b1 - 1)];
            B.sx[v] = bb < b1 ? s * I8_SCALE_DOWN : 0.0f;
        }
    };
    typedef float rows_t __attribute__((ext_vector_type(RT)));
    rows_t acc[MT][J];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int j = 0; j < J; j++) acc[m][j] = rows_t(0.f);
    auto contract = [&](Batch& B) __attribute__((always_inline)) {
#pragma unroll
        for (int v = 0; v < NV; v++) {
            const uint32_t i = v * 64 + lane;
            if (TOK * U % 64 == 0 || i < TOK * U) xs[wave][i % U][i / U] = B.sx[v];
        }
        __builtin_amdgcn_wave_barrier();
        if constexpr (CT) {
            // Lane group g holds the 4 words of block u + g: transposed so
            // that lane group g holds word pi(g) of each block in turn.
#pragma unroll
            for (int u = 0; u < U; u += 4) {
                const auto x = __builtin_amdgcn_permlane32_swap(B.w[u][0], B.w[u + 1][0], false, false);
                const auto y = __builtin_amdgcn_permlane32_swap(B.w[u + 2][0], B.w[u + 3][0], false, false);
                const auto p = __builtin_amdgcn_permlane16_swap(x[0], y[0], false, false);
                const auto q = __builtin_amdgcn_permlane16_swap(x[1], y[1], false, false);
                B.w[u][0] = p[0]; B.w[u + 1][0] = p[1]; B.w[u + 2][0] = q[0]; B.w[u + 3][0] = q[1];
            }
        }
        rows_t ag[MT][J];
#pragma unroll
        for (int u = 0; u < U; u++) {
            long bw[J];
#pragma unroll
            for (int j = 0; j < J; j++) {
                const uint32_t lo = ((B.w[u][j] & 0x0f0f0f0fu) + 0x78787878u) ^ 0x80808080u;
                const uint32_t hi = (((B.w[u][j] >> 4) & 0x0f0f0f0fu) + 0x78787878u) ^ 0x80808080u;
                bw[j] = (long)(((uint64_t)hi << 32) | lo);
            }
#pragma unroll
            for (int m = 0; m < MT; m++) {
                if (u % 2 == 0) {
                    v4i& v = B.a[m][u / 2];
                    if (!PAIRED) {
                        const uint32_t e0 = __builtin_amdgcn_perm((uint32_t)v.y, (uint32_t)v.x, 0x06040200u);
                        const uint32_t o0 = __builtin_amdgcn_perm((uint32_t)v.y, (uint32_t)v.x, 0x07050301u);
                        const uint32_t e1 = __builtin_amdgcn_perm((uint32_t)v.w, (uint32_t)v.z, 0x06040200u);
                        const uint32_t o1 = __builtin_amdgcn_perm((uint32_t)v.w, (uint32_t)v.z, 0x07050301u);
                        v = v4i{(int)e0, (int)o0, (int)e1, (int)o1};
                    }
                    const auto x = __builtin_amdgcn_permlane32_swap((uint32_t)v.x, (uint32_t)v.z, false, false);
                    const auto y = __builtin_amdgcn_permlane32_swap((uint32_t)v.y, (uint32_t)v.w, false, false);
                    v = v4i{(int)x[0], (int)y[0], (int)x[1], (int)y[1]};
                }
                const v4i& v = B.a[m][u / 2];
                const uint32_t a0 = (uint32_t)(u % 2 ? v.z : v.x), a1 = (uint32_t)(u % 2 ? v.w : v.y);
                const long av = (long)(((uint64_t)a1 << 32) | a0);
                const rows_t sx = *reinterpret_cast<const rows_t*>(&xs[wave][u][RT * (4 * m + g)]);
#pragma unroll
                for (int j = 0; j < J; j++) {
                    const v4i d = __builtin_amdgcn_mfma_i32_16x16x32_i8(av, bw[j], v4i{0, 0, 0, 0}, 0, 0, 0);
                    if (u % BPG == 0) ag[m][j] = rows_t(0.f);
#pragma unroll
                    for (int i = 0; i < RT; i++) ag[m][j][i] = fmaf((float)d[i], sx[i], ag[m][j][i]);
                    if (u % BPG == BPG - 1) {
                        const float sw = decode_scale(B.sw[u / BPG][j], A.scale_bf16);
#pragma unroll
                        for (int i = 0; i < RT; i++) acc[m][j][i] = fmaf(ag[m][j][i], sw, acc[m][j][i]);
                    }
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    };
    if (b0 < b1) {
        Batch p, q;
        load(p, b0);
        for (uint32_t b = b0; b < b1; b += 2 * U) {
            const bool two = b + U < b1;
            if (two) load(q, b + U);
            contract(p);
            if (!two) break;
            if (b + 2 * U < b1) load(p, b + 2 * U);
            contract(q);
        }
    }
    // The waves' partial sums meet in LDS one token tile at a time and are
    // added in wave order.
#pragma unroll
    for (int m = 0; m < MT; m++) {
        if (m0 + 4 * RT * m >= M) break;
#pragma unroll
        for (int j = 0; j < J; j++) *reinterpret_cast<rows_t*>(&part[wave][j][lane][0]) = acc[m][j];
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < 64 * RT * J; i += 64 * KS) {
            const uint32_t t = i / (16 * J), c = i % (16 * J), tt = m0 + 4 * RT * m + t;
            if (tt >= M) break;
            const uint32_t l = (t / RT) * 16 + c / J;
            float v = part[0][c % J][l][t % RT];
#pragma unroll
            for (int w = 1; w < KS; w++) v += part[w][c % J][l][t % RT];
            v *= I8_SCALE_UP;
            if (split_part) split_part[((uint64_t)blockIdx.y * M + tt) * N + n0 + c] = v;
            else finalize_store(A, tt, n0 + c, v);
        }
        __syncthreads();
    }
}

// SEG: blocks per scale segment (a divisor of the group's blocks), at most a
// batch.
template <int MT, int J, int KS, int U, int SEG, int RT = 4>
void launch_i8_form(const PpArgs& P, bool paired, bool ct, uint32_t splits, float* part, hipStream_t st) {
    constexpr int BPG = SEG < U ? SEG : U;
    const uint32_t tg = (P.L.B + 4 * RT * MT - 1) / (4 * RT * MT), tiles = P.L.N / (16 * J);
    const dim3 grid((tiles + 7) / 8 * 8 * tg, splits);
    const uint32_t unit = ct ? 4 : BPG > 2 ? BPG : 2, units = (P.L.K / 32 + unit - 1) / unit;
    const uint32_t per = (units + KS * splits - 1) / (KS * splits) * unit;
    if (paired) int4_i8_kernel<MT, J, KS, U, BPG, true, false, RT><<<grid, 64 * KS, 0, st>>>(P, tg, part, per);
    else if (!ct) int4_i8_kernel<MT, J, KS, U, BPG, false, false, RT><<<grid, 64 * KS, 0, st>>>(P, tg, part, per);
    else if constexpr (J == 1) int4_i8_kernel<MT, J, KS, U, BPG, false, true, RT><<<grid, 64 * KS, 0, st>>>(P, tg, part, per);
}

template <int SEG>
void launch_i8_shape(const PpArgs& P, bool paired, bool ct, uint32_t j, uint32_t mt, uint32_t splits, float* part, hipStream_t st) {
    if (j == 4) {
        if (P.L.B <= 4) launch_i8_form<1, 4, 8, 8, SEG, 1>(P, paired, ct, splits, part, st);
        else if (mt == 1) launch_i8_form<1, 4, 8, 8, SEG>(P, paired, ct, splits, part, st);
        else if (mt == 2) launch_i8_form<2, 4, 8, 4, SEG>(P, paired, ct, splits, part, st);
        else if constexpr (SEG != 2) launch_i8_form<3, 4, 8, 4, SEG>(P, paired, ct, splits, part, st);
    } else {
        if (P.L.B <= 4) launch_i8_form<1, 1, 8, 16, SEG, 1>(P, paired, ct, splits, part, st);
        else if (mt == 1) launch_i8_form<1, 1, 8, 16, SEG>(P, paired, ct, splits, part, st);
        else launch_i8_form<2, 1, 8, 8, SEG>(P, paired, ct, splits, part, st);
    }
}

// Launches the matrix-core form when the shape and alignment allow its 16-byte
// loads (whole 16-column tiles; whole 64-column activation pairs, 128 columns
// for CT rows); false otherwise (int4_pp_kernel takes every other shape).
// 64-column tiles (16 bytes a lane) where they fill more than half of the CUs,
// else 16-column ones: at N = 4096 the 64 wide tiles would stream 29 MB through
// 64 CUs, and a CU takes in about 27 GB/s.  17 to 32 rows take wide tiles there
// too, K split over the CUs and the partial sums added by a second launch: 14336
// x 4096 between two 4096 x 14336, 16 / 20 / 32 rows 49.5 / 57.8 / 62.8 us ->
// 46.1 / 53.8 / 56.6, but 9 rows of smaller shapes lose 2 to 5 %.
// one_group: up to 48 rows as one group, wide unsplit tiles only past 32 rows.
bool launch_i8(const PpArgs& P, bool paired, bool ct, bool one_group, const nerve_hip_ctx* ctx, hipStream_t st) {
    const Int4Args& A = P.L;
    const uint32_t cus = (uint32_t)ctx->cu_count;
    if (A.N % 16 || A.K % 64 || ((uintptr_t)P.q & 15) || ((uintptr_t)A.qw & 15)) return false;
    if (ct && A.K % 128) return false;
    const uint32_t mt = A.B <= 16 ? 1 : one_group ? (A.B + 15) / 16 : 2;
    const uint32_t tg = (A.B + 16 * mt - 1) / (16 * mt), wide = A.N / 64 * tg;
    const bool can = !ct && A.N % 64 == 0;
    uint32_t j = can && wide * 2 > cus ? 4 : 1, splits = 1;
    if (j == 1 && can && mt == 2 && tg == 1) {
        const uint64_t most = std::min<uint64_t>(A.K / 1024, nh::kSplitBytes / ((uint64_t)A.B * A.N * 4));
        splits = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(cus / wide, most));
        if (splits > 1) j = 4;
    }
    if (mt > 3 || (mt == 3 && j == 1)) return false;
    // A few rows of a short K, the more with every round of blocks: int4_pp_kernel's
    // lanes are done with their columns in a shorter chain than blocks of 8 waves are
    // placed, loaded and summed (us, int4_pp_kernel / here: one row of 512 x 512 3.1 / 4.0,
    // of 512 x 8192 4.3 / 6.0, of CT 512 x 32768 5.5 / 21.3; two rows of CT 2048 x 32768
    // 27.7 / 34.8, but of 1024 x 2048 6.2 / 3.9 and five of CT 1536 x 32768 42.3 / 33.4).
    // Rows in column order, which it brings into nibble order first, gain half as much.
    const uint32_t blocks = j == 4 ? wide : A.N / 16 * tg, rounds = std::min(8u, (blocks + cus - 1) / cus);
    const uint64_t chain = (uint64_t)A.B * (A.K < 128 ? 256 : std::max(A.K, 512u) * (paired || ct ? 1 : 2));
    if (chain <= (A.B == 1 && (ct || rounds >= 4) ? 1300u : ct ? 720u : 640u) * rounds) return false;
    float* part = splits > 1 ? static_cast<float*>(ctx->split) : nullptr;
    // (three token tiles and two-block segments spill 47 registers: no such form)
    const uint32_t bpg = A.G % 128 == 0 ? 4 : A.G % 64 == 0 && mt < 3 ? 2 : 1;
    if (bpg == 4) launch_i8_shape<4>(P, paired, ct, j, mt, splits, part, st);
    else if (bpg == 2) launch_i8_shape<2>(P, paired, ct, j, mt, splits, part, st);
    else launch_i8_shape<1>(P, paired, ct, j, mt, splits, part, st);
    if (part) nh::int4_split_sum(A, part, splits, st);
    return true;
}

}  // namespace

extern "C" nerve_hip_status nerve_hip_int4_linear(nerve_hip_ctx* ctx, const char* spec, const void* x_bf16,
                                                  const void* qweight, const void* scales, const void* zeros,
                                                  const void* aux_bf16, void* y_bf16, uint32_t batch_width,
                                                  void* stream) {
    nerve_hip_status st = nh::enter(ctx);
    if (st) return st;
    nh::Int4Spec s;
    if ((st = nh::parse_int4_spec(spec, &s))) return st;
    if (s.input != 0)
        return nh::fail(NERVE_HIP_INVALID_SPEC, "INT8-prequantized input goes through nerve_hip_int4_linear_pairpacked");
    if (!x_bf16 || !qweight || !scales || !y_bf16) return nh::fail(NERVE_HIP_INVALID_ARGUMENT, "null buffer");
    if (s.op != 0 && !aux_bf16) return nh::fail(NERVE_HIP_INVALID_ARGUMENT, "bias/residual specialization needs aux");
    if (s.batch_tile == 0 && batch_width > 1)
        return nh::fail(NERVE_HIP_INVALID_ARGUMENT, "unbatched INT4 specialization takes batch_width 1");
    if (batch_width == 0) return nh::ok();
    if ((((uintptr_t)x_bf16) | ((uintptr_t)qweight)) & 15)
        return nh::fail(NERVE_HIP_INVALID_ARGUMENT, "x and qweight must be 16-byte aligned");
    Int4Args A;
    A.x = static_cast<const uint16_t*>(x_bf16);
    A.qw = static_cast<const uint32_t*>(qweight);
    A.scales = static_cast<const uint16_t*>(scales);
    A.qzeros = static_cast<const uint32_t*>(zeros);
    A.aux = static_cast<const uint16_t*>(aux_bf16);
    A.y = static_cast<uint16_t*>(y_bf16);
    A.B = batch_width;
    A.K = s.in;
    A.N = s.out;
    A.G = s.group;
    A.scale_bf16 = s.scale_bf16;
    A.finalize = s.op;
    hipStream_t strm = (hipStream_t)stream;
    // More than 16 rows: the tiled split-K form, which expands the weights once per
    // 64 rows instead of once per 16; from five rows on also where column tiles are
    // few and K is long (16 rows of 14336 x 4096: 25.4 -> 14.6 us).  The 16-row
    // kernels stay where few rounds of their blocks cover the linear and K is short
    // enough for the launch that adds the split sums to count (us, 16-row kernel /
    // tiled form).
    const uint32_t cus = (uint32_t)ctx->cu_count;
    const uint64_t row_tiles16 = (batch_width + 15) / 16;
    bool few_rounds = false;
    if (s.layout == 0 && A.N % 64 == 0) {
        // A block a CU: 64 rows of 4096 x 4096 10.1 / 15.1; of 14336 x 4096 25.9 / 20.0;
        // with most CUs taken by more than 64 rows also a longer K, but for groups of 32
        // (7168 x 2048, 96 rows 15.6 / 17.4, 128 rows 17.7 / 20.1, g64 18.1 / 20.6; 17
        // rows of 8192 x 8192 20.8 / 18.0).  Two blocks of 8 waves a CU (of groups of 128 only a full
        // round has 8): 512 rows of 2048 x 1024 11.4 / 16.1, 128 of 4096 x 4096
        // 18.3 / 20.8, 48 of 1024 x 8192, g64, 9.4 / 11.1; of 512 columns 128 rows of
        // N = 4096 9.2 / 7.7; g32 128 of 4096 x 4096 24.9 / 23.5, of
        // 2304 x 4096 17.1 / 18.8.
        const uint64_t blocks = (uint64_t)(A.N / 64) * row_tiles16;
        const bool eight = A.G == 32 || A.G == 64 || A.G == 256 || (A.G == 128 && blocks == 2 * cus);
        if (blocks <= cus) {
            few_rounds = A.K <= (4 * blocks >= 3 * cus && batch_width > 64 && A.G > 32 ? 8192u : 6144u);
        } else if (blocks <= 2 * cus) {
            // Short of one and a half blocks a CU: g64, 80 rows of 2048 x 4096 10.5 / 12.5,
            // 350 of 1536 x 1024 9.4 / 13.1, of 3072 x 1024 14.6 / 15.9, 300 14.5 / 14.0;
            // g256, 65 of 1280 x 4096 6.5 / 9.8, 350 of 2816 x 1024 12.1 / 13.5;
            // g32, 80 of 1024 x 4096 10.4 / 11.3, 300 of 2048 x 1024 13.7 / 12.8.
            const bool most = 2 * blocks >= 3 * cus || (A.G == 64 && A.K <= 2048) || (A.G == 32 && A.K <= 1536) ||
                              (A.G == 256 && A.K <= 3072);
            few_rounds = eight && most && A.K >= 1024 && A.K <= (A.G > 32 ? 4096u : 2304u);
        } else if (blocks <= 3 * cus ? A.G == 32 || A.G == 64 || A.G == 128 || A.G == 256
                                     : blocks > 4 * cus && blocks <= 5 * cus && (A.G == 64 || A.G == 128 || A.G == 256)) {
            // Three blocks a CU, or five: 300 rows of 2048 x 2048 13.0 / 14.2, g64 13.7 / 16.5, 200 of
            // 2048 x 3072 13.3 / 16.1, g64 14.0 / 18.0; of 1536 x 3072 12.3 / 13.1, g64
            // 12.8 / 14.5, 400 of 2048 x 3072 19.3 / 21.2, g64 20.6 / 23.6, but 300 of 1536 x
            // 2048 12.1 / 11.4; g64 of 1024 x 2048 11.8 / 10.1; g256, 256 of 2816 x 3072
            // 17.5 / 20.7, 65 of 1792 x 8192 11.3 / 13.6.
            few_rounds = A.K <= (A.G == 256 ? 2816u : 2560u) && A.K >= (A.G == 64 && blocks <= 3 * cus ? 1536u : 1792u);
        }
    } else if (s.layout == 1 && A.K <= 4096 && A.N % 16 == 0) {
        // 16 columns a block: 17 rows of 1024 x 512 6.3 / 7.7, 64 of 4096 x 1024
        // 8.3 / 11.5; 32 columns (a full round of them): 32 rows of 4096 x 4096
        // 9.9 / 13.5; 17 of 6144 x 2048 13.0 / 11.8.  A short K leaves a second block's
        // chain short: 33 rows of 512 x 2048 5.0 / 7.2, of 768 x 2048 6.4 / 8.8.
        const uint64_t blocks = (uint64_t)(A.N / 16) * row_tiles16;
        few_rounds = blocks <= cus || (A.N % 32 == 0 && blocks == 2 * cus) ||
                    (A.K <= 512 && blocks <= 2 * cus) || (A.K <= 768 && 2 * blocks <= 3 * cus);
    }
    const bool few = s.layout == 0 && A.N % 64 == 0 && batch_width > GEMV_MAX_M && batch_width <= 16 && A.K > 6144 &&
                     2 * (A.N / 64) <= cus;
    if (((batch_width > 16 && !few_rounds) || few) && !(s.layout == 1 && (zeros || A.G % 128)) &&
        nh::int4_gemm(ctx, A, nullptr, false, s.layout == 1, strm))
        return nh::check_launch("int4_linear_gemm");
    if (s.layout == 0) {
        if (A.N % 16) return nh::fail(NERVE_HIP_UNSUPPORTED, "GPTQ INT4 kernel needs N % 16 == 0");
        if (zeros && A.N % 8) return nh::fail(NERVE_HIP_INVALID_ARGUMENT, "qzeros need N % 8 == 0");
        // 64-column tiles (8 KiB of weights in flight per wave per batch);
        // N % 64 != 0 uses 16-column tiles with deeper batches.
        const uint32_t row_tiles = (batch_width + 15) / 16;
        const bool wide = A.N % 64 == 0;
        const uint32_t tiles = wide ? A.N / 64 : A.N / 16;
        dim3 grid((tiles + 7) / 8 * 8, row_tiles);
        const uint32_t steps = A.G / 32;
        // Decode-sized batches go to the vector-ALU kernel.
        if (wide && batch_width <= GEMV_MAX_M && (A.G == 32 || A.G == 64 || A.G == 128 || A.G == 256) &&
            ((uintptr_t)scales & 7) == 0) {
            // Few column tiles and more than one batch per wave: K is split so
            // that every CU has a block, the partial sums added by a second
            // launch (14336 x 4096, one row: 64 blocks 14.9 us, 256 10.1).  One row
            // gains less: from K > 6144 on (unsplit / split, 4608 x 4096 7.2 / 7.9,
            // 6144 x 8192 9.9 / 10.1, 7168 x 4096 9.9 / 9.2), later where half of the
            // CUs have a tile (9216 x 6144 13.0 / 12.2, but 9216 x 8192 13.3 / 14.2,
            // 11008 x 8192 15.7 / 15.3); two rows of 4608 x 4096 9.0 / 8.9, four
            // 9.3 / 9.0.
            const uint32_t batches = (A.K / 8 + GEMV_ROWS - 1) / GEMV_ROWS;
            const bool gains = batch_width > 1 || A.K > (2 * tiles >= cus ? 10240u : 6144u);
            const uint32_t most = gains ? std::max(1u, std::min((A.K / 256 + 15) / 16, cus / tiles)) : 1u;
            const uint32_t span = (batches + most - 1) / most, splits = (batches + span - 1) / span;
            float* part = splits > 1 ? static_cast<float*>(ctx->split) : nullptr;
            dim3 g1((tiles + 7) / 8 * 8, splits);
            const bool zp = zeros != nullptr;
#define NERVE_INT4_GEMV_FORM(GG, ZP, MT)                                                                  \
    (part ? int4_gptq_gemv_kernel<16, GG, ZP, MT, true><<<g1, 1024, 0, strm>>>(A, part, span)             \
          : int4_gptq_gemv_kernel<16, GG, ZP, MT, false><<<g1, 1024, 0, strm>>>(A, part, span))
#define NERVE_INT4_GEMV(GG)                                                                               \
    (batch_width == 1 ? (zp ? NERVE_INT4_GEMV_FORM(GG, true, 1) : NERVE_INT4_GEMV_FORM(GG, false, 1))     \
                      : (zp ? NERVE_INT4_GEMV_FORM(GG, true, 4) : NERVE_INT4_GEMV_FORM(GG, false, 4)))
            if (A.G == 128) NERVE_INT4_GEMV(128);
            else if (A.G == 64) NERVE_INT4_GEMV(64);
            else if (A.G == 32) NERVE_INT4_GEMV(32);
            else NERVE_INT4_GEMV(256);
#undef NERVE_INT4_GEMV
#undef NERVE_INT4_GEMV_FORM
            if (part) nh::int4_split_sum(A, part, splits, strm);
            return nh::check_launch("int4_linear_gptq_gemv");
        }
        // Few column tiles (decode-sized N): 16 waves split K so that each
        // wave's share is one load batch.
        const bool deep = tiles * row_tiles < 2u * (uint32_t)ctx->cu_count;
        if (wide && steps == 4 && deep) int4_gptq_fixed_kernel<16, 4, 4><<<grid, 1024, 0, strm>>>(A);
        else if (wide && steps == 4) int4_gptq_fixed_kernel<8, 4, 4><<<grid, 512, 0, strm>>>(A);
        else if (wide && steps == 1) int4_gptq_fixed_kernel<8, 4, 1><<<grid, 512, 0, strm>>>(A);
        else if (wide && steps == 2) int4_gptq_fixed_kernel<8, 4, 2><<<grid, 512, 0, strm>>>(A);
        else if (wide && steps == 8) int4_gptq_fixed_kernel<8, 4, 8><<<grid, 512, 0, strm>>>(A);
        else if (!wide && steps == 4) int4_gptq_fixed_kernel<8, 1, 4><<<grid, 512, 0, strm>>>(A);
        else if (wide) int4_gptq_kernel<8, 4, 8><<<grid, 512, 0, strm>>>(A);
        else int4_gptq_kernel<8, 1, 16><<<grid, 512, 0, strm>>>(A);
        return nh::check_launch("int4_linear_gptq");
    }
    if (zeros) return nh::fail(NERVE_HIP_UNSUPPORTED, "asymmetric zeros are supported for the GPTQ layout only");
    if (A.G % 128 || A.N % 16) return nh::fail(NERVE_HIP_UNSUPPORTED, "CT INT4 kernel needs group % 128 == 0 and N % 16 == 0");
    // 32 rows a block where that still gives every CU one and the activations
    // count (16 tokens of 4096 x 14336: 17.7 us against 22.0; one: 12.9, 12.6).
    const uint32_t row_tiles = (batch_width + 15) / 16;
    if (batch_width > 2 && A.N % 32 == 0 && A.N / 32 * row_tiles >= (uint32_t)ctx->cu_count)
        int4_ct_kernel<8, 2><<<dim3(A.N / 32, row_tiles), 512, 0, strm>>>(A);
    else
        int4_ct_kernel<8, 1><<<dim3(A.N / 16, row_tiles), 512, 0, strm>>>(A);
    return nh::check_launch("int4_linear_ct");
}

extern "C" nerve_hip_status nerve_hip_quantize_int8_pairpacked(nerve_hip_ctx* ctx, const char* spec, const void* x_bf16,
                                                              void* q_i8, void* scales_f32, void* sums_i32,
                                                              uint32_t rows, void* stream) {
    nerve_hip_status st = nh::enter(ctx);
    if (st) return st;
    nh::QuantI8Spec qs;
    if ((st = nh::parse_quant_i8_spec(spec, &qs))) return st;
    if (qs.silu) return nh::fail(NERVE_HIP_INVALID_SPEC, "silu_multiply_quantize goes through its own entry point");
    if (!x_bf16 || !q_i8 || !scales_f32 || (qs.paired && !sums_i32))
        return nh::fail(NERVE_HIP_INVALID_ARGUMENT, "null buffer");
    if (qs.batch_tile == 0 && rows > 1)
        return nh::fail(NERVE_HIP_INVALID_ARGUMENT, "unbatched pair-packed quantizer takes one row");
    if (((uintptr_t)x_bf16 & 15) || ((uintptr_t)q_i8 & 7))
        return nh::fail(NERVE_HIP_INVALID_ARGUMENT, "x must be 16-byte and q 8-byte aligned");
    if (rows == 0) return nh::ok();
    const uint64_t octs = (uint64_t)rows * qs.elements / 8;
    const uint32_t grid = (uint32_t)((octs + 255) / 256);
    if (qs.paired)
        quant_i8pp_kernel<false, true><<<grid, 256, 0, (hipStream_t)stream>>>(
            static_cast<const uint16_t*>(x_bf16), nullptr, nullptr, rows, qs.elements, static_cast<uint32_t*>(q_i8),
            static_cast<float*>(scales_f32), static_cast<int32_t*>(sums_i32));
    else
        quant_i8pp_kernel<false, false><<<grid, 256, 0, (hipStream_t)stream>>>(
            static_cast<const uint16_t*>(x_bf16), nullptr, nullptr, rows, qs.elements, static_cast<uint32_t*>(q_i8),
            static_cast<float*>(scales_f32), static_cast<int32_t*>(sums_i32));
    return nh::check_launch("quantize_int8");
}

extern "C" nerve_hip_status nerve_hip_silu_multiply_quantize_int8_pairpacked(nerve_hip_ctx* ctx, const char* spec,
                                                                            const void* gate_bf16, const void* up_bf16,
                                                                            void* y_bf16, void* q_i8, void* scales_f32,
                                                                            void* sums_i32, uint32_t rows,
                                                                            void* stream) {
    nerve_hip_status st = nh::enter(ctx);
    if (st) return st;
    nh::QuantI8Spec qs;
    if ((st = nh::parse_quant_i8_spec(spec, &qs))) return st;
    if (!qs.silu) return nh::fail(NERVE_HIP_INVALID_SPEC, "not a silu_multiply_quantize specialization");
    if (!gate_bf16 || !up_bf16 || !y_bf16 || !q_i8 || !scales_f32 || !sums_i32)
        return nh::fail(NERVE_HIP_INVALID_ARGUMENT, "null buffer");
    if (qs.batch_tile == 0 && rows > 1)
        return nh::fail(NERVE_HIP_INVALID_ARGUMENT, "unbatched pair-packed quantizer takes one row");
    if ((((uintptr_t)gate_bf16) | ((uintptr_t)up_bf16) | ((uintptr_t)y_bf16)) & 15 || ((uintptr_t)q_i8 & 7))
        return nh::fail(NERVE_HIP_INVALID_ARGUMENT, "gate, up and y must be 16-byte and q 8-byte aligned");
    if (rows == 0) return nh::ok();
    // The kernel reads gate and up through restrict pointers while it writes
    // y: y may not overlap either input.
    const uintptr_t bytes = (uintptr_t)rows * qs.elements * 2, yb = (uintptr_t)y_bf16;
    auto overlaps = [&](const void* p) { const uintptr_t a = (uintptr_t)p; return a < yb + bytes && yb < a + bytes; };
    if (overlaps(gate_bf16) || overlaps(up_bf16))
        return nh::fail(NERVE_HIP_INVALID_ARGUMENT, "y must not overlap gate or up");
    const uint64_t octs = (uint64_t)rows * qs.elements / 8;
    quant_i8pp_kernel<true><<<(uint32_t)((octs + 255) / 256), 256, 0, (hipStream_t)stream>>>(
        static_cast<const uint16_t*>(gate_bf16), static_cast<const uint16_t*>(up_bf16), static_cast<uint16_t*>(y_bf16),
        rows, qs.elements, static_cast<uint32_t*>(q_i8), static_cast<float*>(scales_f32),
        static_cast<int32_t*>(sums_i32));
    return nh::check_launch("silu_multiply_quantize_int8_pairpacked");
}

extern "C" nerve_hip_status nerve_hip_int4_linear_pairpacked(nerve_hip_ctx* ctx, const char* spec, const void* q_i8,
                                                            const void* scales_f32, const void* sums_i32,
                                                            const void* qweight, const void* scales,
                                                            const void* aux_bf16, void* y_bf16, uint32_t batch_width,
                                                            void* stream) {
    nerve_hip_status st = nh::enter(ctx);
    if (st) return st;
    nh::Int4Spec s;
    if ((st = nh::parse_int4_spec(spec, &s))) return st;
    if (s.input == 0) return nh::fail(NERVE_HIP_INVALID_SPEC, "not a _prequant[_pairpacked] INT4 specialization");
    const bool paired = s.input == 2;
    if (!q_i8 || !scales_f32 || (paired && !sums_i32) || !qweight || !scales || !y_bf16)
        return nh::fail(NERVE_HIP_INVALID_ARGUMENT, "null buffer");
    if (s.op != 0 && !aux_bf16) return nh::fail(NERVE_HIP_INVALID_ARGUMENT, "bias/residual specialization needs aux");
    if (s.batch_tile == 0 && batch_width > 1)
        return nh::fail(NERVE_HIP_INVALID_ARGUMENT, "unbatched INT4 specialization takes batch_width 1");
    if (((uintptr_t)q_i8 & 3) || ((uintptr_t)qweight & 3))
        return nh::fail(NERVE_HIP_INVALID_ARGUMENT, "q and qweight must be 4-byte aligned");
    if (batch_width == 0) return nh::ok();
    PpArgs P;
    P.q = static_cast<const uint32_t*>(q_i8);
    P.s = static_cast<const float*>(scales_f32);
    P.sums = static_cast<const int32_t*>(sums_i32);
    P.L.x = nullptr;
    P.L.qw = static_cast<const uint32_t*>(qweight);
    P.L.scales = static_cast<const uint16_t*>(scales);
    P.L.qzeros = nullptr;
    P.L.aux = static_cast<const uint16_t*>(aux_bf16);
    P.L.y = static_cast<uint16_t*>(y_bf16);
    P.L.B = batch_width;
    P.L.K = s.in;
    P.L.N = s.out;
    P.L.G = s.group;
    P.L.scale_bf16 = s.scale_bf16;
    P.L.finalize = s.op;
    const uint32_t grid = (s.out + 63) / 64;
    hipStream_t strm = (hipStream_t)stream;
    // Up to 32 rows, and 33 to 48 that fill the CUs with 64-column tiles: one
    // group of rows over the weights (48 rows of 4096 x 14336: 19.7 us against
    // 25.5; 16-column tiles 33 against 24.5 for 14336 x 4096).  Else the tiled
    // split-K form.
    const bool ct = s.layout == 1;
    if (launch_i8(P, paired, ct, true, ctx, strm)) return nh::check_launch("int4_linear_prequant");
    if (batch_width > 32 && nh::int4_gemm(ctx, P.L, &P, paired, ct, strm)) return nh::check_launch("int4_linear_prequant");
    if (launch_i8(P, paired, ct, false, ctx, strm)) return nh::check_launch("int4_linear_prequant");
    if (paired) int4_pp_kernel<true, false><<<grid, 256, 0, strm>>>(P);
    else if (s.layout == 0) int4_pp_kernel<false, false><<<grid, 256, 0, strm>>>(P);
    else int4_pp_kernel<false, true><<<grid, 256, 0, strm>>>(P);
    return nh::check_launch("int4_linear_prequant");
}
