// Sparse-expert INT4 (compressed-tensors) projections on gfx950:
// gate/up + SwiGLU and down + route weight.
//
// Reference: sparse_moe_gate_up_int4_ct.comp.template:97-227 and
// sparse_moe_down_int4_ct.comp.template:106-193 (rendered by
// nerve/model_package_sparse_projection_shaders.py:80-232).  Per route the
// shaders compute, for every output row, the f32 sum over packed words of
// fma(dot8(x, q - 8), scale[row, group], sum) with a 64-lane strided loop and
// subgroupAdd; gate/up then give bf16(bf16(silu(bf16 g)) * bf16 u) and down
// gives bf16(bf16(y) * route_weight).
//
// sparse_tile_kernel contracts an expert's weights against a tile of its routes
// on the matrix cores (further down); sparse_int4_kernel takes the shapes and the
// small calls that it does not (launch_tiles).  The latter is HBM-bound weight
// streaming (one activation row per route), so it is organised around keeping 16-byte weight loads in flight:
//   * a block (4 waves) owns one route position and a tile of output rows;
//     each wave owns 8 weight rows (gate/up: 4 gate + the 4 matching up rows;
//     down: 8 rows) and issues all of its weight and scale loads of a pass
//     before the first arithmetic;
//   * lanes split a row into 16-byte chunks (32 codes), LU lanes per row, so
//     rows whose chunk count is not a multiple of 64 still fill the lanes;
//   * the activation row is staged once per block in LDS (4-byte loads: route
//     slices of the intermediate frames are only 4-byte aligned);
//   * codes become bf16 (128 + q) pairs with one and-or per two codes and
//     v_dot2_f32_bf16 contracts them with the activation pairs; the per-word
//     term 136 * sum(x) restores (q - 8).  Products are exact in f32; only the
//     summation order differs from the shader's (whose subgroupAdd order is
//     itself unspecified).
// Blocks are dealt to the XCDs in contiguous runs of (tile, position) work
// with positions fastest, so the routes of one expert (adjacent in the
// compacted map, which sorts routes by expert) read its rows through one L2.
#include "common.h"

namespace {

typedef __bf16 v2bf __attribute__((ext_vector_type(2)));

constexpr uint32_t SM_WAVES = 4;
constexpr uint32_t SM_WROWS = 8;            // weight rows per wave
constexpr uint32_t SM_MAX_K = 16384;        // activation row staged in LDS
constexpr uint32_t SM_UNBOUND = 0xffffffffu;
constexpr uint32_t SM_ONES = 0x3F803F80u;   // bf16 (1, 1)

struct SmArgs {
    const uint16_t* x;          // gate_up: hidden bf16 [B, H]; down: the frames as bf16
    const uint32_t* routes;     // [B * k] route words
    const uint32_t* frames;     // intermediate frames (route map in the tails)
    uint16_t* out;              // gate_up: the frames as bf16; down: expert_outputs [B * k, H]
    const uint32_t* addr;
    const uint32_t* slots;
    const uint32_t* control;    // BatchControl, or null (unbatched form without an expert range)
    uint32_t n_records, n_slot_words;
    uint32_t batch_width, k, E;
    uint32_t K, N, I, G;        // contraction, output rows, intermediate size, group
    uint64_t frame_words;       // u32 words per frame (k * I / 2, + k route-map words when batched)
    uint32_t data_words;        // k * I / 2
    uint32_t tiles;             // row tiles per route
    uint32_t npos;              // route positions in the grid
    uint32_t per_xcd;           // grid / 8
    uint64_t w_bytes, s_bytes;  // bytes one expert's weight / scale tensor must span
    int batched, scale_bf16;
};

__device__ __forceinline__ float dot2_bf16(uint32_t a, uint32_t b, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2bf, a), __builtin_bit_cast(v2bf, b), c, false);
}

__device__ __forceinline__ float decode_scale(uint32_t v, int bf16) {
    return bf16 ? bf16_to_f32(v) : (float)__builtin_bit_cast(_Float16, (uint16_t)v);
}

// Pairs (0,4),(1,5),(2,6),(3,7) of 8 contiguous bf16: the order in which
// sm_word_dot decodes the codes of one packed word.
__device__ __forceinline__ v4i sm_permute(v4i a) {
    const uint32_t d0 = (uint32_t)a.x, d1 = (uint32_t)a.y, d2 = (uint32_t)a.z, d3 = (uint32_t)a.w;
    return v4i{(int)((d0 & 0xFFFFu) | (d2 << 16)), (int)((d0 >> 16) | (d2 & 0xFFFF0000u)),
               (int)((d1 & 0xFFFFu) | (d3 << 16)), (int)((d1 >> 16) | (d3 & 0xFFFF0000u))};
}

// sum_{i<8} x_i (128 + q_i) of one word (codes low nibble first along k)
// against permuted activations.
__device__ __forceinline__ float sm_word_dot(uint32_t w, v4i xp) {
    float d = dot2_bf16((uint32_t)xp.x, (w & 0x000F000Fu) | 0x43004300u, 0.0f);
    d = dot2_bf16((uint32_t)xp.y, ((w >> 4) & 0x000F000Fu) | 0x43004300u, d);
    d = dot2_bf16((uint32_t)xp.z, ((w >> 8) & 0x000F000Fu) | 0x43004300u, d);
    return dot2_bf16((uint32_t)xp.w, ((w >> 12) & 0x000F000Fu) | 0x43004300u, d);
}

__device__ __forceinline__ float sm_word_sum(v4i xp) {
    float s = dot2_bf16((uint32_t)xp.x, SM_ONES, 0.0f);
    s = dot2_bf16((uint32_t)xp.y, SM_ONES, s);
    s = dot2_bf16((uint32_t)xp.z, SM_ONES, s);
    return dot2_bf16((uint32_t)xp.w, SM_ONES, s);
}

// One 8-word address record (u32 {addr_lo, addr_hi, bytes_lo, bytes_hi, ...})
// behind parameter slot `idx`, or null.  The shaders only skip unbound slots
// (…gate_up_int4_ct.comp.template:163-166); slots beyond the table, null
// addresses, misaligned addresses and records shorter than the expert's tensor
// are treated the same way here instead of being read out of bounds.
__device__ __forceinline__ const void* sm_param(const SmArgs& A, uint32_t idx, uint64_t need, uint32_t align) {
    if (idx >= A.n_slot_words) return nullptr;
    const uint32_t slot = A.slots[idx];
    if (slot == SM_UNBOUND || slot >= A.n_records) return nullptr;
    const uint32_t* rec = A.addr + (uint64_t)slot * 8;
    const uint64_t a = (uint64_t)rec[0] | ((uint64_t)rec[1] << 32);
    const uint64_t bytes = (uint64_t)rec[2] | ((uint64_t)rec[3] << 32);
    if (a == 0 || (a & (align - 1)) || bytes < need) return nullptr;
    return reinterpret_cast<const void*>(a);
}

// LU: lanes per weight row (64, 32 or 16).  SPW: one scale per packed word
// (group sizes that are not a multiple of 32) instead of one per chunk.
template <bool GATE_UP, uint32_t LU, bool SPW>
__global__ __launch_bounds__(64 * SM_WAVES) void sparse_int4_kernel(SmArgs A) {
    constexpr uint32_t RS = 64 / LU;                  // rows loaded side by side
    constexpr uint32_t RPL = SM_WROWS / RS;           // rows per lane
    constexpr uint32_t NUP = 16 / RPL;                // chunks per lane per pass
    constexpr uint32_t OR = GATE_UP ? SM_WROWS / 2 : SM_WROWS;   // output rows per wave
    constexpr uint32_t NSC = SPW ? 4 : 1;
    extern __shared__ __attribute__((aligned(16))) uint16_t xs[];   // K activations

    // Work item: position fastest; contiguous runs of items per XCD.
    const uint32_t w = (blockIdx.x % 8) * A.per_xcd + blockIdx.x / 8;
    const uint32_t pos = w % A.npos, tile = w / A.npos;
    if (tile >= A.tiles) return;

    // Route of this position (…gate_up_int4_ct.comp.template:142-166 with
    // the batched ROUTE_MAPPING of nerve/model_package_sparse_projection_
    // shaders.py:194-212).
    // The map word and the control words are read together (every position
    // below B * k has a map word), so the chain of dependent loads before the
    // weights is map -> route -> slots -> records.
    const uint32_t cap = A.batch_width * A.k;
    uint32_t c = pos;
    uint32_t start = 0, count = 0, owned = cap;
    if (A.batched) c = A.frames[(uint64_t)(pos / A.k) * A.frame_words + A.data_words + pos % A.k];
    if (A.control) {
        start = A.control[1];
        count = A.control[2];
        if (A.batched) owned = A.control[3];
    }
    if (A.batched && count != 0u && pos >= owned) return;
    if (c >= cap) return;
    const uint32_t rw = A.routes[c];
    const uint32_t e = rw & 0xffffu;
    if (e >= A.E || (count != 0u && (e < start || e - start >= count))) return;
    const uint32_t* W = static_cast<const uint32_t*>(sm_param(A, 2 * e, A.w_bytes, 16));
    const uint16_t* S = static_cast<const uint16_t*>(sm_param(A, 2 * e + 1, A.s_bytes, 2));
    if (!W || !S) return;
    const uint32_t b = c / A.k, r = c % A.k;

    const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const uint32_t rsub = lane / LU, cl = lane % LU;
    const uint32_t K = A.K, kw = K / 8, units = K / 32, ng = K / A.G;
    const uint32_t orow0 = tile * (SM_WAVES * OR) + wave * OR;

    // Weight rows of this lane (clamped into the matrix; results of rows past
    // N are not stored).
    const uint32_t* wrow[RPL];
    const uint16_t* srow[RPL];
#pragma unroll
    for (uint32_t j = 0; j < RPL; j++) {
        const uint32_t li = rsub * RPL + j;
        uint32_t row;
        if constexpr (GATE_UP) row = min(orow0 + (li % OR), A.N - 1) + (li >= OR ? A.I : 0u);
        else row = min(orow0 + li, A.N - 1);
        wrow[j] = W + (uint64_t)row * kw;
        srow[j] = S + (uint64_t)row * ng;
    }

    // Activation row -> LDS.
    const uint16_t* xg = GATE_UP ? A.x + (uint64_t)b * K : A.x + (uint64_t)b * A.frame_words * 2 + (uint64_t)r * A.I;
    {
        const uint32_t* xg32 = reinterpret_cast<const uint32_t*>(xg);
        uint32_t* xs32 = reinterpret_cast<uint32_t*>(xs);
        for (uint32_t i = tid; i < K / 2; i += 64 * SM_WAVES) xs32[i] = xg32[i];
    }
    bool staged = false;

    float acc[RPL];
#pragma unroll
    for (uint32_t j = 0; j < RPL; j++) acc[j] = 0.0f;

    for (uint32_t u0 = 0; u0 < units; u0 += LU * NUP) {
        v4i wv[NUP][RPL];
        uint16_t sv[NUP][RPL][NSC];
#pragma unroll
        for (uint32_t i = 0; i < NUP; i++) {
            if (u0 + i * LU >= units) break;      // chunk slots past the row (uniform)
            const uint32_t un = min(u0 + i * LU + cl, units - 1);
            uint32_t gi[NSC];
#pragma unroll
            for (uint32_t q = 0; q < NSC; q++) gi[q] = (un * 32 + 8 * q) / A.G;
#pragma unroll
            for (uint32_t j = 0; j < RPL; j++) {
                wv[i][j] = *reinterpret_cast<const v4i*>(wrow[j] + un * 4);
#pragma unroll
                for (uint32_t q = 0; q < NSC; q++) sv[i][j][q] = srow[j][gi[q]];
            }
        }
        if (!staged) {
            __syncthreads();
            staged = true;
        }
#pragma unroll
        for (uint32_t i = 0; i < NUP; i++) {
            const uint32_t un = u0 + i * LU + cl;
            if (un >= units) continue;
            v4i xp[4];
            float sx[4];
#pragma unroll
            for (uint32_t q = 0; q < 4; q++) {
                xp[q] = sm_permute(*reinterpret_cast<const v4i*>(xs + un * 32 + 8 * q));
                sx[q] = -136.0f * sm_word_sum(xp[q]);
            }
#pragma unroll
            for (uint32_t j = 0; j < RPL; j++) {
                const uint32_t wj[4] = {(uint32_t)wv[i][j].x, (uint32_t)wv[i][j].y, (uint32_t)wv[i][j].z,
                                        (uint32_t)wv[i][j].w};
                if constexpr (SPW) {
#pragma unroll
                    for (uint32_t q = 0; q < 4; q++)
                        acc[j] = fmaf(sm_word_dot(wj[q], xp[q]) + sx[q], decode_scale(sv[i][j][q], A.scale_bf16), acc[j]);
                } else {
                    const float sc = decode_scale(sv[i][j][0], A.scale_bf16);
#pragma unroll
                    for (uint32_t q = 0; q < 4; q++) acc[j] = fmaf(sm_word_dot(wj[q], xp[q]) + sx[q], sc, acc[j]);
                }
            }
        }
    }

    // Row sums across the LU lanes of each row.
#pragma unroll
    for (uint32_t j = 0; j < RPL; j++) {
        acc[j] = lanes_sum_down<LU>(acc[j]);   // the __shfl_xor butterfly LU / 2, ..., 1
    }

    if constexpr (GATE_UP) {
        // Output row orow0 + t (t < OR) on lane t: gate = weight row t, up =
        // weight row OR + t.
        float gate = 0.0f, up = 0.0f;
#pragma unroll
        for (uint32_t li = 0; li < SM_WROWS; li++) {
            // lanes of row group li / RPL hold row li in acc[li % RPL]
            const float v = lane_bcast(acc[li % RPL], (li / RPL) * LU);
            if (li < OR && lane == li) gate = v;
            if (li >= OR && lane == li - OR) up = v;
        }
        const uint32_t row = orow0 + lane;
        if (lane < OR && row < A.N) {
            // …gate_up_int4_ct.comp.template:205-213
            const float g = round_bf16(gate), u = round_bf16(up);
            const float act = round_bf16(round_bf16(g / (1.0f + expf(-g))) * u);
            A.out[(uint64_t)b * A.frame_words * 2 + (uint64_t)r * A.I + row] = (uint16_t)f32_to_bf16(act);
        }
    } else {
        float y = 0.0f;
#pragma unroll
        for (uint32_t li = 0; li < SM_WROWS; li++) {
            const float v = lane_bcast(acc[li % RPL], (li / RPL) * LU);
            if (lane == li) y = v;
        }
        const uint32_t row = orow0 + lane;
        if (lane < OR && row < A.N) {
            // …down_int4_ct.comp.template:176-181
            const float wr = bf16_to_f32(rw >> 16);
            A.out[(uint64_t)c * A.N + row] = (uint16_t)f32_to_bf16(round_bf16(round_bf16(y) * wr));
        }
    }
}

// ---------------------------------------------------------------------------
// Tiles of routes on the matrix cores (groups of whole 32-column blocks,
// K % 128 == 0).
//
// A block owns a window of `group` route positions and 16 NW output channels.
// Positions of one expert that follow each other in the map form a run (the
// compaction sorts the map, so an expert is one run), and every TS-th position of
// a run starts a tile of up to TS routes.  The block takes the tiles that start
// in its window, so an expert's weights are decoded once per TS routes and not
// once per route.
//
// An owned range leaves the map in source order, where runs are mostly one route
// long, and fills only a part of it.  Its positions are dealt to all windows and a
// run is then the expert's positions within SM_CHUNK, whose expert ids the block
// stages in LDS where the tile's rows go afterwards (2 KB of their own cost
// K = 4096 its third block a CU: 16 tokens over 128 experts top 8 174 us against
// 163).  The routed block at h3072 i1024 e256 k10, us with a block per route /
// runs of neighbours in windows of the whole map / this: 32 owned experts and 103
// tokens 278 / 271 / 114, 128 and 256 1585 / 1847 / 635, 256 and 1024
// 10665 / 12618 / 5360.
//
// A wave owns 16 channels: 16 weight rows of gate and the same of up (down: 32
// rows).  Panels of PANEL columns of these rows stream through registers two
// panels ahead (whole 128-byte lines, nontemporal: every block reads weights of
// its own) into a wave-private LDS slot and are read back as MFMA operands: lane
// (g = l / 16, r = l % 16) takes word g of a 32-column block of row r, which
// the and-or expansion turns into the bf16 values 128 + q.  The tile's rows sit
// in LDS in the pair order of that expansion.  Per block
//   sum_k x (q - 8) = sum_k x (-136) + sum_k x (128 + q),
// two chained MFMAs (the first one serves both row tiles; the matrix cores have
// room for it, the LDS has little for stored sums), then acc = fma(that, scale,
// acc).  Rows past the tile's count are never written: they only reach result
// rows that are not stored.
//
// Bound: the weight stream (bytes of the distinct experts), with code expansion
// and LDS reads each at about half of their units and a chain of five dependent
// loads before a block's first weights.  Small panels and blocks (4 waves, 256
// columns: three blocks a CU) hide that chain best: the routed block at h3072
// i1024 e256 k10 with 16 tokens takes 180 us (213 with 512-column panels, 236
// with a block per route), 64 tokens 396 (761), 256 tokens 594 (2673).
// ---------------------------------------------------------------------------
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

__device__ __forceinline__ uint32_t sm_pair_exponent() {   // see pair_exponent() of the INT4 linears
    uint32_t e;
    asm("v_mov_b32 %0, 0x43004300" : "=v"(e));
    return e;
}

constexpr uint32_t SM_CHUNK = 1024;

// LDS rows are padded by 16 bytes: 16 rows' operand reads hit distinct banks
// at immediate offsets.  LDS bytes of one block:
constexpr uint32_t TILE_LDS_MOST = 160 * 1024 - 256;     // beside the static tables
constexpr uint32_t tile_lds(uint32_t K, uint32_t TS, uint32_t NW, uint32_t PANEL) {
    return TS * (K * 2 + 16) + NW * 2 * 16 * (PANEL / 2 + 16 + PANEL / 16);
}

template <bool GATE_UP, uint32_t TS, uint32_t NW, uint32_t PANEL, uint32_t WPE, bool SBF16>
__global__ __launch_bounds__(64 * NW, WPE) void sparse_tile_kernel(SmArgs A, uint32_t group, uint32_t gshift) {
    constexpr uint32_t PB = PANEL / 2, PP = PB / 16, PS = PANEL / 32;   // bytes, 16-byte pieces and scales of a panel row
    constexpr uint32_t NL = 16 * PP / 64;                               // weight loads per lane, row tile and panel
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ uint32_t t_route[TS], t_word[TS];
    const uint32_t K = A.K, N = A.N, ng = K / A.G, nblk = K / 32;   // G = 32 << gshift
    const uint32_t tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const uint32_t g = lane >> 4, rr = lane & 15;
    constexpr uint32_t WS = PB + 16;                                    // LDS stride of a weight row
    const uint32_t xstr = K * 2 + 16;
    uint8_t* xs = lds;                                                  // [TS] rows of K bf16 in pair order
    uint8_t* slot = lds + TS * xstr + wave * (2 * 16 * (WS + 2 * PS));
    uint16_t* sslot = reinterpret_cast<uint16_t*>(slot + 2 * 16 * WS);  // [2][16][PS]

    const uint32_t w = (blockIdx.x % 8) * A.per_xcd + blockIdx.x / 8;
    const uint32_t win = w % A.npos, tile = w / A.npos;                 // npos: windows
    if (tile >= A.tiles) return;
    const uint32_t cap = A.batch_width * A.k;
    const uint32_t n0 = tile * (NW * 16 * (GATE_UP ? 1 : 2)) + wave * (GATE_UP ? 16 : 32);
    const uint32_t exponent = sm_pair_exponent();

    uint32_t start = 0, count = 0, npos = cap;
    if (A.control) {
        start = A.control[1];
        count = A.control[2];
        if (A.batched && count != 0u) npos = min(cap, A.control[3]);
    }
    // Route and expert of position p (0xffffffff: none).
    auto route_at = [&](uint32_t p, uint32_t& c, uint32_t& word) -> uint32_t {
        c = p;
        word = 0;
        if (p >= npos) return 0xffffffffu;
        if (A.batched) c = A.frames[(uint64_t)(p / A.k) * A.frame_words + A.data_words + p % A.k];
        if (c >= cap) return 0xffffffffu;
        word = A.routes[c];
        const uint32_t e = word & 0xffffu;
        return (e >= A.E || (count != 0u && (e < start || e - start >= count))) ? 0xffffffffu : e;
    };
    // Owned: windows take every A.npos-th position, since the first positions of a
    // chunk hold most of its tiles.
    const bool owned = count != 0u;
    const uint32_t step = owned ? A.npos : 1u, last = owned ? npos : min(npos, (win + 1) * group);
    uint16_t* chunk_e = reinterpret_cast<uint16_t*>(lds);               // owned: experts of the chunk's positions
    uint32_t staged = 0xffffffffu;                                      // first position of the chunk in LDS
    for (uint32_t p = owned ? win : win * group; p < last; p += step) {
        // ---- the tile at position p, by every wave for itself.
        const uint32_t c0 = p / SM_CHUNK * SM_CHUNK, c1 = min(npos, c0 + SM_CHUNK);
        uint32_t e, back = 0, nt = 0, c = 0, word = 0;                  // back: positions of the run before p
        if (owned) {
            if (staged != c0) {
                __syncthreads();                                        // the previous tile's reads are done
                for (uint32_t i = c0 + tid; i < c1; i += 64 * NW) chunk_e[i - c0] = (uint16_t)route_at(i, c, word);
                __syncthreads();
                staged = c0;
            }
            e = (uint32_t)__builtin_amdgcn_readfirstlane((int)chunk_e[p - c0]);
            if (e == 0xffffu) continue;
            for (uint32_t i = c0; i < p; i += 64)
                back += (uint32_t)__popcll(__ballot(i + lane < p && chunk_e[i + lane - c0] == e));
            if (back % TS) continue;
        } else {
            // Lane l looks at position p + l (the tile's routes) and p - 1 - l (the
            // run's start).
            uint32_t cb, wb;
            const uint32_t ef = route_at(p + lane, c, word);
            uint32_t eb = route_at(lane < p ? p - 1 - lane : 0xffffffffu, cb, wb);
            e = (uint32_t)__builtin_amdgcn_readfirstlane((int)ef);
            if (e == 0xffffffffu) continue;
            for (;;) {
                const uint64_t other = __ballot(eb != e);
                if (other) {
                    back += (uint32_t)__builtin_ctzll(other);
                    break;
                }
                back += 64;
                eb = route_at(back + lane < p ? p - 1 - back - lane : 0xffffffffu, cb, wb);
            }
            if (back % TS) continue;
            const uint64_t fend = __ballot(ef != e);
            nt = min(TS, fend ? (uint32_t)__builtin_ctzll(fend) : 64u);
        }
        const uint32_t* W = static_cast<const uint32_t*>(sm_param(A, 2 * e, A.w_bytes, 16));
        const uint16_t* S = static_cast<const uint16_t*>(sm_param(A, 2 * e + 1, A.s_bytes, 2));
        if (!W || !S) continue;                                         // uniform over the block
        __syncthreads();                                                // the previous tile's reads are done
        if (owned) {
            for (uint32_t i = p; i < c1 && nt < TS; i += 64) {
                const bool mine = i + lane < c1 && chunk_e[i + lane - c0] == e;
                const uint64_t m = __ballot(mine);
                const uint32_t t = nt + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
                if (wave == 0 && mine && t < TS) {
                    route_at(i + lane, c, word);
                    t_route[t] = c;
                    t_word[t] = word;
                }
                nt += (uint32_t)__popcll(m);
            }
            nt = min(TS, nt);
            staged = 0xffffffffu;                                       // the rows overwrite the ids
        } else if (tid < TS) {
            t_route[tid] = c;
            t_word[tid] = word;
        }
        // ---- weight stream: row tile m's 16 rows start at row0[m].
        const uint32_t row0[2] = {min(n0, N - 16), GATE_UP ? A.I + min(n0, N - 16) : min(n0 + 16, N - 16)};
        const bool words = gshift == 0 && ((uintptr_t)S & 3) == 0;          // scales in dwords (K / 32 is even)
        struct Panel {
            v4i w[2][NL];
            uint32_t s[2][PS / 8];
        };
        auto load = [&](Panel& R, uint32_t k0) __attribute__((always_inline)) {
            if (k0 >= K) return;
#pragma unroll
            for (uint32_t m = 0; m < 2; m++) {
#pragma unroll
                for (uint32_t i = 0; i < NL; i++) {
                    const uint32_t x = i * 64 + lane, row = x / PP, pc = x % PP;
                    const v4i* wp = reinterpret_cast<const v4i*>(W + (uint64_t)(row0[m] + row) * (K / 8) + min(k0 / 32 + pc, nblk - 1) * 4);
                    R.w[m][i] = TS < 16 ? __builtin_nontemporal_load(wp) : *wp;
                }
                // Scales: lane (g, r) loads blocks PS / 4 g .. of row r.
                const uint16_t* sp = S + (uint64_t)(row0[m] + rr) * ng;
#pragma unroll
                for (uint32_t i = 0; i < PS / 8; i++) {
                    const uint32_t b = min(k0 / 32 + PS / 4 * g + 2 * i, nblk - 2);
                    if (words) R.s[m][i] = *reinterpret_cast<const uint32_t*>(sp + b);
                    else R.s[m][i] = (uint32_t)sp[b >> gshift] | ((uint32_t)sp[(b + 1) >> gshift] << 16);
                }
            }
        };
        Panel ra, rb;
        load(ra, 0);
        load(rb, PANEL);
        __syncthreads();                                                // t_route is written
        // ---- the tile's rows into LDS
        for (uint32_t x = tid; x < nt * (K / 8); x += 64 * NW) {
            const uint32_t t = x / (K / 8), o = x % (K / 8);
            const uint32_t ct = t_route[t], b = ct / A.k, r = ct % A.k;
            const uint16_t* xg = GATE_UP ? A.x + (uint64_t)b * K : A.x + (uint64_t)b * A.frame_words * 2 + (uint64_t)r * A.I;
            v4i v;
            __builtin_memcpy(&v, __builtin_assume_aligned(xg + 8 * o, 4), 16);
            *reinterpret_cast<v4i*>(xs + t * xstr + o * 16) = sm_permute(v);
        }
        __syncthreads();
        v4f acc[2] = {v4f{0.f, 0.f, 0.f, 0.f}, v4f{0.f, 0.f, 0.f, 0.f}};
        const v4i minus136 = v4i{(int)0xC308C308u, (int)0xC308C308u, (int)0xC308C308u, (int)0xC308C308u};
        const uint32_t tr = rr % TS;
        auto contract = [&](Panel& R, uint32_t k0) __attribute__((always_inline)) {
#pragma unroll
            for (uint32_t m = 0; m < 2; m++) {
#pragma unroll
                for (uint32_t i = 0; i < NL; i++) {
                    const uint32_t x = i * 64 + lane, row = x / PP, pc = x % PP;
                    *reinterpret_cast<v4i*>(slot + (m * 16 + row) * WS + pc * 16) = R.w[m][i];
                }
#pragma unroll
                for (uint32_t i = 0; i < PS / 8; i++)
                    *reinterpret_cast<uint32_t*>(sslot + (m * 16 + rr) * PS + PS / 4 * g + 2 * i) = R.s[m][i];
            }
            load(R, k0 + 2 * PANEL);
            __builtin_amdgcn_wave_barrier();
            const uint8_t* xp = xs + tr * xstr + k0 * 2 + 16 * g;
            const uint8_t* wq = slot + rr * WS + 4 * g;
#pragma unroll
            for (uint32_t ch = 0; ch < PANEL / 128; ch++) {
                if (k0 + 128 * ch >= K) break;                          // uniform
                v2i sv[2];
#pragma unroll
                for (uint32_t m = 0; m < 2; m++) sv[m] = *reinterpret_cast<const v2i*>(sslot + (m * 16 + rr) * PS + 4 * ch);
#pragma unroll
                for (uint32_t u = 0; u < 4; u++) {
                    const uint32_t pc = 4 * ch + u;
                    const v4i av = *reinterpret_cast<const v4i*>(xp + pc * 64);
                    const v4f cs = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, av), __builtin_bit_cast(v8bf, minus136),
                                                                           v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                    for (uint32_t m = 0; m < 2; m++) {
                        const uint32_t wd = *reinterpret_cast<const uint32_t*>(wq + m * 16 * WS + pc * 16);
                        const v4i bw = v4i{(int)((wd & 0x000F000Fu) | exponent), (int)(((wd >> 4) & 0x000F000Fu) | exponent),
                                           (int)(((wd >> 8) & 0x000F000Fu) | exponent), (int)(((wd >> 12) & 0x000F000Fu) | exponent)};
                        const v4f d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, av),
                                                                              __builtin_bit_cast(v8bf, bw), cs, 0, 0, 0);
                        const uint32_t sb = (uint32_t)sv[m][u / 2];
                        const float sc = !SBF16 ? (float)__builtin_bit_cast(_Float16, (uint16_t)(u % 2 ? sb >> 16 : sb))
                                         : __uint_as_float(u % 2 ? sb & 0xffff0000u : sb << 16);
#pragma unroll
                        for (int i = 0; i < 4; i++) acc[m][i] = fmaf(d[i], sc, acc[m][i]);
                    }
                }
            }
            __builtin_amdgcn_wave_barrier();
        };
        for (uint32_t k0 = 0; k0 < K; k0 += 2 * PANEL) {
            contract(ra, k0);
            if (k0 + PANEL < K) contract(rb, k0 + PANEL);
        }
        // ---- result lane (g, r): routes 4 g + i, row r of each row tile.
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) {
            const uint32_t t = 4 * g + i;
            if (t >= nt) continue;
            const uint32_t ct = t_route[t % TS];
            if constexpr (GATE_UP) {
                // …gate_up_int4_ct.comp.template:205-213
                if (n0 + rr >= N) continue;
                const float gv = round_bf16(acc[0][i]), uv = round_bf16(acc[1][i]);
                const float act = round_bf16(round_bf16(gv / (1.0f + expf(-gv))) * uv);
                A.out[(uint64_t)(ct / A.k) * A.frame_words * 2 + (uint64_t)(ct % A.k) * A.I + n0 + rr] = (uint16_t)f32_to_bf16(act);
            } else {
                // …down_int4_ct.comp.template:176-181
                const float wr = bf16_to_f32(t_word[t % TS] >> 16);
#pragma unroll
                for (uint32_t m = 0; m < 2; m++)
                    if (n0 + 16 * m + rr < N)
                        A.out[(uint64_t)ct * N + n0 + 16 * m + rr] = (uint16_t)f32_to_bf16(round_bf16(round_bf16(acc[m][i]) * wr));
            }
        }
    }
}

template <bool GATE_UP, uint32_t TS, uint32_t NW, uint32_t PANEL, uint32_t WPE>
nerve_hip_status launch_tile_form(SmArgs A, uint32_t group, hipStream_t stream) {
    const uint32_t rows = NW * 16 * (GATE_UP ? 1 : 2), lds = tile_lds(A.K, TS, NW, PANEL);
    A.tiles = (A.N + rows - 1) / rows;
    A.npos = (A.npos + group - 1) / group;
    A.per_xcd = (uint32_t)(((uint64_t)A.npos * A.tiles + 7) / 8);
    auto* kernel = A.scale_bf16 ? sparse_tile_kernel<GATE_UP, TS, NW, PANEL, WPE, true> : sparse_tile_kernel<GATE_UP, TS, NW, PANEL, WPE, false>;
    static bool attr_set[2] = {false, false};
    if (!attr_set[A.scale_bf16 ? 1 : 0]) {
        if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, TILE_LDS_MOST) != hipSuccess)
            return nh::fail(NERVE_HIP_DEVICE_ERROR, "hipFuncSetAttribute failed for sparse_tile_kernel");
        attr_set[A.scale_bf16 ? 1 : 0] = true;
    }
    kernel<<<A.per_xcd * 8, 64 * NW, lds, stream>>>(A, group, (uint32_t)__builtin_ctz(A.G / 32));
    return nh::check_launch(GATE_UP ? "int4_moe_gate_up" : "int4_moe_down");
}

// The tile form, or UNSUPPORTED where its loads do not fit or where a block per
// route is the faster one.
template <bool GATE_UP>
nerve_hip_status launch_tiles(const SmArgs& A, uint32_t cus, hipStream_t stream) {
    if (A.G % 32 || (A.G & (A.G - 1)) || A.K % 128 || A.N % 16) return NERVE_HIP_UNSUPPORTED;
    // Few blocks: a tile's chain (route, record, rows, panels two ahead) is longer
    // than that of the kernel per route, which has all of its weights in flight at
    // once, and only several rounds of blocks hide it.  One token, gate_up, us by
    // tile / by route: h3072 i1024 top 10 20.4 / 15.1, h2048 i768 top 4 13.9 / 6.8;
    // from 8 blocks a CU on: 160 routes of h3072 i1024 93.8 / 115.4, 96 of h2048
    // i1408 48.3 / 59.1.
    const uint64_t rows = GATE_UP ? 64 : 128;
    if ((uint64_t)A.npos * ((A.N + rows - 1) / rows) < 8ull * cus) return NERVE_HIP_UNSUPPORTED;
    // Routes per expert if they spread evenly.  Groups longer than 32 take their
    // scales two bytes a load and need two (60 experts, h2048 i1408 g64, 64 routes
    // 53.5 / 42.3, 128 routes 73.4 / 76.6).
    const uint32_t per = A.npos / A.E;
    if (A.G != 32 && per < 2) return NERVE_HIP_UNSUPPORTED;
    // A tile takes 4, 8 or 16 routes: its rows in LDS (2 K bytes each) cost blocks
    // per CU.  The routed block at h3072 i1024 e256 k10, us by tile size 4 / 8 / 16
    // at 16, 64 and 256 tokens: 180 / 191 / 219, 396 / 403 / 457, 976 / 740 / 594.
    // Blocks of four waves need a second one on the CU (gate_up of 128 routes of 16
    // experts, K = 4096, by 4 / 8 / route: 484 / 581 / 1048 us; down of 64 routes of
    // 8, K = 14336, 403 by 4, 282 by route), or 8 routes from four per expert on
    // (128 routes of 32, K = 8192: 460 / 731).
    const uint32_t lds4 = tile_lds(A.K, 4, 4, 256), lds8 = tile_lds(A.K, 8, 4, 256), lds16 = tile_lds(A.K, 16, 8, 256);
    constexpr uint32_t LDS = 160 * 1024;
    uint32_t ts = per < 3 ? 4 : per < 8 ? 8 : 16;
    if (ts == 16 && lds16 > TILE_LDS_MOST) ts = 8;
    if (2 * lds4 > LDS) {
        if (per < 4 || lds8 > TILE_LDS_MOST) return NERVE_HIP_UNSUPPORTED;
        ts = 8;
    } else if (ts == 8 && 2 * lds8 > LDS) {
        ts = 4;
    }
    // Windows of 8 positions where most of them start no tile.
    const uint32_t group = per >= 4 ? 8 : 1;
    if (ts == 4) return launch_tile_form<GATE_UP, 4, 4, 256, 3>(A, group, stream);
    if (ts == 8) return launch_tile_form<GATE_UP, 8, 4, 256, 2>(A, group, stream);
    return launch_tile_form<GATE_UP, 16, 8, 256, 2>(A, group, stream);
}

template <bool GATE_UP>
nerve_hip_status launch_sparse(const SmArgs& A, uint32_t cus, hipStream_t stream) {
    const nerve_hip_status tiled = launch_tiles<GATE_UP>(A, cus, stream);
    if (tiled != NERVE_HIP_UNSUPPORTED) return tiled;
    const uint32_t units = A.K / 32;
    const bool spw = A.G % 32 != 0;
    const uint32_t lu = units % 64 == 0 ? 64u : (units % 32 == 0 || units > 32) ? 32u : 16u;
    const dim3 grid(A.per_xcd * 8), block(64 * SM_WAVES);
#define SM_LAUNCH(LU, SPW) sparse_int4_kernel<GATE_UP, LU, SPW><<<grid, block, A.K * 2, stream>>>(A)
    if (spw) {
        if (lu == 64) SM_LAUNCH(64, true);
        else if (lu == 32) SM_LAUNCH(32, true);
        else SM_LAUNCH(16, true);
    } else {
        if (lu == 64) SM_LAUNCH(64, false);
        else if (lu == 32) SM_LAUNCH(32, false);
        else SM_LAUNCH(16, false);
    }
#undef SM_LAUNCH
    return nh::check_launch(GATE_UP ? "int4_moe_gate_up" : "int4_moe_down");
}

nerve_hip_status sparse_common(nerve_hip_ctx* ctx, const char* spec, bool gate_up, const void* x,
                               const void* routes, void* intermediates, void* expert_outputs,
                               const void* addresses, uint32_t address_records, const void* slots,
                               uint32_t slot_words, const void* control, uint32_t batch_width, void* stream) {
    nerve_hip_status st = nh::enter(ctx);
    if (st) return st;
    nh::MoeSpec ms;
    if ((st = nh::parse_moe_spec(spec, &ms))) return st;
    if (ms.family != 1) return nh::fail(NERVE_HIP_INVALID_SPEC, std::string("not an INT4 sparse expert kernel: ") + spec);
    if (ms.gate_up != gate_up)
        return nh::fail(NERVE_HIP_INVALID_SPEC, gate_up ? "gate_up entry given a down specialization"
                                                        : "down entry given a gate_up specialization");
    if (!x || !routes || !intermediates || !addresses || !slots || (gate_up ? false : !expert_outputs) ||
        (ms.batch1 && !control))
        return nh::fail(NERVE_HIP_INVALID_ARGUMENT, "null buffer");
    const uint32_t H = ms.hidden, I = ms.inter, k = ms.k;
    const uint32_t K = gate_up ? H : I, N = gate_up ? I : H;
    if (K % 32) return nh::fail(NERVE_HIP_UNSUPPORTED, "INT4 sparse experts need an input width that is a multiple of 32");
    if (K > SM_MAX_K) return nh::fail(NERVE_HIP_UNSUPPORTED, "INT4 sparse experts take input widths up to 16384");
    if (!ms.batch1 && batch_width != 1)
        return nh::fail(NERVE_HIP_INVALID_ARGUMENT, "the unbatched INT4 expert form runs one token (batch_width 1)");
    if (((uintptr_t)x | (uintptr_t)intermediates) & 3) return nh::fail(NERVE_HIP_INVALID_ARGUMENT, "activation buffers must be 4-byte aligned");
    const uint64_t cap = (uint64_t)batch_width * k;
    if (cap == 0) return nh::ok();
    if (cap > (1u << 24)) return nh::fail(NERVE_HIP_UNSUPPORTED, "too many routes");
    SmArgs A{};
    A.x = static_cast<const uint16_t*>(x);
    A.routes = static_cast<const uint32_t*>(routes);
    A.frames = static_cast<const uint32_t*>(intermediates);
    A.out = static_cast<uint16_t*>(gate_up ? intermediates : expert_outputs);
    A.addr = static_cast<const uint32_t*>(addresses);
    A.slots = static_cast<const uint32_t*>(slots);
    A.control = static_cast<const uint32_t*>(control);
    A.n_records = address_records;
    A.n_slot_words = slot_words;
    A.batch_width = batch_width;
    A.k = k;
    A.E = ms.experts;
    A.K = K;
    A.N = N;
    A.I = I;
    A.G = ms.group;
    A.data_words = k * I / 2;
    A.frame_words = (uint64_t)A.data_words + (ms.batch1 ? k : 0u);
    A.tiles = (N + SM_WAVES * (gate_up ? SM_WROWS / 2 : SM_WROWS) - 1) / (SM_WAVES * (gate_up ? SM_WROWS / 2 : SM_WROWS));
    A.npos = (uint32_t)cap;
    A.per_xcd = (uint32_t)(((uint64_t)A.npos * A.tiles + 7) / 8);
    const uint64_t wrows = gate_up ? 2ull * I : (uint64_t)H;
    A.w_bytes = wrows * K / 2;
    A.s_bytes = wrows * (K / ms.group) * 2;
    A.batched = ms.batch1 ? 1 : 0;
    A.scale_bf16 = ms.scale_bf16;
    const uint32_t cus = (uint32_t)ctx->cu_count;
    return gate_up ? launch_sparse<true>(A, cus, (hipStream_t)stream) : launch_sparse<false>(A, cus, (hipStream_t)stream);
}

}  // namespace

extern "C" {

nerve_hip_status nerve_hip_int4_moe_gate_up(nerve_hip_ctx* ctx, const char* spec, const void* hidden_bf16,
                                            const void* routes_u32, void* intermediates, const void* addresses_u32,
                                            uint32_t address_records, const void* param_slots_u32,
                                            uint32_t param_slot_words, const void* control_u32, uint32_t batch_width,
                                            void* stream) {
    return sparse_common(ctx, spec, true, hidden_bf16, routes_u32, intermediates, nullptr, addresses_u32,
                         address_records, param_slots_u32, param_slot_words, control_u32, batch_width, stream);
}

nerve_hip_status nerve_hip_int4_moe_down(nerve_hip_ctx* ctx, const char* spec, const void* intermediates,
                                         const void* routes_u32, void* expert_outputs, const void* addresses_u32,
                                         uint32_t address_records, const void* param_slots_u32,
                                         uint32_t param_slot_words, const void* control_u32, uint32_t batch_width,
                                         void* stream) {
    return sparse_common(ctx, spec, false, intermediates, routes_u32, const_cast<void*>(intermediates),
                         expert_outputs, addresses_u32, address_records, param_slots_u32, param_slot_words,
                         control_u32, batch_width, stream);
}

}  // extern "C"
