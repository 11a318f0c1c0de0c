// tile_moe.hip - the grouped expert stages on the wide matrix-core tile
// (pk_tile.h).
#include "pk_tile.h"
#include "pk_route.h"

namespace pk {

// One pair tile of a group: rows [rb, rb + kRows) of expert p times the np
// pairs that pair(t) gives. PAIR: row tile 0 of a wave is 16 gate rows, row
// tile 1 the same rows of up, so a lane ends with both values of a (row, pair)
// and applies the combine itself.
template <uint32_t Q, bool PAIR, uint32_t NS>
struct GroupTile {
    using T = GroupedTile<Q, NS>;
    static constexpr uint32_t kRows = PAIR ? 64u : 128u;

    template <typename PairOf>
    PK_DEV static void run(uint8_t *buf0, uint8_t *buf1, const uint2 *lut, uint32_t *pr_l, float *out,
                           const pulsar_expert_ptrs &p, const float *weights, const pulsar_block_q8_K *act, uint32_t nb,
                           uint32_t n_rows, uint32_t n_used, uint64_t row_bytes, uint32_t act_op, uint32_t rb,
                           uint32_t np, PairOf pair_of) {
        const uint32_t lane = threadIdx.x & 63u, i = lane & 15u, q = lane >> 4, wave = threadIdx.x >> 6;
        const uint32_t row0 = rb + (PAIR ? 16u : 32u) * wave + i, row1 = PAIR ? row0 : row0 + 16u;
        const uint8_t *m0 = (const uint8_t *)(PAIR ? p.gate : p.down), *m1 = (const uint8_t *)(PAIR ? p.up : p.down);
        const uint8_t *w0 = as_global(m0) + (uint64_t)(row0 < n_rows ? row0 : n_rows - 1u) * row_bytes;
        const uint8_t *w1 = as_global(m1) + (uint64_t)(row1 < n_rows ? row1 : n_rows - 1u) * row_bytes;
        const float gb = PAIR && p.gate_b && row0 < n_rows ? ldwf(p.gate_b + row0) : 0.0f;
        const float ub = PAIR && p.up_b && row0 < n_rows ? ldwf(p.up_b + row0) : 0.0f;
        __syncthreads();  // the previous tile's pairs are stored
        if (threadIdx.x < np) pr_l[threadIdx.x] = pair_of(threadIdx.x);
        __syncthreads();
        T tile;
        auto row = [&](uint32_t t) {
            const uint32_t pr = pr_l[t];
            return PAIR ? pr >> 4 : (pr >> 4) * n_used + (pr & 15u);
        };
        auto part = [&](auto nc) {
            constexpr uint32_t NC = decltype(nc)::value;
            tile.template run<NC>(buf0, buf1, lut, w0, w1, nb, np, (const uint8_t *)act, row);
#pragma unroll
            for (uint32_t n = 0; n < NC; n++)
#pragma unroll
                for (uint32_t r = 0; r < 4; r++) {
                    const uint32_t t = 16u * n + 4u * q + r;
                    if (t >= np) continue;
                    const uint32_t pr = pr_l[t];
                    const uint64_t so = (uint64_t)(pr >> 4) * n_used + (pr & 15u);
                    float *o = out + so * n_rows;
                    if (PAIR) {
                        float gv = tile.acc[n][0][r], uv = tile.acc[n][1][r];
                        if (p.gate_b) gv += gb;
                        if (p.up_b) uv += ub;
                        if (row0 < n_rows) o[row0] = glu(gv, uv, act_op) * weights[so];
                    } else {
                        if (row0 < n_rows) o[row0] = tile.acc[n][0][r];
                        if (row1 < n_rows) o[row1] = tile.acc[n][1][r];
                    }
                }
        };
        // the 16-token slices that hold pairs
        if (np <= 16u)
            part(std::integral_constant<uint32_t, 1>{});
        else if (np <= 32u)
            part(std::integral_constant<uint32_t, 2>{});
        else if (NS > 4u && np <= 64u)
            part(std::integral_constant<uint32_t, 4>{});
        else
            part(std::integral_constant<uint32_t, NS>{});
    }
};

// Groups found from the router's ids: block = (row block, group), the group's
// pairs in tiles of 16 NS one after the other. shared_only: the groups are the
// shared slots' alone.
template <uint32_t Q, bool PAIR, uint32_t NS>
__global__ __launch_bounds__(256, 2) void tile_experts_kernel(float *__restrict__ out, const ExpertGroups src,
                                                              const float *__restrict__ weights,
                                                              const pulsar_block_q8_K *__restrict__ act, uint32_t nb,
                                                              uint32_t n_rows, uint32_t n_used, uint64_t row_bytes,
                                                              uint32_t act_op, uint32_t shared_only) {
    using GT = GroupTile<Q, PAIR, NS>;
    __shared__ __align__(16) uint8_t buf0[GT::T::kBuf];
    __shared__ __align__(16) uint8_t buf1[GT::T::kBuf];
    __shared__ uint32_t pr_l[GT::T::kTok];
    extern __shared__ uint32_t lst[];
    const ExpertGroups::Group grp = shared_only ? src.shared_group(blockIdx.y) : src.group(blockIdx.y);
    const pulsar_expert_ptrs &p = grp.p;
    const bool nul = grp.is_null();  // block-uniform, as every exit below
    if (!nul && !(PAIR ? p.gate && p.up : p.down != nullptr)) return;
    uint32_t s0, s1;
    src.range_block(grp, lst, s0, s1);
    if (s0 >= s1) return;
    const uint32_t rb = blockIdx.x * GT::kRows;
    if (nul) {  // unrouted slots: their rows of this block are 0
        for (uint32_t it = threadIdx.x; it < (s1 - s0) * GT::kRows; it += 256u) {
            const uint32_t pr = lst[s0 + it / GT::kRows], row = rb + it % GT::kRows;
            if (row < n_rows) out[((uint64_t)(pr >> 4) * n_used + (pr & 15u)) * n_rows + row] = 0.0f;
        }
        return;
    }
    PK_FMT_LUT(Q)
    for (uint32_t t0 = s0; t0 < s1; t0 += GT::T::kTok)
        GT::run(buf0, buf1, lut, pr_l, out, p, weights, act, nb, n_rows, n_used, row_bytes, act_op, rb,
                s1 - t0 < GT::T::kTok ? s1 - t0 : GT::T::kTok, [&](uint32_t t) { return lst[t0 + t]; });
}

// A caller's CSR, whose group sizes only the device knows. A launch of
// kTileSlots blocks, however few the groups: each counts the tiles of every group (one round trip),
// and block b takes the (tile, row block) items b, b + grid, ...: uneven groups
// spread evenly, and where the groups are short on average (the kernel launched
// before has taken them) the blocks end after one load.
template <uint32_t Q, bool PAIR, uint32_t NS>
__global__ __launch_bounds__(256, 2) void tile_csr_kernel(float *__restrict__ out, const CsrGroups src,
                                                          const float *__restrict__ weights,
                                                          const pulsar_block_q8_K *__restrict__ act, uint32_t nb,
                                                          uint32_t n_rows, uint32_t n_used, uint64_t row_bytes,
                                                          uint32_t act_op) {
    using GT = GroupTile<Q, PAIR, NS>;
    constexpr uint32_t kTok = GT::T::kTok;
    if (!src.tiled()) return;
    const uint32_t n_group = src.n_group;
    __shared__ __align__(16) uint8_t buf0[GT::T::kBuf];
    __shared__ __align__(16) uint8_t buf1[GT::T::kBuf];
    __shared__ uint32_t pr_l[kTok];
    __shared__ uint32_t first[kCsrGroups + 1u];  // tiles before group g
    __shared__ uint32_t wsum[4];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    uint32_t n[4], sum = 0u;  // groups 4 tid .. 4 tid + 3
#pragma unroll
    for (uint32_t k = 0; k < 4u; k++) {
        const uint32_t g = 4u * tid + k;
        const uint32_t b = src.starts[g < n_group ? g : n_group], e = src.starts[g < n_group ? g + 1u : n_group];
        n[k] = e > b ? (e - b + kTok - 1u) / kTok : 0u;
        sum += n[k];
    }
    uint32_t incl = sum;
#pragma unroll
    for (uint32_t d = 1; d < 64u; d <<= 1) {
        const uint32_t o = (uint32_t)__shfl_up((int)incl, d, 64);
        incl += lane >= d ? o : 0u;
    }
    if (lane == 63u) wsum[wave] = incl;
    __syncthreads();
    uint32_t at = incl - sum;
#pragma unroll
    for (uint32_t w = 0; w < 3u; w++) at += w < wave ? wsum[w] : 0u;
#pragma unroll
    for (uint32_t k = 0; k < 4u; k++) {
        first[4u * tid + k] = at;
        at += n[k];
    }
    if (tid == 255u) first[kCsrGroups] = at;
    PK_FMT_LUT(Q)
    __syncthreads();
    const uint32_t n_rb = (n_rows + GT::kRows - 1u) / GT::kRows;
    const uint64_t total = (uint64_t)first[kCsrGroups] * n_rb;
    for (uint64_t item = blockIdx.x; item < total; item += gridDim.x) {
        const uint32_t tl = (uint32_t)(item / n_rb), rb = (uint32_t)(item % n_rb) * GT::kRows;
        uint32_t g = 0u;  // the last group with first[g] <= tl
#pragma unroll
        for (uint32_t s = kCsrGroups / 2u; s != 0u; s >>= 1)
            if (first[g + s] <= tl) g += s;
        g = (uint32_t)__builtin_amdgcn_readfirstlane((int)g);
        const pulsar_expert_ptrs p = src.gptrs[g];
        if (!(PAIR ? p.gate && p.up : p.down != nullptr)) continue;  // block-uniform
        const uint32_t t0 = src.starts[g] + (tl - first[g]) * kTok, t1 = src.starts[g + 1u];
        GT::run(buf0, buf1, lut, pr_l, out, p, weights, act, nb, n_rows, n_used, row_bytes, act_op, rb,
                t1 - t0 < kTok ? t1 - t0 : kTok, [&](uint32_t t) { return src.pairs[t0 + t]; });
    }
}

// Pairs per group, in quarters, from which the tile beats the kernel it takes
// over from (0: no tile kernel); a CSR's mean decides on the device, in either
// kernel alike. nb: super-blocks of a row; groups, n_rows: the stage's;
// pmax: pairs per tile of the 16-row kernel (mmq.hip), 0 where it cannot hold a
// row.
//
// The 16-row kernel reads an expert's weights once per pmax pairs, the tile once
// per 64 or 128 with more work per super-block: a group of m pairs costs the one
// about m / pmax + 1/2 passes and the other a fixed number of them, which grows
// with the row length (a pass over a short row is mostly its staging) up to a
// bound. That number, in hundredths, is fitted to stages timed on both (10 layer
// shapes of 8 to 256 experts, rows of 2 to 56 super-blocks, gate / up of 8 and
// more, 1 to 400 pairs per expert, weights from HBM). It is lower for groups
// found from the router's ids, which the 16-row kernel scans a wave at a time
// before its passes, than for a CSR, where the tile is a launch of its own.
//   router's ids, 1444 stages: none more than 1% slower than on the 16-row
//   kernel, the faster kernel missed by 0.7% on average. us by pairs per expert,
//   16-row / tile: gate / up IQ2_XXS 128 experts of 1536 x 4096, 4: 239 / 321,
//   6: 331 / 330, 12: 615 / 338; 32 of 2816 x 2816, 6: 82 / 123, 10: 139 / 126;
//   Q2_K 16 of 6400 x 4096, 4: 77 / 90, 8: 133 / 117; Q4_K 128 of 768 x 2048, 4:
//   74 / 70; down Q6_K 128 of 2048 x 768, 12: 88 / 97, 16: 112 / 100.
//   CSR, 2024 stages: 5 more than 3% slower (the worst 13%), the faster kernel
//   missed by 0.1% on average. Gate / up Q4_K 128 of 768 x 2048, 7: 73 / 78, 8:
//   85 / 79; Q2_K 128 of 1536 x 4096, 6: 205 / 225, 7: 231 / 227; IQ2_XXS, 7: 294 /
//   349, 8: 364 / 352; down Q6_K 128 of 2048 x 768, 24: 105 / 109, 28: 115 / 111;
//   Q4_K 256 of 2048 x 512, 12: 66 / 75, 16: 81 / 79.
// Where a launch's blocks leave CUs idle the 16-row kernel's passes are one
// after the other (router's ids, 8 experts of 2048 x 4096, IQ2_XXS, 4: 56 / 48).
// Against the lane kernels the line lies at 2 to 3 pairs for the rows the
// 16-row kernel cannot hold (8 experts of 4096 x 14336, down, lane / tile, 2:
// Q6_K 216 / 188, Q4_K 169 / 103, IQ2_XXS 119 / 163; 3: IQ2_XXS 179 / 164) and
// at 1.5 (CSR: 2) for Q3_K and IQ4_XS (router's ids, IQ4_XS 128 of 768 x 2048,
// 1: 51 / 57, 1.5: 89 / 72), half a pair later in down stages of one or two
// super-blocks.
uint32_t tile_min_quarter_pairs(bool csr, bool pair, uint32_t quant, uint32_t nb, uint32_t n_rows, uint32_t groups,
                                uint32_t pmax) {
    struct Passes {
        uint32_t base, per_sb, most;
    } p;
    switch (quant) {
    case PULSAR_QUANT_Q4_K:
        p = csr ? pair ? Passes{45, 10, 150} : Passes{125, 2, 150} : pair ? Passes{70, 5, 150} : Passes{45, 10, 160};
        break;
    case PULSAR_QUANT_Q5_K:
        p = csr ? pair ? Passes{60, 10, 170} : Passes{140, 6, 170} : pair ? Passes{93, 5, 180} : Passes{68, 13, 170};
        break;
    case PULSAR_QUANT_Q6_K:
        p = csr ? pair ? Passes{40, 18, 230} : Passes{195, 4, 280} : pair ? Passes{100, 8, 220} : Passes{90, 15, 290};
        break;
    case PULSAR_QUANT_Q2_K:
        p = csr ? pair ? Passes{125, 4, 210} : Passes{150, 2, 170} : pair ? Passes{84, 6, 180} : Passes{65, 13, 170};
        break;
    case PULSAR_QUANT_IQ2_XXS:
        p = csr ? pair ? Passes{130, 6, 280} : Passes{145, 28, 230} : pair ? Passes{90, 10, 260} : Passes{120, 15, 240};
        break;
    case PULSAR_QUANT_Q3_K:
    case PULSAR_QUANT_IQ4_XS: return (csr ? 8u : 6u) + (!pair && nb <= 2u ? 2u : 0u);
    default: return 0u;
    }
    if (pmax == 0u) return quant == PULSAR_QUANT_IQ2_XXS ? 12u : 8u;
    uint32_t passes = p.base + p.per_sb * (pair && nb < 8u ? 8u : nb);
    if (passes > p.most) passes = p.most;
    const uint32_t rows = pair ? 64u : 128u;
    if (quant != PULSAR_QUANT_Q6_K && (uint64_t)((n_rows + rows - 1u) / rows) * groups <= 256u && passes > 130u)
        passes = 130u;
    const uint32_t bound = passes > 50u ? ((passes - 50u) * pmax * 4u + 99u) / 100u : 0u;
    return bound > 8u ? bound : 8u;
}

#define PK_TILE_FORMATS(F)                                                                                            \
    F(PULSAR_QUANT_Q4_K) F(PULSAR_QUANT_Q5_K) F(PULSAR_QUANT_Q6_K) F(PULSAR_QUANT_Q2_K) F(PULSAR_QUANT_Q3_K)          \
    F(PULSAR_QUANT_IQ4_XS) F(PULSAR_QUANT_IQ2_XXS)

// The grouped stages of an ExpertGroups source on the tile, n_group groups
// (shared_only: the shared slots).
int launch_tile_experts(bool pair, uint32_t quant, float *out, const ExpertGroups &src, const float *weights,
                        const pulsar_block_q8_K *act, uint32_t k_dim, uint32_t n_rows, uint32_t n_used,
                        uint32_t n_group, uint64_t row_bytes, uint32_t act_op, uint32_t lst_bytes, bool shared_only) {
#define PK_LAUNCH(Q, P)                                                                                               \
    hipLaunchKernelGGL((tile_experts_kernel<Q, P, 4>),                                                                \
                       dim3((n_rows + GroupTile<Q, P, 4>::kRows - 1u) / GroupTile<Q, P, 4>::kRows, n_group), dim3(256), \
                       lst_bytes, pk::stream(), out, src, weights, act, k_dim / 256u, n_rows, n_used, row_bytes,      \
                       act_op, (uint32_t)shared_only)
#define PK_CASE(Q)                  \
    case Q:                         \
        if (pair)                   \
            PK_LAUNCH(Q, true);     \
        else                        \
            PK_LAUNCH(Q, false);    \
        break;
    switch (quant) {
        PK_TILE_FORMATS(PK_CASE)
    default: return reject("grouped tile (quant)");
    }
#undef PK_LAUNCH
    return launch_ok(pair ? "moe pair swiglu experts (tile) launch" : "moe down experts (tile) launch");
}

// The grouped stages of a caller's CSR on the tile, where src.tiled() (what the
// kernel launched before it on the same src leaves). 128-pair tiles where the
// format's registers allow it (Q2_K gate / up, 96 pairs per group: 685 -> 562
// us, 16 pairs 240 / 235; Q4_K spills: 279 -> 319).
int launch_tile_csr(bool pair, uint32_t quant, float *out, const CsrGroups &src, const float *weights,
                    const pulsar_block_q8_K *act, uint32_t k_dim, uint32_t n_rows, uint32_t n_used,
                    uint64_t row_bytes, uint32_t act_op) {
    if (src.n_group > kCsrGroups) return reject("grouped tile (groups)");
#define PK_LAUNCH(Q, P)                                                                                              \
    do {                                                                                                             \
        constexpr uint32_t NS = Q == PULSAR_QUANT_Q4_K || Q == PULSAR_QUANT_Q5_K ? 4 : 8;                            \
        hipLaunchKernelGGL((tile_csr_kernel<Q, P, NS>), dim3(kTileSlots), dim3(256), 0, pk::stream(), out, src,      \
                           weights, act, k_dim / 256u, n_rows, n_used, row_bytes, act_op);                           \
    } while (0)
    switch (quant) {
        PK_TILE_FORMATS(PK_CASE)
    default: return reject("grouped tile (quant)");
    }
#undef PK_CASE
#undef PK_LAUNCH
    return launch_ok(pair ? "moe pair swiglu grouped (tile) launch" : "moe down grouped (tile) launch");
}

}  // namespace pk
