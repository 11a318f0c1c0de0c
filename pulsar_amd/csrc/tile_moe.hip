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
// pairs in tiles of 16 NS one after the other.
template <uint32_t Q, bool PAIR, uint32_t NS>
__global__ __launch_bounds__(256, 2) void tile_experts_kernel(float *__restrict__ out, const ExpertGroups src,
                                                              const float *__restrict__ weights,
                                                              const pulsar_block_q8_K *__restrict__ act, uint32_t nb,
                                                              uint32_t n_rows, uint32_t n_used, uint64_t row_bytes,
                                                              uint32_t act_op) {
    using GT = GroupTile<Q, PAIR, NS>;
    __shared__ __align__(16) uint8_t buf0[GT::T::kBuf];
    __shared__ __align__(16) uint8_t buf1[GT::T::kBuf];
    __shared__ uint32_t pr_l[GT::T::kTok];
    extern __shared__ uint32_t lst[];
    const ExpertGroups::Group grp = src.group(blockIdx.y);
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
// kernel alike. The 16-row kernel of mmq.hip wastes less on
// short groups and its smaller blocks keep more weight bytes in flight; for
// Q3_K and IQ4_XS the lane kernels. Both sides by pairs per expert (us, gate /
// up stage of 128-expert layers unless noted, the tile second): Q4_K 2048 x
// 768: 4: 66 / 66, 6: 87 / 69, 14: 152 / 73; Q2_K 4096 x 1536: 2.5: 145 / 190,
// 4: 210 / 195, 14: 577 / 207; IQ2_XXS: 4: 255 / 345, 6: 365 / 347, 14: 693 / 353;
// Q5_K: 6: 107 / 96, 14: 198 / 106; IQ4_XS: 1: 62 / 68, 2.5: 124 / 83, 14: 515 /
// 93; Q3_K 64 experts of 2048 x 1024: 0.8: 35 / 44, 1.5: 57 / 51, 21: 568 / 62.
// Down stages, whose rows have few super-blocks: Q6_K 768 x 2048: 16: 98 / 115;
// Q2_K 1536 x 4096: 14: 186 / 124; IQ2_XXS: 14: 191 / 195; Q5_K: 14: 77 / 58.
uint32_t tile_min_quarter_pairs(bool pair, uint32_t quant) {
    switch (quant) {
    case PULSAR_QUANT_Q4_K:
    case PULSAR_QUANT_Q5_K: return pair ? 20u : 48u;
    case PULSAR_QUANT_Q6_K: return pair ? 48u : 128u;
    case PULSAR_QUANT_Q2_K: return pair ? 16u : 48u;
    case PULSAR_QUANT_IQ2_XXS: return pair ? 24u : 60u;
    case PULSAR_QUANT_Q3_K:
    case PULSAR_QUANT_IQ4_XS: return 6u;
    default: return 0u;
    }
}

#define PK_TILE_FORMATS(F)                                                                                            \
    F(PULSAR_QUANT_Q4_K) F(PULSAR_QUANT_Q5_K) F(PULSAR_QUANT_Q6_K) F(PULSAR_QUANT_Q2_K) F(PULSAR_QUANT_Q3_K)          \
    F(PULSAR_QUANT_IQ4_XS) F(PULSAR_QUANT_IQ2_XXS)

// The grouped stages of an ExpertGroups source on the tile, n_group groups.
int launch_tile_experts(bool pair, uint32_t quant, float *out, const ExpertGroups &src, const float *weights,
                        const pulsar_block_q8_K *act, uint32_t k_dim, uint32_t n_rows, uint32_t n_used,
                        uint32_t n_group, uint64_t row_bytes, uint32_t act_op, uint32_t lst_bytes) {
#define PK_LAUNCH(Q, P)                                                                                               \
    hipLaunchKernelGGL((tile_experts_kernel<Q, P, 4>),                                                                \
                       dim3((n_rows + GroupTile<Q, P, 4>::kRows - 1u) / GroupTile<Q, P, 4>::kRows, n_group), dim3(256), \
                       lst_bytes, pk::stream(), out, src, weights, act, k_dim / 256u, n_rows, n_used, row_bytes, act_op)
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
