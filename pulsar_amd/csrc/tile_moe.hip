// tile_moe.hip - the grouped expert stages on the wide matrix-core tile
// (pk_tile.h).
#include "pk_tile.h"
#include "pk_route.h"

namespace pk {

// Grouped expert stages: block = (row block, expert group), the group's
// (token, slot) pairs in tiles of 16 NS. PAIR: row tile 0 of a wave is 16 gate
// rows, row tile 1 the same rows of up, so a lane ends with both values of a
// (row, pair) and applies the combine itself.
template <uint32_t Q, bool PAIR, uint32_t WR, uint32_t WK, uint32_t NS, typename G>
__global__ __launch_bounds__(256, 2) void tile_grouped_kernel(float *__restrict__ out, const G src,
                                                              const float *__restrict__ weights,
                                                              const pulsar_block_q8_K *__restrict__ act, uint32_t nb,
                                                              uint32_t n_rows, uint32_t n_used, uint64_t row_bytes,
                                                              uint32_t act_op, uint32_t min_pairs) {
    using T = Tile<Q, WR, WK, NS>;
    constexpr uint32_t kRows = PAIR ? 16u * WR : 32u * WR;
    __shared__ __align__(16) uint8_t buf0[T::kBuf];
    __shared__ __align__(16) uint8_t buf1[T::kBuf];
    __shared__ uint32_t pr_l[T::kTok];
    extern __shared__ uint32_t lst[];
    const typename G::Group grp = src.group(blockIdx.y);
    const pulsar_expert_ptrs &p = grp.p;
    const uint8_t *m0 = (const uint8_t *)(PAIR ? p.gate : p.down), *m1 = (const uint8_t *)(PAIR ? p.up : p.down);
    const bool nul = grp.is_null();  // block-uniform, as every exit below
    if (!nul && (!m0 || !m1)) return;
    uint32_t s0, s1;
    src.range_block(grp, lst, s0, s1);
    // with a bound the other kernel takes the shorter groups and the NULL one
    if (s0 >= s1 || s1 - s0 < min_pairs || (nul && min_pairs != 0u)) return;
    const uint32_t rb = blockIdx.x * kRows;
    if (nul) {  // unrouted slots: their rows of this block are 0
        for (uint32_t it = threadIdx.x; it < (s1 - s0) * kRows; it += 256u) {
            const uint32_t pr = src.pair(s0 + it / kRows, lst), row = rb + it % kRows;
            if (row < n_rows) out[((uint64_t)(pr >> 4) * n_used + (pr & 15u)) * n_rows + row] = 0.0f;
        }
        return;
    }
    PK_FMT_LUT(Q)
    const uint32_t lane = threadIdx.x & 63u, i = lane & 15u, q = lane >> 4, wave = threadIdx.x >> 6;
    const uint32_t row0 = rb + (PAIR ? 16u : 32u) * (wave % WR) + i, row1 = PAIR ? row0 : row0 + 16u;
    const uint8_t *w0 = as_global(m0) + (uint64_t)(row0 < n_rows ? row0 : n_rows - 1u) * row_bytes;
    const uint8_t *w1 = as_global(m1) + (uint64_t)(row1 < n_rows ? row1 : n_rows - 1u) * row_bytes;
    const float gb = PAIR && p.gate_b && row0 < n_rows ? ldwf(p.gate_b + row0) : 0.0f;
    const float ub = PAIR && p.up_b && row0 < n_rows ? ldwf(p.up_b + row0) : 0.0f;
    for (uint32_t t0 = s0; t0 < s1; t0 += T::kTok) {
        const uint32_t np = s1 - t0 < T::kTok ? s1 - t0 : T::kTok;
        if (t0 != s0) __syncthreads();  // the previous tile's pairs are stored
        if (threadIdx.x < np) pr_l[threadIdx.x] = src.pair(t0 + threadIdx.x, lst);
        __syncthreads();
        T tile;
        auto off = [&](uint32_t t) {
            const uint32_t pr = pr_l[t];
            return (uint64_t)(PAIR ? pr >> 4 : (pr >> 4) * n_used + (pr & 15u)) * (nb * 292u);
        };
        auto part = [&](auto nc) {
            constexpr uint32_t NC = decltype(nc)::value;
            tile.template run<NC>(buf0, buf1, lut, w0, w1, nb, np, (const uint8_t *)act, off);
#pragma unroll
            for (uint32_t n = 0; n < NC; n++)
#pragma unroll
                for (uint32_t r = 0; r < 4; r++) {
                    const uint32_t t = 16u * n + 4u * q + r;
                    if (!T::mine(n, r, wave / WR) || t >= np) continue;
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
        if (NS > 1u && np <= 16u)
            part(std::integral_constant<uint32_t, 1>{});
        else if (NS > 2u && np <= 32u)
            part(std::integral_constant<uint32_t, NS < 2u ? 1u : 2u>{});
        else if (NS > 4u && np <= 64u)
            part(std::integral_constant<uint32_t, NS < 4u ? 1u : 4u>{});
        else
            part(std::integral_constant<uint32_t, NS>{});
    }
}

// Pairs per group, in quarters, from which the tile beats the kernel it takes
// over from (0: no tile kernel): the 16-row kernel of mmq.hip wastes less on
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

template <uint32_t Q, bool PAIR, typename G>
static int launch_tile_grouped_q(float *out, const G &src, const float *weights, const pulsar_block_q8_K *act,
                                 uint32_t nb, uint32_t n_rows, uint32_t n_used, uint32_t n_group, uint64_t row_bytes,
                                 uint32_t act_op, uint32_t lst_bytes, uint32_t min_pairs) {
    // 64-pair tiles; 128 where a caller's CSR may hold long groups and the
    // format's registers allow it (Q2_K gate / up, 96 pairs: 685 -> 562 us,
    // 16 pairs 240 / 235; Q4_K spills: 279 -> 319)
    constexpr uint32_t NS = std::is_same<G, CsrGroups>::value && Q != PULSAR_QUANT_Q4_K && Q != PULSAR_QUANT_Q5_K ? 8 : 4;
    constexpr uint32_t kRows = PAIR ? 64u : 128u;
    hipLaunchKernelGGL((tile_grouped_kernel<Q, PAIR, 4, 1, NS, G>), dim3((n_rows + kRows - 1u) / kRows, n_group),
                       dim3(256), lst_bytes, pk::stream(), out, src, weights, act, nb, n_rows, n_used, row_bytes,
                       act_op, min_pairs);
    return launch_ok(PAIR ? "moe pair swiglu grouped (tile) launch" : "moe down grouped (tile) launch");
}

// The grouped stages on the tile, for the groups of at least min_pairs pairs.
template <typename G>
int launch_tile_grouped(bool pair, uint32_t quant, float *out, const G &src, const float *weights,
                        const pulsar_block_q8_K *act, uint32_t k_dim, uint32_t n_rows, uint32_t n_used,
                        uint32_t n_group, uint64_t row_bytes, uint32_t act_op, uint32_t lst_bytes,
                        uint32_t min_pairs) {
    const uint32_t nb = k_dim / 256u;
#define PK_TG(Q)                                                                                                     \
    case Q:                                                                                                          \
        return pair ? launch_tile_grouped_q<Q, true, G>(out, src, weights, act, nb, n_rows, n_used, n_group, row_bytes, \
                                                        act_op, lst_bytes, min_pairs)                                \
                    : launch_tile_grouped_q<Q, false, G>(out, src, weights, act, nb, n_rows, n_used, n_group,          \
                                                         row_bytes, act_op, lst_bytes, min_pairs);
    switch (quant) {
        PK_TG(PULSAR_QUANT_Q4_K)
        PK_TG(PULSAR_QUANT_Q5_K)
        PK_TG(PULSAR_QUANT_Q6_K)
        PK_TG(PULSAR_QUANT_Q2_K)
        PK_TG(PULSAR_QUANT_Q3_K)
        PK_TG(PULSAR_QUANT_IQ4_XS)
        PK_TG(PULSAR_QUANT_IQ2_XXS)
    default: return reject("grouped tile (quant)");
    }
#undef PK_TG
}
template int launch_tile_grouped<CsrGroups>(bool, uint32_t, float *, const CsrGroups &, const float *,
                                            const pulsar_block_q8_K *, uint32_t, uint32_t, uint32_t, uint32_t,
                                            uint64_t, uint32_t, uint32_t, uint32_t);
template int launch_tile_grouped<ExpertGroups>(bool, uint32_t, float *, const ExpertGroups &, const float *,
                                               const pulsar_block_q8_K *, uint32_t, uint32_t, uint32_t, uint32_t,
                                               uint64_t, uint32_t, uint32_t, uint32_t);

}  // namespace pk
