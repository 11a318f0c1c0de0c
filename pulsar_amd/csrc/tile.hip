// tile.hip - kernels on the wide matrix-core tile (pk_tile.h):
//   tile_gemm_kernel: pulsar_matmul_kq for prompt chunks. Against the kernels
//     it takes over from (mmq.hip's 16-row tiles, or four tokens per pass in
//     the lane kernels), weights from HBM: Q4_K 14336 x 4096, 512 tokens 183 ->
//     76 us (0.79 P int8-op/s), 1024 tokens 369 -> 153; IQ4_XS 8192 x 2816, 250
//     tokens 372 -> 27; Q2_K 14336 x 4096, 512 tokens 1137 -> 60. What bounds it
//     (counters, Q4_K, 512 tokens): vector units busy 42% of the time, matrix
//     cores 34%; its 256 registers leave two waves per SIMD, which overlap
//     these only in part: 30% of a wave's time waits for LDS and memory, 30%
//     for an issue slot.
#include "pk_tile.h"

namespace pk {

// Block = 32 WR weight rows x 16 NS tokens. Blocks go to the 8 XCDs round-
// robin, each with its own L2: XCD x takes the x-th eighth of the (row block,
// token tile) items, token tiles fastest, so a row block's weights are read
// by one XCD.
template <uint32_t Q, uint32_t WR, uint32_t WK, uint32_t NS>
__global__ __launch_bounds__(256, 2) void tile_gemm_kernel(float *__restrict__ out, const uint8_t *__restrict__ w,
                                                           const pulsar_block_q8_K *__restrict__ xq, uint32_t nb,
                                                           uint32_t out_dim, uint32_t n_tok, uint64_t row_bytes,
                                                           uint32_t n_tt, uint32_t n_item) {
    using T = Tile<Q, WR, WK, NS>;
    __shared__ __align__(16) uint8_t buf0[T::kBuf];
    __shared__ __align__(16) uint8_t buf1[T::kBuf];
    PK_FMT_LUT(Q)
    const uint32_t item = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (item >= n_item) return;  // block-uniform
    const uint32_t t0 = (item % n_tt) * T::kTok;
    const uint32_t lane = threadIdx.x & 63u, q = lane >> 4, wave = threadIdx.x >> 6;
    const uint32_t row = (item / n_tt * WR + wave % WR) * 32u + (lane & 15u);
    const uint32_t np = n_tok - t0 < T::kTok ? n_tok - t0 : T::kTok;
    auto wrow = [&](uint32_t r) { return w + (uint64_t)(r < out_dim ? r : out_dim - 1u) * row_bytes; };
    T tile;
    tile.run(buf0, buf1, lut, wrow(row), wrow(row + 16u), nb, np, (const uint8_t *)(xq + (uint64_t)t0 * nb),
             [&](uint32_t t) { return t * (nb * 292u); });
#pragma unroll
    for (uint32_t n = 0; n < NS; n++)
#pragma unroll
        for (uint32_t r = 0; r < 4; r++) {
            const uint32_t t = 16u * n + 4u * q + r;
            if (!T::mine(n, r, wave / WR) || t >= np) continue;
            float *o = out + (uint64_t)(t0 + t) * out_dim + row;
            if (row < out_dim) o[0] = tile.acc[n][0][r];
            if (row + 16u < out_dim) o[16] = tile.acc[n][1][r];
        }
}

template <uint32_t Q, uint32_t WR, uint32_t WK, uint32_t NS>
static uint64_t tile_items(uint32_t out_dim, uint32_t n_tok) {
    return (uint64_t)((n_tok + 16u * NS - 1u) / (16u * NS)) * ((out_dim + 32u * WR - 1u) / (32u * WR));
}

template <uint32_t Q>
static int launch_tile_gemm_q(float *out, const uint8_t *w, const pulsar_block_q8_K *xq, uint32_t nb,
                              uint32_t out_dim, uint32_t n_tok, uint64_t row_bytes) {
#define PK_TILE_FITS(WR, WK, NS) (tile_items<Q, WR, WK, NS>(out_dim, n_tok) <= kTileSlots)
#define PK_TILE(WR, WK, NS)                                                                                        \
    do {                                                                                                           \
        const uint64_t n_item = tile_items<Q, WR, WK, NS>(out_dim, n_tok);                                         \
        if (n_item > 0x7ffffff0ull) return -1;                                                                     \
        hipLaunchKernelGGL((tile_gemm_kernel<Q, WR, WK, NS>), dim3((uint32_t)((n_item + 7u) & ~7ull)), dim3(256), 0, \
                           pk::stream(), out, w, xq, nb, out_dim, n_tok, row_bytes,                                 \
                           (n_tok + 16u * NS - 1u) / (16u * NS), (uint32_t)n_item);                                 \
    } while (0)
    // The finest tile whose blocks are all in flight at once, else the widest:
    // a block's time falls with its rows and tokens (fewer steps with K split),
    // the work per product with them (a row is decoded once per token tile).
    // Q4_K 4096 x 4096, (1, 4, 2) / (2, 2, 4) / (4, 1, 4) / (4, 1, 8): 64 tokens
    // 11 / 22 / 32 / 52 us, 256 tokens 26 / 24 / 33 / 54, 512 tokens 49 / 34 /
    // 36 / 57; 14336 x 4096: 256 tokens 80 / 59 / 50 / 62, 512 tokens 180 / 105 /
    // 100 / 83, 1024 tokens 385 / 202 / 174 / 153
    if (PK_TILE_FITS(1, 4, 2))
        PK_TILE(1, 4, 2);
    else if (PK_TILE_FITS(2, 2, 4))
        PK_TILE(2, 2, 4);
    else if (PK_TILE_FITS(4, 1, 4))
        PK_TILE(4, 1, 4);
    else
        PK_TILE(4, 1, 8);
#undef PK_TILE
#undef PK_TILE_FITS
    return launch_ok("matmul_kq tile launch");
}

// -1: no tile kernel for the format or the shape
int launch_tile_gemm(uint32_t quant, float *out, const uint8_t *w, const pulsar_block_q8_K *xq, uint32_t in_dim,
                     uint32_t out_dim, uint32_t n_tok, uint64_t row_bytes) {
    const uint32_t nb = in_dim / 256u;
    if (nb > 65536u) return -1;  // a tile's activation offsets are 32 bits
    // the tile's copies to LDS move whole dwords of xq, the other kernels load
    // it at any alignment
    if ((uintptr_t)xq % 4u != 0u) return -1;
    // Where the other kernels are at least as fast (weights from HBM, both
    // sides timed on the same matrices: 13636 of 32 to 14336 rows, 256 to 14336
    // columns, 5 to 512 tokens; 3 in a thousand are more than 3% slower than
    // there, and the faster side is missed by 1% on average):
    // Q4_K, Q5_K, Q6_K have the 16-row kernel of mmq.hip, which takes chunks of
    // up to 16 tokens in one pass and, below 8192 rows, of up to 31 in two
    // cheap ones (Q4_K 4096 x 4096: 16 tokens 6.5 against 10.4 us, 33 tokens
    // 14.7 against 10.6; 14336 x 4096, 17 tokens: 25.5 against 15.1). Q6_K's
    // decode is the longest of them, and as long as the 32-row tile is all
    // that fills the chip the 16-row kernel stays ahead (3000 x 2048, 100
    // tokens: 14.2 against 15.3 us). So it does for the others where rows of
    // one or two super-blocks leave the tile's start and end its whole time
    // (Q5_K 8192 x 512, 64 tokens: 6.1 against 7.0 us), and for Q5_K up to
    // 64 tokens and the 768 blocks that its own kernel holds at once, where the
    // tile has a third of the chip (11008 x 8192, 64 tokens: 51.0 against 54.6).
    const uint64_t items = tile_items<PULSAR_QUANT_Q4_K, 1, 4, 2>(out_dim, n_tok);
    if (quant == PULSAR_QUANT_Q4_K || quant == PULSAR_QUANT_Q5_K || quant == PULSAR_QUANT_Q6_K) {
        if (n_tok < 17u || (n_tok < 32u && out_dim < 8192u)) return -1;
        if (n_tok >= 32u && items <= kTileSlots && (nb <= 2u || quant == PULSAR_QUANT_Q6_K)) return -1;
        if (n_tok >= 32u && n_tok <= 64u && quant == PULSAR_QUANT_Q5_K && items > kTileSlots && items <= 768u &&
            nb >= 16u)
            return -1;
    } else {
        // The other formats run four tokens per pass over the rows in the lane
        // kernels; both sides grow with the row length, so rows times passes
        // decide (IQ4_XS 4096 x 4096: two passes 11.6 against 12.4 us, three
        // 16 against 12.4; 2000 x 8192: four 19.3 against 20.8 us), and for
        // rows of up to three super-blocks, where the tile's start and end
        // outweigh its decode, rows times passes times length (IQ4_XS 1024 x
        // 256, 64 tokens: 3.9 against 5.0 us; 4096 x 512, 17: 5.8 against 4.8).
        const uint64_t rows4 = (uint64_t)((n_tok + 3u) / 4u) * out_dim;
        uint32_t least = 7000u, least_nb = 18000u;  // Q2_K
        switch (quant) {
        case PULSAR_QUANT_Q3_K: least_nb = 32000u; break;
        case PULSAR_QUANT_IQ4_XS: least = 9000u, least_nb = nb == 1u ? 45000u : 36000u; break;
        case PULSAR_QUANT_IQ2_XXS:
            // the lane kernels give a row a power of two of lanes: rows of
            // 24 super-blocks are on the tile earlier than rows of 32 (4096
            // rows, 8 tokens: 25.8 against 18.9 us, 5: 21.6 against 25.9)
            least = nb < 8u || (nb & (nb - 1u)) == 0u ? 8300u : 8000u, least_nb = nb == 1u ? 45000u : 36000u;
            break;
        default: break;
        }
        if (rows4 < least || (nb < 4u && rows4 * nb < least_nb)) return -1;
    }
#define PK_TG(Q) \
    case Q: return launch_tile_gemm_q<Q>(out, w, xq, nb, out_dim, n_tok, row_bytes);
    switch (quant) {
        PK_TG(PULSAR_QUANT_Q4_K)
        PK_TG(PULSAR_QUANT_Q5_K)
        PK_TG(PULSAR_QUANT_Q6_K)
        PK_TG(PULSAR_QUANT_Q2_K)
        PK_TG(PULSAR_QUANT_Q3_K)
        PK_TG(PULSAR_QUANT_IQ4_XS)
        PK_TG(PULSAR_QUANT_IQ2_XXS)
    default: return -1;
    }
#undef PK_TG
}

}  // namespace pk
