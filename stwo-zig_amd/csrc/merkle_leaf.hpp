// Message loads of the lifted Merkle leaves (device only): 16 column words per block, from the
// descriptor table of merkle_leaf_plan.
#pragma once
#include "blake2s.hpp"
#include "runtime.hpp"

namespace sr {

// boff: byte offset of the proof's columns in a batch (0 for one tree).
__device__ __forceinline__ void leaf_block_load(const LeafColDev* __restrict__ cd, uint32_t p, uint32_t m[16],
                                                uint64_t boff) {
#pragma unroll
    for (int w = 0; w < 16; w++) {
        const LeafColDev d = cd[w];
        m[w] = ((gcu32*)((const uint8_t*)d.col + boff))[((p >> d.shift) << 1) + (p & 1)] & d.mask;
    }
}

// The same for a segment whose columns all have the segment's size (lift(p) = p): every
// word is the column pointer (uniform) plus the lane's byte offset p * 4 (rows < 2^30), and
// the padding mask applies only to a padded last block (MASKED).
template <bool MASKED>
__device__ __forceinline__ void leaf_block_load_ident(const LeafColDev* __restrict__ cd, uint32_t voff,
                                                      uint32_t m[16], uint64_t boff) {
#pragma unroll
    for (int w = 0; w < 16; w++) {
        const LeafColDev d = cd[w];
        const uint32_t x = *(gcu32*)((const SR_GLOBAL uint8_t*)d.col + boff + voff);
        m[w] = MASKED ? (x & d.mask) : x;
    }
}

// h <- the state after blocks [blk0, blk_end) of the row at byte offset voff of every column
// (the leaf hash if blk_end is the last block), the blocks alternating between two buffers.
__device__ __forceinline__ void leaf_hash_ident(const LeafColDev* __restrict__ cols, uint32_t blk0, uint32_t blk_end,
                                                uint32_t n_cols, uint32_t voff, uint64_t boff, uint32_t h[8]) {
    const uint32_t nblocks_total = (n_cols + 15) >> 4;
    // blocks of 16 real columns, then at most one padded block (the last of the leaf)
    const uint32_t full_end = ((n_cols & 15) && blk_end == nblocks_total) ? blk_end - 1 : blk_end;
    uint32_t a[16], b[16];
    uint32_t blk = blk0;
    if (blk < full_end) leaf_block_load_ident<false>(cols + 16 * blk, voff, a, boff);
    for (; blk + 1 < full_end; blk += 2) {
        leaf_block_load_ident<false>(cols + 16 * (blk + 1), voff, b, boff);
        b2_compress(h, a, 64 + 64 * (blk + 1), blk + 1 == nblocks_total);
        if (blk + 2 < full_end) leaf_block_load_ident<false>(cols + 16 * (blk + 2), voff, a, boff);
        b2_compress(h, b, 64 + 64 * (blk + 2), blk + 2 == nblocks_total);
    }
    if (blk < full_end) {
        b2_compress(h, a, 64 + 64 * (blk + 1), blk + 1 == nblocks_total);
        blk++;
    }
    if (blk < blk_end) {
        leaf_block_load_ident<true>(cols + 16 * blk, voff, a, boff);
        b2_compress(h, a, 64 + 4 * n_cols, true);
    }
}

}  // namespace sr
