// FRI folds on gfx950 (src/core/fri/folding.zig:316-380,558-602).
//
// fold_line:   dst[i] = (f0 + f1) + alpha * (f0 - f1) * x_i^-1, (f0, f1) = src[2i], src[2i+1],
//              x_i = LineDomain(halfOdds(log)).at(bitrev(i)).x.  x_i^-1 is read from the
//              inverse twiddle tower: its layer for halfOdds(log) holds exactly these values.
// fold_circle: dst[i] = dst[i] * alpha^2 + (f0 + f1) + alpha * (f0 - f1) * y_i^-1 with
//              y_i = halfOdds(log-1).at(bitrev(i)).y (resident table per log size).
// Both optionally hash the folded value as the next layer's Merkle leaf
// (prefix || 4 LE words, one compression), fusing fold and leaf hashing.
//
// tree_layer: one FRI layer commitment per launch (prover/fri.zig:377-621): the fold into
// the layer's line, its leaf hashes, every parent level (layers.zig:99-140) and the channel
// step on the root; the top levels are reduced by the last workgroup to finish, so the next
// layer's launch finds its alpha in the device channel.  The same kernel reduces the top
// levels of any tree from hashes already in HBM.
// fri_tail: the layers below FRI_TAIL_MAX_LOG + 1 in one workgroup with the line and the
// hash level resident in LDS.
#include <type_traits>

#include "chan.hpp"
#include "merkle_leaf.hpp"

namespace sr {

__device__ __forceinline__ void leaf_qm31(uint8_t* __restrict__ leaves, uint64_t i, const B2State& seed, qm31 v) {
    uint32_t m[16] = {v.c0.a, v.c0.b, v.c1.a, v.c1.b, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    uint32_t h[8];
#pragma unroll
    for (int k = 0; k < 8; k++) h[k] = seed.h[k];
    b2_compress(h, m, 80, true);
    uint4* o = (uint4*)(leaves + i * 32);
    o[0] = make_uint4(h[0], h[1], h[2], h[3]);
    o[1] = make_uint4(h[4], h[5], h[6], h[7]);
}

__global__ __launch_bounds__(256) void fold_line_kernel(const uint4* __restrict__ src, uint32_t log_src,
                                                        const uint32_t* __restrict__ inv_x, qm31 alpha,
                                                        const DevChannel* __restrict__ dch,
                                                        uint4* __restrict__ dst, uint8_t* __restrict__ leaves,
                                                        B2State seed) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (1u << (log_src - 1))) return;
    if (dch) alpha = qload(dch->alpha);
    uint4 a = src[2 * i], b = src[2 * i + 1];
    qm31 f0 = {{a.x, a.y}, {a.z, a.w}}, f1 = {{b.x, b.y}, {b.z, b.w}};
    qm31 r = qadd(qadd(f0, f1), qmul(qmulm(qsub(f0, f1), inv_x[i]), alpha));
    dst[i] = make_uint4(r.c0.a, r.c0.b, r.c1.a, r.c1.b);
    if (leaves) leaf_qm31(leaves, i, seed, r);
}

__global__ __launch_bounds__(256) void fold_circle_kernel(const uint32_t* __restrict__ c0,
                                                          const uint32_t* __restrict__ c1,
                                                          const uint32_t* __restrict__ c2,
                                                          const uint32_t* __restrict__ c3, uint32_t log_src,
                                                          const uint32_t* __restrict__ inv_y, qm31 alpha, qm31 alpha2,
                                                          const DevChannel* __restrict__ dch, bool accumulate,
                                                          uint4* __restrict__ dst, uint8_t* __restrict__ leaves,
                                                          B2State seed, uint64_t bstride) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (1u << (log_src - 1))) return;
    if (blockIdx.y) {  // proof blockIdx.y of a batch: its buffers bstride bytes further on
        const uint64_t boff = (uint64_t)blockIdx.y * bstride;
        c0 = (const uint32_t*)((const uint8_t*)c0 + boff);
        c1 = (const uint32_t*)((const uint8_t*)c1 + boff);
        c2 = (const uint32_t*)((const uint8_t*)c2 + boff);
        c3 = (const uint32_t*)((const uint8_t*)c3 + boff);
        if (dch) dch = (const DevChannel*)((const uint8_t*)dch + boff);
        dst = (uint4*)((uint8_t*)dst + boff);
        if (leaves) leaves += boff;
    }
    if (dch) {
        alpha = qload(dch->alpha);
        alpha2 = qload(dch->alpha2);
    }
    uint2 w0 = ((const uint2*)c0)[i], w1 = ((const uint2*)c1)[i], w2 = ((const uint2*)c2)[i],
          w3 = ((const uint2*)c3)[i];
    qm31 f0 = {{w0.x, w1.x}, {w2.x, w3.x}}, f1 = {{w0.y, w1.y}, {w2.y, w3.y}};
    qm31 r = qadd(qadd(f0, f1), qmul(qmulm(qsub(f0, f1), inv_y[i]), alpha));
    if (accumulate) {
        uint4 d = dst[i];
        r = qadd(qmul(qm31{{d.x, d.y}, {d.z, d.w}}, alpha2), r);
    }
    dst[i] = make_uint4(r.c0.a, r.c0.b, r.c1.a, r.c1.b);
    if (leaves) leaf_qm31(leaves, i, seed, r);
}

// ---------------------------------------------------------------------------
// Tree levels inside one workgroup.  A level of c <= 128 parents uses one quad of lanes per
// compression (blake2s_quad.hpp); wider levels use one lane per compression, which does the
// same work in fewer instructions once the SIMDs are full.  A quad level's hashes go to the
// next level through a board in LDS (words in lane order).  From 16 parents on the quads of
// wave 0 are enough, and LDS serves its accesses in order: no barrier until the root.
// Shared by the layer and tail kernels.

constexpr uint32_t TL_THREADS = 256;    // tree-layer workgroup: one wave per SIMD
constexpr uint32_t TAIL_THREADS = 512;   // tail workgroup: two waves per SIMD keep it issuing on the wide layers
constexpr uint32_t TR_QUAD_MAX = 128;    // widest level hashed by quads
constexpr uint32_t TR_WAVE_MAX = 16;     // widest level hashed by the quads of one wave
constexpr uint32_t TR_BOARD = 64;        // messages of the widest level that reads the board

// LDS of the levels: plain hashes (8 words each) of the one-lane levels, hA then hB, or the
// board of the quad levels over the same words (a level's inputs are all read before its board
// is written); the channel's boards lie before them.
constexpr uint32_t TR_PLAIN_A = 1024 * 8, TR_PLAIN_B = 512 * 8;
constexpr uint32_t TR_LEVEL_WORDS = TR_PLAIN_A + TR_PLAIN_B;
static_assert(TR_LEVEL_WORDS >= 160 * TR_BOARD, "plain hashes and the board share their words");
constexpr uint32_t TR_CHAN_WORDS = 2 * 160;

__device__ __forceinline__ void tr_load16(const uint32_t* in, uint32_t m[16]) {
    const uint4* m4 = (const uint4*)in;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint4 v = m4[i];
        m[4 * i] = v.x, m[4 * i + 1] = v.y, m[4 * i + 2] = v.z, m[4 * i + 3] = v.w;
    }
}

// Words q and 4 + q of a hash; `off` = 32 * its index + 4 q.
__device__ __forceinline__ void tr_store_quad(uint8_t* __restrict__ g, uint32_t off, uint32_t hlo, uint32_t hhi) {
    *(uint32_t*)(g + off) = hlo;
    *(uint32_t*)(g + off + 16) = hhi;
}

__device__ __forceinline__ void tr_put_lane(uint32_t* lds, uint8_t* __restrict__ g, const uint32_t h[8]) {
    const uint4 x = make_uint4(h[0], h[1], h[2], h[3]), y = make_uint4(h[4], h[5], h[6], h[7]);
    *(uint4*)lds = x;
    *(uint4*)(lds + 4) = y;
    uint4* o = (uint4*)g;
    o[0] = x;
    o[1] = y;
}

// Per-lane constants of the quad levels.
struct TrQuad {
    uint32_t t, q;
    QuadLane L;
    QuadIo io;
    uint32_t nlo, nhi;  // node seed words q, 4 + q
    __device__ __forceinline__ TrQuad(uint32_t t_, const B2State& node_seed)
        : t(t_), q(t_ & 3), L(t_ & 3), io(t_ >> 2, t_ & 3) {
        nlo = L.sel(node_seed.h[0], node_seed.h[1], node_seed.h[2], node_seed.h[3]);
        nhi = L.sel(node_seed.h[4], node_seed.h[5], node_seed.h[6], node_seed.h[7]);
    }
};

// The levels of c, c/2, ..., 1 parents by quads; the 2c children are on the board, written by
// quads 0 .. 2c - 1.  Level `lev` has c parents of this workgroup, from parent blk * c on.  The
// root ends as (rlo, rhi) = words (q, 4 + q) in every quad of the first wave; the other waves
// leave once the first is alone with the rest.  There its quads all compress, also those beyond
// the level (on words that nothing valid comes from: quad i writes slot i / 2, and only slots
// below the next level's count are read for a result): what a level costs is one wave's
// instructions, and masks and branches are among them.
__device__ __forceinline__ void tr_quad_levels(const TrQuad& Q, uint32_t* board, uint32_t c, uint8_t* tree,
                                               uint32_t lev, uint32_t blk, uint32_t& rlo, uint32_t& rhi) {
    const uint32_t p = Q.t >> 2, wave = __builtin_amdgcn_readfirstlane(Q.t >> 6);
    const uint32_t node = 32 * p + 4 * Q.q;
    uint32_t at = (1u << lev) - 1 + blk * c;  // this workgroup's first parent among the tree's hashes
    for (; 2 * c > TR_WAVE_MAX; c >>= 1, at >>= 1) {
        __syncthreads();
        rlo = Q.nlo;
        rhi = Q.nhi;
        if (TR_WAVE_MAX * wave < c)
            qboard_compress<TR_BOARD>(Q.L, rlo, rhi, board, Q.io.rd, 128, true);
        if (c > TR_WAVE_MAX) __syncthreads();  // every message is read
        if (TR_WAVE_MAX * wave < c) {
            qboard_put<TR_BOARD>(board, Q.io, rlo, rhi);
            tr_store_quad(tree, 32 * at + node, rlo, rhi);
        }
    }
    if (wave) return;
    uint32_t rd = c == 1 ? 16 * Q.q : Q.io.rd;
    uint4 m[10];
    qboard_wave_fence();
#pragma unroll
    for (int r = 0; r < 10; r++) m[r] = qboard_get_round<TR_BOARD>(board, rd, r);
    for (;; at >>= 1) {
        rlo = Q.nlo;
        rhi = Q.nhi;
        b2q_compress(Q.L, rlo, rhi, [&](int r) { return m[r]; }, 128, true);
        if (p < c) tr_store_quad(tree, 32 * at + node, rlo, rhi);
        if (c == 1) return;
        c >>= 1;
        rd = c == 1 ? 16 * Q.q : rd;
#pragma unroll
        for (int r = 0; r < 10; r++) {
            qboard_put_round<TR_BOARD>(board, Q.io, r, rlo, rhi);
            qboard_wave_fence();
            m[r] = qboard_get_round<TR_BOARD>(board, rd, r);
        }
    }
}

// From 2c hashes, plain in hA (their writes are behind a barrier) or, if `on_board`, on the board:
// the one-lane levels between hA and hB, a first quad level that selects its message words, then
// the levels on the board, which may overlap that level's inputs.
template <uint32_t T>
__device__ __forceinline__ void tr_levels(const TrQuad& Q, uint32_t* lds, bool on_board, uint32_t c, uint8_t* tree,
                                          uint32_t lev, uint32_t blk, const B2State& seed, uint32_t& rlo,
                                          uint32_t& rhi) {
    if (!on_board) {
        uint32_t *in = lds, *out = lds + TR_PLAIN_A;
        for (; c > TR_QUAD_MAX; c >>= 1, lev--) {
            uint8_t* g = tree + 32ull * ((1u << lev) - 1 + blk * c);
            for (uint32_t p = Q.t; p < c; p += T) {
                uint32_t m[16], h[8];
                tr_load16(in + 16 * p, m);
#pragma unroll
                for (int k = 0; k < 8; k++) h[k] = seed.h[k];
                b2_compress(h, m, 128, true);
                tr_put_lane(out + 8 * p, g + 32 * p, h);
            }
            __syncthreads();
            uint32_t* x = in;
            in = out;
            out = x;
        }
        constexpr uint32_t STEP = T / 4, IT = (TR_QUAD_MAX + STEP - 1) / STEP;
        uint32_t lo[IT], hi[IT];
        uint8_t* g = tree + 32ull * ((1u << lev) - 1 + blk * c);
        // one copy of the compression's code
#pragma unroll 1
        for (uint32_t k = 0; k < IT; k++) {
            const uint32_t p = (Q.t >> 2) + k * STEP;
            uint32_t hlo = Q.nlo, hhi = Q.nhi;
            if (p < c || (c == 1 && Q.t < 64 && k == 0)) {
                uint32_t m[16];
                tr_load16(in + (c == 1 ? 0 : 16 * p), m);
                b2_compress_quad(Q.L, hlo, hhi, m, 128, true);
                if (p < c) tr_store_quad(g, 32 * p + 4 * Q.q, hlo, hhi);
            }
#pragma unroll
            for (uint32_t i = 0; i < IT; i++) {
                lo[i] = i == k ? hlo : lo[i];
                hi[i] = i == k ? hhi : hi[i];
            }
        }
        rlo = lo[0];
        rhi = hi[0];
        if (c == 1) return;
        __syncthreads();
#pragma unroll
        for (uint32_t k = 0; k < IT; k++)
            if ((Q.t >> 2) + k * STEP < c) qboard_put<TR_BOARD>(lds, Q.io, lo[k], hi[k], k * STEP / 2);
        c >>= 1;
        lev--;
    }
    tr_quad_levels(Q, lds, c, tree, lev, blk, rlo, rhi);
}

// Leaf hash of one QM31 value (leaf_qm31 above) by a quad, the value in every lane.
__device__ __forceinline__ void tr_leaf_quad(const QuadLane& L, const B2State& seed, qm31 v, uint32_t& hlo,
                                             uint32_t& hhi) {
    const uint32_t m[16] = {v.c0.a, v.c0.b, v.c1.a, v.c1.b, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    hlo = L.sel(seed.h[0], seed.h[1], seed.h[2], seed.h[3]);
    hhi = L.sel(seed.h[4], seed.h[5], seed.h[6], seed.h[7]);
    b2_compress_quad(L, hlo, hhi, m, 80, true);
}

__device__ __forceinline__ void tr_leaf_lane(const B2State& seed, qm31 v, uint32_t h[8]) {
    const uint32_t m[16] = {v.c0.a, v.c0.b, v.c1.a, v.c1.b, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < 8; k++) h[k] = seed.h[k];
    b2_compress(h, m, 80, true);
}

__device__ __forceinline__ qm31 tr_fold(uint4 a, uint4 b, qm31 alpha, uint32_t inv) {
    const qm31 f0 = {{a.x, a.y}, {a.z, a.w}}, f1 = {{b.x, b.y}, {b.z, b.w}};
    return qadd(qadd(f0, f1), qmul(qmulm(qsub(f0, f1), inv), alpha));
}

// Fold input i of a layer kernel: line (fold_line_kernel) or circle (fold_circle_kernel,
// no accumulation) source.
template <int SRC>
__device__ __forceinline__ qm31 tr_fold_at(const FriLayerArgs& a, uint64_t i, qm31 alpha) {
    if constexpr (SRC == FRI_SRC_LINE) {
        return tr_fold(a.src_line[2 * i], a.src_line[2 * i + 1], alpha, a.inv[i]);
    } else {
        const uint2 w0 = ((const uint2*)a.coord[0])[i], w1 = ((const uint2*)a.coord[1])[i],
                    w2 = ((const uint2*)a.coord[2])[i], w3 = ((const uint2*)a.coord[3])[i];
        return tr_fold(make_uint4(w0.x, w1.x, w2.x, w3.x), make_uint4(w0.y, w1.y, w2.y, w3.y), alpha, a.inv[i]);
    }
}

// The channel beside the levels: the digest as words (q, 4 + q) in every quad of the first wave,
// the draws since the last mix, the last drawn element; in LDS two one-slot boards, the message of
// mixRoot (digest || root) and that of drawSecureFelt (digest || draw counter || zeros).
struct TrChan {
    uint32_t dlo, dhi, n_draws;
    qm31 alpha;
};

// All threads; the caller's barrier ends it.
template <uint32_t T>
__device__ __forceinline__ TrChan tr_chan_init(const TrQuad& Q, uint32_t* chan, const DevChannel* ch) {
    if (Q.t >= 64) {
        for (uint32_t i = Q.t - 64; i < 160; i += T - 64) chan[160 + i] = 0;
    }
    return TrChan{ch->digest[Q.q], ch->digest[4 + Q.q], 0, qzero()};
}

// Channel step on a root held by every quad of the first wave, which runs it, as (rlo, rhi)
// (MerkleChannel.mixRoot then drawSecureFelt, as chan_mix_root_draw_thread).
__device__ __forceinline__ void tr_chan_step(const TrQuad& Q, uint32_t* chan, uint32_t rlo, uint32_t rhi, TrChan& C,
                                             DevChannel* __restrict__ ch) {
    const QuadLane& L = Q.L;
    const uint32_t ilo = L.sel(SR_B2_IV0 ^ 0x01010020u, SR_B2_IV1, SR_B2_IV2, SR_B2_IV3);
    const uint32_t ihi = L.sel(SR_B2_IV4, SR_B2_IV5, SR_B2_IV6, SR_B2_IV7);
    uint32_t *const mix = chan, *const draw = chan + 160;
    // quad 0 writes the first half of a message, quad 1 the second
    if (Q.t < 8) qboard_put<1>(mix, Q.io, Q.t < 4 ? C.dlo : rlo, Q.t < 4 ? C.dhi : rhi);
    // compression 0 is the mix, the others are draws (more than one with probability ~2^-28)
#pragma unroll 1
    for (uint32_t k = 0; k <= 64; k++) {
        qboard_wave_fence();
        uint32_t hlo = ilo, hhi = ihi;
        qboard_compress<1>(L, hlo, hhi, k ? draw : mix, 16 * Q.q, k ? 37 : 64, true);
        if (k == 0) {
            C.dlo = hlo;
            C.dhi = hhi;
            if (Q.t < 4) qboard_put<1>(draw, Q.io, hlo, hhi);
            continue;
        }
        uint32_t bad = (hlo >= 2u * P || hhi >= 2u * P) ? 1u : 0u;
        bad |= quad_perm<QP_ROT1>(bad);
        bad |= quad_perm<QP_ROT2>(bad);  // OR over the quad (the same in all)
        bad = __builtin_amdgcn_readfirstlane(bad);
        if (bad || k > 1) {
            // message word 8, the draw counter (the first word of the second half): the next one,
            // or zero again for the next step
            if (Q.t == 4) {
#pragma unroll
                for (int r = 0; r < 10; r++) *(uint32_t*)((uint8_t*)draw + 64 * r + Q.io.wr[2 * r]) = bad ? k : 0u;
            }
            if (bad) continue;
        }
        C.n_draws = k;
        C.alpha = {{mred64(quad_bcast<0>(hlo)), mred64(quad_bcast<1>(hlo))},
                   {mred64(quad_bcast<2>(hlo)), mred64(quad_bcast<3>(hlo))}};
        return;
    }
    if (Q.t == 0) ch->status = 1;
}

// The state of the first wave's channel to the DevChannel.
__device__ __forceinline__ void tr_chan_store(const TrQuad& Q, const TrChan& C, DevChannel* __restrict__ ch) {
    if (Q.t >= 4) return;
    ch->digest[Q.q] = C.dlo;
    ch->digest[4 + Q.q] = C.dhi;
    if (Q.q == 0) {
        ch->n_draws = C.n_draws;
        qstore(C.alpha, ch->alpha);
        qstore(qsqr(C.alpha), ch->alpha2);
    }
}

// One tree (or its top levels) in one launch.  Workgroup b owns the 2^s hashes
// [b 2^s, (b+1) 2^s) of level k0: it produces them (SRC = FRI_SRC_LINE / FRI_SRC_CIRCLE:
// fold the previous layer with the alpha in `ch`, store the folded value and hash it as a
// leaf; FRI_SRC_COLUMNS: hash the rows of a tree's columns) or loads them (FRI_SRC_HASHES), then reduces them to its subtree root at level
// k0 - s.  The last workgroup to finish (split completion counters; the subtree roots are
// exchanged through device-coherent stores and loads, so no workgroup writes back its L2)
// reduces the 2^(k0-s) subtree roots to the root and, with `ch`, runs the channel step on
// it.  The counters are left at zero.
template <int SRC>
__global__ __launch_bounds__(TL_THREADS) void tree_layer_kernel(FriLayerArgs a0) {
    FriLayerArgs a = a0;
    if (blockIdx.y) {
        // tree blockIdx.y of a batch: its line, tree, channel and root copy bstride bytes further
        // on, its counters and root exchange TREE_CNT_WORDS words further on
        const uint64_t boff = (uint64_t)blockIdx.y * a.bstride;
        if (a.src_line) a.src_line = (const uint4*)((const uint8_t*)a.src_line + boff);
        for (int k = 0; k < 4; k++)
            if (a.coord[k]) a.coord[k] = (const uint32_t*)((const uint8_t*)a.coord[k] + boff);
        if (a.dst_line) a.dst_line = (uint4*)((uint8_t*)a.dst_line + boff);
        a.tree += boff;
        if (a.ch) a.ch = (DevChannel*)((uint8_t*)a.ch + boff);
        if (a.root_out) a.root_out = (uint32_t*)((uint8_t*)a.root_out + boff);
        a.cnt += (uint64_t)blockIdx.y * TREE_CNT_WORDS;
        a.xr += (uint64_t)blockIdx.y * TREE_CNT_WORDS;
    }
    __shared__ __align__(16) uint32_t sh[TR_CHAN_WORDS + TR_LEVEL_WORDS];
    __shared__ uint32_t last;
    uint32_t *const chan = sh, *const lds = sh + TR_CHAN_WORDS;
    const uint32_t t = threadIdx.x, q = t & 3;
    const TrQuad Q(t, a.node_seed);
    const uint32_t n1 = 1u << a.s;
    const uint64_t base = (uint64_t)blockIdx.x * n1;
    uint8_t* lev_k0 = a.tree + (((uint64_t)1 << a.k0) - 1) * 32;
    uint32_t rlo = 0, rhi = 0;
    bool boards = false;  // the hashes of level k0 are on the board
    if constexpr (SRC == FRI_SRC_HASHES) {
        for (uint32_t p = t; p < n1; p += TL_THREADS) {
            const uint4* s4 = (const uint4*)(lev_k0 + (base + p) * 32);
            const uint4 x = s4[0], y = s4[1];
            *(uint4*)&lds[8 * p] = x;
            *(uint4*)&lds[8 * p + 4] = y;
        }
    } else if constexpr (SRC == FRI_SRC_COLUMNS) {
        const uint64_t boff = (uint64_t)blockIdx.y * a.bstride;
        const uint32_t nblk = (a.n_cols + 15) >> 4;
        boards = n1 <= TR_QUAD_MAX;
        if (boards) {
#pragma unroll 1
            for (uint32_t k = 0; k < TR_QUAD_MAX / (TL_THREADS / 4); k++) {
                const uint32_t p = (t >> 2) + k * (TL_THREADS / 4);
                if (p >= n1) break;
                const uint32_t voff = (uint32_t)(base + p) << 2;
                uint32_t hlo = Q.L.sel(a.leaf_seed.h[0], a.leaf_seed.h[1], a.leaf_seed.h[2], a.leaf_seed.h[3]);
                uint32_t hhi = Q.L.sel(a.leaf_seed.h[4], a.leaf_seed.h[5], a.leaf_seed.h[6], a.leaf_seed.h[7]);
                uint32_t m[16], nx[16];
                leaf_block_load_ident<true>(a.cols, voff, m, boff);
#pragma unroll 1
                for (uint32_t b = 0; b < nblk; b++) {
                    const bool lst = b + 1 == nblk;
                    if (!lst) leaf_block_load_ident<true>(a.cols + 16 * (b + 1), voff, nx, boff);
                    b2_compress_quad(Q.L, hlo, hhi, m, 64 + (lst ? 4 * a.n_cols : 64 * (b + 1)), lst);
#pragma unroll
                    for (int w = 0; w < 16; w++) m[w] = nx[w];
                }
                qboard_put<TR_BOARD>(lds, Q.io, hlo, hhi, k * (TL_THREADS / 8));
                tr_store_quad(lev_k0 + base * 32, 32 * p + 4 * q, hlo, hhi);
            }
        } else {
            for (uint32_t p = t; p < n1; p += TL_THREADS) {
                uint32_t h[8];
#pragma unroll
                for (int k = 0; k < 8; k++) h[k] = a.leaf_seed.h[k];
                leaf_hash_ident(a.cols, 0, nblk, a.n_cols, (uint32_t)(base + p) << 2, boff, h);
                tr_put_lane(lds + 8 * p, lev_k0 + (base + p) * 32, h);
            }
        }
    } else {
        const qm31 alpha = qload(a.ch->alpha);
        boards = n1 <= TR_QUAD_MAX;
        if (boards) {
#pragma unroll
            for (uint32_t k = 0; k < TR_QUAD_MAX / (TL_THREADS / 4); k++) {
                const uint32_t p = (t >> 2) + k * (TL_THREADS / 4);
                if (p < n1) {
                    const qm31 r = tr_fold_at<SRC>(a, base + p, alpha);
                    if (q == 0) a.dst_line[base + p] = make_uint4(r.c0.a, r.c0.b, r.c1.a, r.c1.b);
                    uint32_t hlo, hhi;
                    tr_leaf_quad(Q.L, a.leaf_seed, r, hlo, hhi);
                    qboard_put<TR_BOARD>(lds, Q.io, hlo, hhi, k * (TL_THREADS / 8));
                    tr_store_quad(lev_k0 + base * 32, 32 * p + 4 * q, hlo, hhi);
                }
            }
        } else {
            for (uint32_t p = t; p < n1; p += TL_THREADS) {
                const qm31 r = tr_fold_at<SRC>(a, base + p, alpha);
                a.dst_line[base + p] = make_uint4(r.c0.a, r.c0.b, r.c1.a, r.c1.b);
                uint32_t h[8];
                tr_leaf_lane(a.leaf_seed, r, h);
                tr_put_lane(lds + 8 * p, lev_k0 + (base + p) * 32, h);
            }
        }
    }
    const uint32_t nb = gridDim.x;
    // nothing of the top pass is kept for the first one: the channel's boards are written by the
    // workgroup that reaches the root
    uint32_t c = n1 >> 1, lev = a.k0 - 1;
    uint32_t blk = blockIdx.x;
    TrChan C{};
    for (bool top = nb == 1;; top = true) {
        if (top && a.ch) C = tr_chan_init<TL_THREADS>(Q, chan, a.ch);
        if (!boards || top) __syncthreads();
        tr_levels<TL_THREADS>(Q, lds, boards, c, a.tree, lev, blk, a.node_seed, rlo, rhi);
        if (top) break;
        // Hand-off without an L2 writeback: quad 0 publishes the subtree root with
        // device-coherent stores (agent-scope atomic stores, global_store sc1), the wave waits
        // until they are acknowledged, and thread 0 counts the workgroup; the last workgroup
        // reads the roots with device-coherent loads.  The tree's own copy of the roots (plain
        // stores) is read by later launches only.
        if (t < 4) {
            __hip_atomic_store(&a.xr[8 * blockIdx.x + q], rlo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&a.xr[8 * blockIdx.x + 4 + q], rhi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (t < 64) {
            __builtin_amdgcn_s_waitcnt(0);
            if (t == 0) {
                const uint32_t b = blockIdx.x, g = b % TREE_CNT_GROUPS, ng = nb < TREE_CNT_GROUPS ? nb : TREE_CNT_GROUPS;
                const uint32_t gsize = (nb - g + TREE_CNT_GROUPS - 1) / TREE_CNT_GROUPS;
                uint32_t lst = 0;
                if (atomicAdd(&a.cnt[TREE_CNT_STRIDE * g], 1u) == gsize - 1)
                    lst = atomicAdd(&a.cnt[TREE_CNT_STRIDE * TREE_CNT_GROUPS], 1u) == ng - 1 ? 1u : 0u;
                last = lst;
            }
        }
        __syncthreads();
        if (!last) return;
        // Acquire: the loads of the other workgroups' roots below are ordered after the counter
        // update that observed their arrival (each publisher's roots were acknowledged, s_waitcnt,
        // before its count).  One fence per launch, in the last workgroup only.
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        if (t <= TREE_CNT_GROUPS) atomicExch(&a.cnt[TREE_CNT_STRIDE * t], 0u);
        // top levels from the nb subtree roots
        for (uint32_t i = t; i < 8 * nb; i += TL_THREADS)
            lds[i] = __hip_atomic_load(&a.xr[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        boards = false;
        c = nb >> 1;
        lev = a.k0 - a.s - 1;
        blk = 0;
    }
    if (t >= 64) return;
    if (t < 4 && a.root_out) tr_store_quad((uint8_t*)a.root_out, 4 * q, rlo, rhi);
    if (a.ch) {
        tr_chan_step(Q, chan, rlo, rhi, C, a.ch);
        tr_chan_store(Q, C, a.ch);
    }
}

// fri_tail: the inner layers below the committed line top_log (<= FRI_TAIL_MAX_LOG + 1) run
// in one workgroup with the current line and hash level resident in LDS and the channel
// messages on LDS boards: per layer the fold into the next line, its leaf hashes,
// the parent levels (layers.zig:99-140) and the channel step on the root, separated by
// workgroup barriers instead of kernel boundaries (prover/fri.zig:377-621 runs the same
// sequence per layer).  The last fold (into last_log) stores the line only.  Layers of at most
// 16 values run in the first wave alone, without a barrier.
__global__ __launch_bounds__(TAIL_THREADS) void fri_tail_kernel(const FriTailArgs a) {
    // The per-log pointer arrays are read from the kernel arguments with the (uniform) log as
    // index and proof blockIdx.x's offset added at each use: a local copy of the arguments
    // indexed by a runtime log would live in scratch memory, and every scratch load's wait
    // would also wait for the tree stores of the previous level.
    const uint64_t boff = (uint64_t)blockIdx.x * a.bstride;
    const auto at = [boff](auto* p) { return (decltype(p))((uint8_t*)p + boff); };
    DevChannel* __restrict__ ch = at(a.ch);
    const B2State leaf_seed = a.leaf_seed, node_seed = a.node_seed;
    constexpr uint32_t NV = 1u << FRI_TAIL_MAX_LOG, PER = NV / TAIL_THREADS;
    static_assert(TAIL_THREADS / 4 >= TR_QUAD_MAX, "a quad per value of a narrow layer");
    __shared__ __align__(16) uint32_t sh[TR_CHAN_WORDS + TR_LEVEL_WORDS + 4 * NV + 4];
    uint32_t *const chan = sh, *const lds = sh + TR_CHAN_WORDS;
    uint4* const vs = (uint4*)(lds + TR_LEVEL_WORDS);  // current line
    uint32_t* const sa = (uint32_t*)(vs + NV);         // alpha
    const uint32_t t = threadIdx.x, q = t & 3;
    const TrQuad Q(t, node_seed);
    uint32_t l = a.top_log;
    TrChan C = tr_chan_init<TAIL_THREADS>(Q, chan, ch);
    C.alpha = qload(ch->alpha);
    // This thread's value k of a layer of n values: its quad's on narrow layers, else its lane's.
    // The next layer's pointers and inverse x are loaded while this one's tree is hashed.
    uint32_t inv[PER];
    uint4* line;
    uint8_t* tree;
    uint32_t* root;
    const auto value = [&](uint32_t n, uint32_t k) {
        return n <= TR_QUAD_MAX ? (k ? n : t >> 2) : t + k * TAIL_THREADS;
    };
    const auto load_layer = [&](uint32_t log) {
        const uint32_t n = 1u << log;
        const uint32_t* inv_x = a.itw_half - 2 * (size_t)n;
#pragma unroll
        for (uint32_t k = 0; k < PER; k++) inv[k] = value(n, k) < n ? inv_x[value(n, k)] : 0u;
        line = at(a.lines[log]);
        tree = at(a.trees[log]);
        root = a.roots[log] ? at(a.roots[log]) : nullptr;
        asm volatile("" : "+s"(line), "+s"(tree), "+s"(root));  // here, not where they are used
    };
    load_layer(l - 1);
    __syncthreads();
    const uint4* __restrict__ src = at(a.lines[l]);
    bool first = true;
    for (;;) {
        l--;
        const uint32_t n = 1u << l;
        const bool quads = n <= TR_QUAD_MAX;
        qm31 r[PER];
#pragma unroll
        for (uint32_t k = 0; k < PER; k++) {
            const uint32_t p = value(n, k);
            if (p < n) {
                const uint4 x = first ? src[2 * p] : vs[2 * p];
                const uint4 y = first ? src[2 * p + 1] : vs[2 * p + 1];
                r[k] = tr_fold(x, y, C.alpha, inv[k]);
            }
        }
        first = false;
        if (n <= TR_WAVE_MAX) qboard_wave_fence();
        else __syncthreads();
#pragma unroll
        for (uint32_t k = 0; k < PER; k++) {
            const uint32_t p = value(n, k);
            if (p < n && (!quads || q == 0)) {
                const uint4 rv = make_uint4(r[k].c0.a, r[k].c0.b, r[k].c1.a, r[k].c1.b);
                vs[p] = rv;
                line[p] = rv;
            }
        }
        if (l == a.last_log) break;
        const uint64_t leaves = 32ull * (n - 1);
        uint8_t* const tr = tree;
        uint32_t* const ro = root;
        load_layer(l - 1);
        uint32_t rlo = 0, rhi = 0;
        if (quads) {
            const uint32_t p = t >> 2;
            if (p < n) {
                uint32_t hlo, hhi;
                tr_leaf_quad(Q.L, leaf_seed, r[0], hlo, hhi);
                qboard_put<TR_BOARD>(lds, Q.io, hlo, hhi);
                tr_store_quad(tr + leaves, 32 * p + 4 * q, hlo, hhi);
            }
        } else {
#pragma unroll
            for (uint32_t k = 0; k < PER; k++) {
                const uint32_t p = value(n, k);
                if (p < n) {
                    uint32_t h[8];
                    tr_leaf_lane(leaf_seed, r[k], h);
                    tr_put_lane(lds + 8 * p, tr + leaves + 32 * p, h);
                }
            }
            __syncthreads();
        }
        tr_levels<TAIL_THREADS>(Q, lds, quads, n >> 1, tr, l - 1, 0, node_seed, rlo, rhi);
        // the next layer folds in the first wave alone if it has at most 16 values
        const bool alone = n <= 2 * TR_WAVE_MAX;
        if (t < 64) {
            if (t < 4 && ro) tr_store_quad((uint8_t*)ro, 4 * q, rlo, rhi);
            tr_chan_step(Q, chan, rlo, rhi, C, ch);
            if (t == 0 && !alone) qstore(C.alpha, sa);
        } else if (alone) {
            return;
        }
        if (alone) {
            qboard_wave_fence();
        } else {
            __syncthreads();
            if (t >= 64) C.alpha = qload(sa);
        }
    }
    if (t < 64 && C.n_draws) tr_chan_store(Q, C, ch);
}

// Hashes per workgroup (log) for a tree reduction from level k0: the whole tree in one
// workgroup up to 2^8 leaves; above, the levels split about evenly between the workgroups'
// subtrees and the last workgroup's top, with at most 2^8 workgroups (one per CU: a second
// workgroup on a CU halves the issue rate of both) as long as a workgroup's hashes fit its LDS (2^10):
// a level of 2^19 takes 2^9 workgroups (TREE_MAX_BLOCKS).
static uint32_t tree_chunk_log(uint32_t k0) { return k0 <= 8 ? k0 : std::min(10u, std::max(k0 / 2, k0 - 8)); }

template <int SRC>
static void launch_tree_layer(Ctx& c, FriLayerArgs& a, const std::string& cls, double bytes, uint32_t batch,
                              uint64_t bstride, uint32_t* d_cnt) {
    SR_CHECK(a.k0 >= 1 && a.k0 <= TREE_LAYER_MAX_LOG, "tree layer: level out of range");
    SR_CHECK(batch >= 1 && batch <= 65535, "tree layer: batch size");
    // one tree: spread over the CUs; a batch fills the device with its trees, so each workgroup
    // takes as many hashes as it can hold (fewer workgroups, shorter top reductions)
    a.s = batch > 1 ? std::min(a.k0, 10u) : tree_chunk_log(a.k0);
    const uint32_t nb = 1u << (a.k0 - a.s);
    SR_CHECK(nb <= TREE_MAX_BLOCKS && a.s >= 1 && a.s <= 10, "tree layer: chunking");
    // one tree: the context's counters; a batch: the caller's, one region per tree
    SR_CHECK(batch == 1 || d_cnt, "tree layer: a batch needs its own completion counters");
    uint32_t* cnt = batch > 1 ? d_cnt : c.d_tree_cnt;
    SR_CHECK(cnt, "tree layer: context without completion counters");
    a.cnt = cnt;
    a.xr = cnt + TREE_XR_OFFSET;
    a.leaf_seed = c.leaf_seed;
    a.node_seed = c.node_seed;
    a.bstride = bstride;
    KTimer kt(c, cls, batch * bytes);
    hipLaunchKernelGGL(tree_layer_kernel<SRC>, dim3(nb, batch), dim3(TL_THREADS), 0, c.stream, a);
    SR_HIP(hipGetLastError());
}

void launch_tree_top(Ctx& c, DeviceTree& t, uint32_t k0, DevChannel* d_ch, uint8_t* d_root_out, uint32_t batch,
                     uint64_t bstride, uint32_t* d_cnt) {
    SR_CHECK(k0 <= t.max_log, "tree top: level above the leaves");
    FriLayerArgs a{};
    a.tree = t.layers;
    a.k0 = k0;
    a.ch = d_ch;
    a.root_out = (uint32_t*)d_root_out;
    launch_tree_layer<FRI_SRC_HASHES>(c, a, "merkle_top L=" + std::to_string(k0) + (d_ch ? " +channel" : ""),
                                      32.0 * (double)((2ull << k0) - 1), batch, bstride, d_cnt);
}

void launch_tree_from_columns(Ctx& c, const LeafColDev* d_tab, uint32_t n_cols, DeviceTree& t, uint8_t* d_root_out,
                              uint32_t batch, uint64_t bstride, uint32_t* d_cnt) {
    SR_CHECK(d_tab && n_cols >= 1, "tree: no columns");
    FriLayerArgs a{};
    a.cols = d_tab;
    a.n_cols = n_cols;
    a.tree = t.layers;
    a.k0 = t.max_log;
    a.root_out = (uint32_t*)d_root_out;
    const double n = (double)(1ull << t.max_log);
    launch_tree_layer<FRI_SRC_COLUMNS>(c, a,
                                       "merkle_tree L=" + std::to_string(t.max_log) + " cols=" + std::to_string(n_cols),
                                       4.0 * n_cols * n + 32.0 * (2.0 * n - 1.0), batch, bstride, d_cnt);
}

void launch_fri_commit_line(Ctx& c, const uint32_t* d_src, uint32_t log_src, uint32_t* d_dst, DeviceTree& t,
                            DevChannel* d_ch, uint8_t* d_root_out, uint32_t batch, uint64_t bstride, uint32_t* d_cnt) {
    const uint32_t l = log_src - 1;
    SR_CHECK(log_src >= 1 && t.max_log == l && d_ch, "fri commit: layer shape");
    if (l == 0 || l > FRI_LAYER_MAX_LOG) {
        SR_CHECK(batch == 1, "fri commit: batches of layers above 2^18");
        launch_fold_line(c, d_src, log_src, qzero(), d_dst, t.layer(l), d_ch);
        launch_merkle_parents(c, t, d_ch, d_root_out);
        return;
    }
    c.ensure_tower(log_src + 1);
    FriLayerArgs a{};
    a.src_line = (const uint4*)d_src;
    a.inv = c.d_itw + ((1u << (c.tower_log - 1)) - (1u << log_src));
    a.dst_line = (uint4*)d_dst;
    a.tree = t.layers;
    a.k0 = l;
    a.ch = d_ch;
    a.root_out = (uint32_t*)d_root_out;
    const double n = (double)(1ull << l);
    launch_tree_layer<FRI_SRC_LINE>(c, a, "fri_layer", (32.0 + 4.0 + 16.0) * n + 32.0 * (2.0 * n - 1.0), batch,
                                    bstride, d_cnt);
}

void launch_fri_commit_circle(Ctx& c, const uint32_t* const* coords, uint32_t log_src, uint32_t* d_dst,
                              DeviceTree& t, DevChannel* d_ch, uint8_t* d_root_out, uint32_t batch, uint64_t bstride,
                              uint32_t* d_cnt) {
    const uint32_t l = log_src - 1;
    SR_CHECK(log_src >= 1 && t.max_log == l && d_ch, "fri commit: layer shape");
    if (l == 0 || l > FRI_LAYER_MAX_LOG) {
        SR_CHECK(batch == 1, "fri commit: batches of layers above 2^18");
        launch_fold_circle_into_line(c, coords, log_src, qzero(), d_dst, false, t.layer(l), d_ch);
        launch_merkle_parents(c, t, d_ch, d_root_out);
        return;
    }
    FriLayerArgs a{};
    for (int k = 0; k < 4; k++) a.coord[k] = coords[k];
    a.inv = c.inv_circle_y(log_src);
    a.dst_line = (uint4*)d_dst;
    a.tree = t.layers;
    a.k0 = l;
    a.ch = d_ch;
    a.root_out = (uint32_t*)d_root_out;
    const double n = (double)(1ull << l);
    launch_tree_layer<FRI_SRC_CIRCLE>(c, a, "fri_layer_circle", (32.0 + 4.0 + 16.0) * n + 32.0 * (2.0 * n - 1.0),
                                      batch, bstride, d_cnt);
}

void launch_fri_tail(Ctx& c, FriTailArgs& a, uint32_t batch) {
    SR_CHECK(a.top_log <= FRI_TAIL_MAX_LOG + 1 && a.top_log > a.last_log, "fri_tail: layer range");
    SR_CHECK(batch >= 1 && batch <= 65535, "fri_tail: batch size");
    c.ensure_tower(a.top_log + 1);
    // inverse twiddles of halfOdds(l) live at [2^(M-1) - 2^l, 2^(M-1) - 2^(l-1)) of the inverse tower
    a.itw_half = c.d_itw + (1u << (c.tower_log - 1));
    a.leaf_seed = c.leaf_seed;
    a.node_seed = c.node_seed;
    KTimer kt(c, "fri_tail", 0.0);
    hipLaunchKernelGGL(fri_tail_kernel, dim3(batch), dim3(TAIL_THREADS), 0, c.stream, a);
    SR_HIP(hipGetLastError());
}

void launch_fold_line(Ctx& c, const uint32_t* d_src, uint32_t log_src, qm31 alpha, uint32_t* d_dst,
                      uint8_t* d_leaf_out, const DevChannel* d_alpha) {
    SR_CHECK(log_src >= 1, "fold_line: source too short");
    c.ensure_tower(log_src + 1);
    // inverse twiddle layer of halfOdds(log_src): length 2^(log_src-1) at 2^(M-1) - 2^log_src.
    const uint32_t* inv_x = c.d_itw + ((1u << (c.tower_log - 1)) - (1u << log_src));
    uint32_t n = 1u << (log_src - 1);
    KTimer kt(c, "fri_fold_line", (32.0 + 4.0 + 16.0 + (d_leaf_out ? 32.0 : 0.0)) * n);
    hipLaunchKernelGGL(fold_line_kernel, dim3((n + 255) / 256), dim3(256), 0, c.stream, (const uint4*)d_src, log_src,
                       inv_x, alpha, d_alpha, (uint4*)d_dst, d_leaf_out, c.leaf_seed);
    SR_HIP(hipGetLastError());
}

void launch_fold_circle_into_line(Ctx& c, const uint32_t* const* coords, uint32_t log_src, qm31 alpha,
                                  uint32_t* d_dst, bool accumulate, uint8_t* d_leaf_out, const DevChannel* d_alpha,
                                  uint32_t batch, uint64_t bstride) {
    SR_CHECK(log_src >= 1, "fold_circle: source too short");
    SR_CHECK(batch >= 1 && batch <= 65535, "fold_circle: batch size");
    const uint32_t* inv_y = c.inv_circle_y(log_src);
    uint32_t n = 1u << (log_src - 1);
    KTimer kt(c, "fri_fold_circle", batch * (32.0 + 4.0 + 16.0 + (d_leaf_out ? 32.0 : 0.0)) * n);
    hipLaunchKernelGGL(fold_circle_kernel, dim3((n + 255) / 256, batch), dim3(256), 0, c.stream, coords[0], coords[1],
                       coords[2], coords[3], log_src, inv_y, alpha, qsqr(alpha), d_alpha, accumulate,
                       (uint4*)d_dst, d_leaf_out, c.leaf_seed, bstride);
    SR_HIP(hipGetLastError());
}

}  // namespace sr
