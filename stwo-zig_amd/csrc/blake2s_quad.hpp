// One Blake2s compression spread over the four lanes of a quad (device only).
//
// Lane q of the quad (q = lane & 3) holds column q of the 4x4 working state:
// a = v[q], b = v[4+q], c = v[8+q], d = v[12+q], and the chaining words h[q],
// h[4+q].  The column step is one G per lane.  For the diagonal step row b stays and rows
// a, c, d move by 3, 1, 2 lanes: lane j then works on diagonal j - 1.  Moving a instead of b
// keeps the moves off the end of the chain (b is the last row a G writes), so each is the DPP
// operand of the first instruction that reads the row and costs none of its own.
//
// A lone wave issues one instruction per 4 cycles and the G chain has no parallelism to fill,
// so a compression takes its instruction count: 13 per half round.  The message words are
// part of it.  From 16 words in registers every lane selects its 2 words of a half round (6
// selects; fewer where words are constant zeros).  From LDS in lane order (QuadIo below) a
// round's 4 words are one 16-byte read: 1170 cycles for a compression on a lone wave against 1620
// with the selects, 1500 with the write to the next board.  With it and the levels' last-wave loop
// (kernels_fri.hip) FRI layers of 2^15 / 2^12 and 2^11 values went from 30 / 22 to 23 / 15 us, the
// one-workgroup tail from 110 to 87 us (2^16-row XOR proof).
// All four lanes of a quad must be active together.
#pragma once
#include "blake2s.hpp"

namespace sr {

// quad_perm controls: lane q of each quad reads lane (q + k) & 3.
template <int CTRL>
__device__ __forceinline__ uint32_t quad_perm(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xF, 0xF, false);
}
constexpr int QP_ROT1 = 0x39, QP_ROT2 = 0x4E, QP_ROT3 = 0x93;
// quad_perm [k,k,k,k]: every lane reads lane k.
template <int K>
__device__ __forceinline__ uint32_t quad_bcast(uint32_t x) {
    return quad_perm<K * 0x55>(x);
}

struct QuadLane {
    bool q0, q1, q2, q3;
    __device__ __forceinline__ explicit QuadLane(uint32_t q) : q0(q == 0), q1(q == 1), q2(q == 2), q3(q == 3) {}
    // Word q of four; words the compiler knows to be zero cost nothing.
    __device__ __forceinline__ uint32_t sel(uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3) const {
#define SR_Q_ZERO(w) (__builtin_constant_p(w) && (w) == 0)
        if (SR_Q_ZERO(w0) || SR_Q_ZERO(w1) || SR_Q_ZERO(w2) || SR_Q_ZERO(w3)) {
            uint32_t x = 0;
            if (!SR_Q_ZERO(w3)) x = q3 ? w3 : x;
            if (!SR_Q_ZERO(w2)) x = q2 ? w2 : x;
            if (!SR_Q_ZERO(w1)) x = q1 ? w1 : x;
            if (!SR_Q_ZERO(w0)) x = q0 ? w0 : x;
            return x;
        }
#undef SR_Q_ZERO
        return q0 ? w0 : (q1 ? w1 : (q2 ? w2 : w3));
    }
};

constexpr uint8_t B2Q_SIGMA[10][16] = {
    {0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15}, {14, 10, 4, 8, 9, 15, 13, 6, 1, 12, 0, 2, 11, 7, 5, 3},
    {11, 8, 12, 0, 5, 2, 15, 13, 10, 14, 3, 6, 7, 1, 9, 4}, {7, 9, 3, 1, 13, 12, 11, 14, 2, 6, 5, 10, 4, 0, 15, 8},
    {9, 0, 5, 7, 2, 4, 10, 15, 14, 1, 11, 12, 6, 8, 3, 13}, {2, 12, 6, 10, 0, 11, 8, 3, 4, 13, 7, 5, 15, 14, 1, 9},
    {12, 5, 1, 15, 14, 13, 4, 10, 0, 7, 6, 3, 9, 2, 8, 11}, {13, 11, 7, 14, 12, 1, 3, 9, 5, 0, 15, 4, 8, 6, 2, 10},
    {6, 15, 14, 9, 11, 3, 0, 8, 12, 2, 13, 7, 1, 4, 10, 5}, {10, 2, 8, 4, 7, 6, 1, 5, 15, 11, 9, 14, 3, 12, 13, 0}};

// Lane order of round r: words 4 j .. 4 j + 3 are lane j's column x, y and diagonal x, y.
// Nibble w of the result is the place of message word w.
constexpr uint64_t b2q_places(int r) {
    uint64_t m = 0;
    for (int k = 0; k < 16; k++) {
        const int lane = k < 8 ? k / 2 : ((k - 8) / 2 + 1) & 3;
        m |= (uint64_t)(4 * lane + (k < 8 ? 0 : 2) + (k & 1)) << (4 * B2Q_SIGMA[r][k]);
    }
    return m;
}

// From the second half of one half round's G to the first half of the next one's, in which rows
// a, c, d are read through quad permutes PA, PC, PD.  13 instructions in this order: every row
// read through a permute was written at least three instructions before, which the DPP operand
// needs (two wait states) and the compiler would otherwise fill with s_nop, since it puts the
// addition that a permuted operand's partner comes from right before it: 1360 cycles for the 20 half
// rounds of a compression instead of 1040.  All permuted rows are written inside the block, so nothing
// that the compiler puts before it matters.  The rows are early-clobber: x is read after a is written.
#define SR_B2Q_STEP(PA, PC, PD)                                                    \
    asm("v_add3_u32 %0, %0, %1, %4\n\t"                                            \
        "v_xor_b32_e32 %3, %3, %0\n\t"                                             \
        "v_perm_b32 %3, %3, %3, %7\n\t"                                            \
        "v_add_u32_e32 %2, %2, %3\n\t"                                             \
        "v_xor_b32_e32 %1, %1, %2\n\t"                                             \
        "v_alignbit_b32 %1, %1, %1, 7\n\t"                                         \
        "v_add_u32_dpp %0, %0, %5 quad_perm:" PA " row_mask:0xf bank_mask:0xf\n\t" \
        "v_add_u32_e32 %0, %0, %1\n\t"                                             \
        "v_xor_b32_dpp %3, %3, %0 quad_perm:" PD " row_mask:0xf bank_mask:0xf\n\t" \
        "v_perm_b32 %3, %3, %3, %6\n\t"                                            \
        "v_add_u32_dpp %2, %2, %3 quad_perm:" PC " row_mask:0xf bank_mask:0xf\n\t" \
        "v_xor_b32_e32 %1, %1, %2\n\t"                                             \
        "v_alignbit_b32 %1, %1, %1, 12"                                            \
        : "+&v"(a), "+&v"(b), "+&v"(c), "+&v"(d)                                   \
        : "v"(y), "v"(x), "s"(0x01000302u), "s"(0x00030201u))

// (hlo, hhi) = chaining words (q, 4+q) in and out; msg(r) = this lane's words of round r in
// lane order; t = byte counter after this block.
template <class Msg>
__device__ __forceinline__ void b2q_compress(const QuadLane& L, uint32_t& hlo, uint32_t& hhi, const Msg& msg,
                                             uint32_t t, bool last) {
    uint32_t a = hlo, b = hhi;
    uint32_t c = L.sel(SR_B2_IV0, SR_B2_IV1, SR_B2_IV2, SR_B2_IV3);
    uint32_t d = L.sel(SR_B2_IV4 ^ t, SR_B2_IV5, last ? ~SR_B2_IV6 : SR_B2_IV6, SR_B2_IV7);
    uint4 m = msg(0);
    a = a + b + m.x;
    d = rotr16(d ^ a);
    c = c + d;
    b = rotr32(b ^ c, 12);
    uint32_t y = m.y, x;
#pragma unroll
    for (int r = 0; r < 10; r++) {
        x = m.z;
        SR_B2Q_STEP("[3,0,1,2]", "[1,2,3,0]", "[2,3,0,1]");  // to the diagonals
        y = m.w;
        if (r == 9) break;
        m = msg(r + 1);
        x = m.x;
        SR_B2Q_STEP("[1,2,3,0]", "[3,0,1,2]", "[2,3,0,1]");  // to the columns
        y = m.y;
    }
    a = a + b + y;
    d = rotr8(d ^ a);
    c = c + d;
    b = rotr32(b ^ c, 7);
    hlo ^= quad_perm<QP_ROT1>(a) ^ quad_perm<QP_ROT3>(c);
    hhi ^= b ^ quad_perm<QP_ROT2>(d);
}

// m = the 16 message words (the same in all four lanes).
__device__ __forceinline__ void b2_compress_quad(const QuadLane& L, uint32_t& hlo, uint32_t& hhi,
                                                 const uint32_t m[16], uint32_t t, bool last) {
    b2q_compress(
        L, hlo, hhi,
        [&](int r) {
            const uint8_t* s = B2Q_SIGMA[r];
            return make_uint4(L.sel(m[s[0]], m[s[2]], m[s[4]], m[s[6]]), L.sel(m[s[1]], m[s[3]], m[s[5]], m[s[7]]),
                              L.sel(m[s[14]], m[s[8]], m[s[10]], m[s[12]]),
                              L.sel(m[s[15]], m[s[9]], m[s[11]], m[s[13]]));
        },
        t, last);
}

// Messages in LDS in lane order: a board of N slots holds one message per slot, round r of slot
// s as 16 words at byte 64 (N r + s).  A quad that has computed hash i of a level writes it as
// half i & 1 of slot i / 2 (each word to its place in every round: 20 word writes at offsets
// fixed per lane) and parent p reads slot p (10 reads of 16 bytes; the lanes of a wave read
// consecutive bytes).
struct QuadIo {
    uint32_t wr[20];  // byte offsets of words q and 4 + q of half i & 1 in the 10 rounds, slot i / 2
    uint32_t rd;      // byte offset of this lane's words of a round, slot i
    __device__ __forceinline__ QuadIo(uint32_t i, uint32_t q) {
        const uint32_t s = 4 * (8 * (i & 1) + q);
#pragma unroll
        for (int r = 0; r < 10; r++) {
            const uint64_t pl = b2q_places(r);
            wr[2 * r] = 64 * (i >> 1) + 4 * ((uint32_t)(pl >> s) & 15);
            wr[2 * r + 1] = 64 * (i >> 1) + 4 * ((uint32_t)(pl >> (s + 16)) & 15);
        }
        rd = 64 * i + 16 * q;
    }
};

// Round r of hash (hlo, hhi) to the board; of the message at byte offset rd from it.
template <uint32_t N>
__device__ __forceinline__ void qboard_put_round(uint32_t* board, const QuadIo& io, int r, uint32_t hlo, uint32_t hhi) {
    *(uint32_t*)((uint8_t*)board + 64 * N * r + io.wr[2 * r]) = hlo;
    *(uint32_t*)((uint8_t*)board + 64 * N * r + io.wr[2 * r + 1]) = hhi;
}
template <uint32_t N>
__device__ __forceinline__ uint4 qboard_get_round(const uint32_t* board, uint32_t rd, int r) {
    return *(const uint4*)((const uint8_t*)board + rd + 64 * N * r);
}

template <uint32_t N>
__device__ __forceinline__ void qboard_put(uint32_t* board, const QuadIo& io, uint32_t hlo, uint32_t hhi,
                                           uint32_t slot_off = 0) {
#pragma unroll
    for (int r = 0; r < 10; r++) qboard_put_round<N>(board + 16 * slot_off, io, r, hlo, hhi);
}

// The compression of the message at byte offset rd of the board.
template <uint32_t N>
__device__ __forceinline__ void qboard_compress(const QuadLane& L, uint32_t& hlo, uint32_t& hhi,
                                                const uint32_t* board, uint32_t rd, uint32_t t, bool last) {
    uint4 m[10];
#pragma unroll
    for (int r = 0; r < 10; r++) m[r] = qboard_get_round<N>(board, rd, r);
    b2q_compress(L, hlo, hhi, [&](int r) { return m[r]; }, t, last);
}

// Orders a wave's board writes before its later board reads.  LDS serves a wave's accesses in
// order, so this only holds the compiler to the order.
__device__ __forceinline__ void qboard_wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The 8 words of a quad-distributed hash, in every lane of the quad.
__device__ __forceinline__ void quad_gather8(uint32_t hlo, uint32_t hhi, uint32_t out[8]) {
    out[0] = quad_bcast<0>(hlo);
    out[1] = quad_bcast<1>(hlo);
    out[2] = quad_bcast<2>(hlo);
    out[3] = quad_bcast<3>(hlo);
    out[4] = quad_bcast<0>(hhi);
    out[5] = quad_bcast<1>(hhi);
    out[6] = quad_bcast<2>(hhi);
    out[7] = quad_bcast<3>(hhi);
}

}  // namespace sr
