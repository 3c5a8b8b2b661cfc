// Small kernels: proof-of-work grind, decommitment gather, batch inverse,
// bit reversal, accumulation and QM31 AoS -> coordinate columns.
#include <algorithm>

#include "runtime.hpp"

namespace sr {

// PoW (src/core/channel/blake2s.zig:135-166,289-300): H(prefix32 || LE64(nonce)),
// one 40-byte final block; valid when the first 16 bytes, read as a
// little-endian 128-bit integer, have >= bits trailing zeros.  The lowest valid
// nonce of the launch range is kept with a 64-bit atomic min (vector atomic).
//
// The grind is bound by the instruction count of the compression, so it does only what
// depends on the nonce and what the test needs: the nonce enters in the first diagonal step,
// so the 4 column steps before it and the 3 other diagonal steps of that round (all their
// message words are the prefix's or zero) are done once on the host (PowStart), and only
// digest word 0 is formed, which drops half of the last diagonal step (13% of the
// compression).  A nonce whose word 0 passes is hashed in full.
struct PowStart {
    uint32_t v[16];  // working state, the step on (v0, v5, v10, v15) of round 0 still to do
    uint32_t p[8];   // prefix words
    uint32_t h0;     // chaining word 0
};

SR_HD PowStart pow_start(const uint32_t prefix[8]) {
    PowStart s;
    uint32_t h[8];
    b2_init(h);
    const uint32_t* m = prefix;
    for (int k = 0; k < 8; k++) s.p[k] = prefix[k];
    s.h0 = h[0];
    uint32_t v0 = h[0], v1 = h[1], v2 = h[2], v3 = h[3], v4 = h[4], v5 = h[5], v6 = h[6], v7 = h[7];
    uint32_t v8 = SR_B2_IV0, v9 = SR_B2_IV1, v10 = SR_B2_IV2, v11 = SR_B2_IV3;
    uint32_t v12 = SR_B2_IV4 ^ 40u, v13 = SR_B2_IV5, v14 = ~SR_B2_IV6, v15 = SR_B2_IV7;
    SR_B2_G(v0, v4, v8, v12, m[0], m[1])
    SR_B2_G(v1, v5, v9, v13, m[2], m[3])
    SR_B2_G(v2, v6, v10, v14, m[4], m[5])
    SR_B2_G(v3, v7, v11, v15, m[6], m[7])
    SR_B2_G(v1, v6, v11, v12, 0u, 0u)
    SR_B2_G(v2, v7, v8, v13, 0u, 0u)
    SR_B2_G(v3, v4, v9, v14, 0u, 0u)
    const uint32_t v[16] = {v0, v1, v2, v3, v4, v5, v6, v7, v8, v9, v10, v11, v12, v13, v14, v15};
    for (int k = 0; k < 16; k++) s.v[k] = v[k];
    return s;
}

// Digest word 0 of H(prefix || nonce).
__device__ __forceinline__ uint32_t pow_word0(const PowStart& s, uint64_t nonce) {
    const uint32_t m[16] = {s.p[0], s.p[1], s.p[2], s.p[3], s.p[4], s.p[5], s.p[6], s.p[7],
                            (uint32_t)nonce, (uint32_t)(nonce >> 32), 0, 0, 0, 0, 0, 0};
    uint32_t v0 = s.v[0], v1 = s.v[1], v2 = s.v[2], v3 = s.v[3], v4 = s.v[4], v5 = s.v[5], v6 = s.v[6], v7 = s.v[7];
    uint32_t v8 = s.v[8], v9 = s.v[9], v10 = s.v[10], v11 = s.v[11], v12 = s.v[12], v13 = s.v[13], v14 = s.v[14],
             v15 = s.v[15];
    SR_B2_G(v0, v5, v10, v15, m[8], m[9])
    SR_B2_ROUNDS_1_9
    return s.h0 ^ v0 ^ v8;
}

__device__ __forceinline__ void pow_try(const PowStart& s, uint32_t bits, uint64_t nonce,
                                        unsigned long long* __restrict__ best) {
    const uint32_t w0 = pow_word0(s, nonce);
    if (w0 & (bits < 32 ? (1u << bits) - 1 : 0xFFFFFFFFu)) return;
    if (bits > 32) {  // one nonce in 2^32: the further words from the whole digest
        const uint32_t m[16] = {s.p[0], s.p[1], s.p[2], s.p[3], s.p[4], s.p[5], s.p[6], s.p[7],
                                (uint32_t)nonce, (uint32_t)(nonce >> 32), 0, 0, 0, 0, 0, 0};
        uint32_t h[8];
        b2_init(h);
        b2_compress(h, m, 40, true);
        uint32_t tz = 128;
        if (h[1]) tz = 32 + __builtin_ctz(h[1]);
        else if (h[2]) tz = 64 + __builtin_ctz(h[2]);
        else if (h[3]) tz = 96 + __builtin_ctz(h[3]);
        if (tz < bits) return;
    }
    atomicMin(best, (unsigned long long)nonce);
}

// Block b tries nonces [256 PER b, 256 PER (b + 1)) of the range, 256 at a time, and stops at the
// first ones above the best nonce found so far (the load of that word overlaps a compression),
// so a launch may cover several times the expected work.  Every nonce below the result has
// been tried: a block only stops above a valid one.  Blocks start in order, which keeps the
// tried nonces together; threads striding over the whole range do not (the SIMDs run their
// oldest wave first, and it gets far ahead of the others).  At 26 bits, useful nonces per
// second over 12 digests: 41 G; striding threads 22 G; one nonce per thread, the whole
// compression and launches of 2^24, each ground to its end, 34 G.
template <uint32_t PER>
__global__ __launch_bounds__(256) void pow_kernel(PowStart s, uint32_t bits, uint64_t base, uint64_t count,
                                                  unsigned long long* __restrict__ best) {
    const uint64_t first = (uint64_t)blockIdx.x * (256 * PER);
    unsigned long long found = __hip_atomic_load(best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll 1
    for (uint32_t k = 0; k < PER; k++) {
        const uint64_t i = first + 256 * k + threadIdx.x;
        if (i >= count || found < base + first + 256 * k) return;
        if (k + 1 < PER) found = __hip_atomic_load(best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        pow_try(s, bits, base + i, best);
    }
}
// Prefix blockIdx.y of a batch: its 8 words at prefix + 8 y, its best nonce at best[y].  A
// block whose first nonce is above the best one found for its prefix (by an earlier range or
// an earlier block of this launch) has nothing to find.
__global__ __launch_bounds__(256) void pow_batch_kernel(const uint32_t* __restrict__ prefix, uint32_t bits,
                                                        uint64_t base, uint64_t count,
                                                        unsigned long long* __restrict__ best) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= count) return;
    const unsigned long long found =
        __hip_atomic_load(best + blockIdx.y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (found < base + (uint64_t)blockIdx.x * 256) return;
    pow_try(pow_start(prefix + 8 * blockIdx.y), bits, base + i, best + blockIdx.y);
}
void launch_pow_grind_batch(Ctx& c, const uint32_t* d_prefix, uint32_t batch, uint32_t bits, uint64_t base,
                            uint64_t count, unsigned long long* d_best) {
    SR_CHECK(batch >= 1 && batch <= 65535, "pow: batch size");
    const uint64_t blocks = (count + 255) / 256;
    SR_CHECK(blocks < (1ull << 31), "pow: launch range too large");
    KTimer kt(c, "pow_grind", 0.0);
    hipLaunchKernelGGL(pow_batch_kernel, dim3((uint32_t)blocks, batch), dim3(256), 0, c.stream, d_prefix, bits, base,
                       count, d_best);
    SR_HIP(hipGetLastError());
}

uint64_t launch_pow_grind(Ctx& c, const uint8_t prefix[32], uint32_t bits, uint64_t base, uint64_t count) {
    DBuf best(&c, 8);
    uint64_t init = UINT64_MAX;
    SR_HIP(hipMemcpyAsync(best.p, c.stage(&init, 8), 8, hipMemcpyHostToDevice, c.stream));
    uint32_t w[8];
    memcpy(w, prefix, 32);
    // 8 nonces per thread once that still fills the chip several times (the blocks left after the
    // solution only start and end), 1 below
    const uint32_t per = count > (1ull << 20) ? 8u : 1u;
    const uint64_t blocks = (count + 256 * per - 1) / (256 * per);
    SR_CHECK(blocks < (1ull << 31), "pow: launch range too large");
    KTimer kt(c, "pow_grind", 0.0);
    if (per == 8)
        hipLaunchKernelGGL(pow_kernel<8>, dim3((uint32_t)blocks), dim3(256), 0, c.stream, pow_start(w), bits, base,
                           count, best.as<unsigned long long>());
    else
        hipLaunchKernelGGL(pow_kernel<1>, dim3((uint32_t)blocks), dim3(256), 0, c.stream, pow_start(w), bits, base,
                           count, best.as<unsigned long long>());
    SR_HIP(hipGetLastError());
    uint64_t* h = (uint64_t*)c.pinned(8);
    SR_HIP(hipMemcpyAsync(h, best.p, 8, hipMemcpyDeviceToHost, c.stream));
    c.sync();
    return *h;
}

// Nonces of one launch: 16 times the expected work up to 2^24 (a launch misses with
// probability e^-16), 4 times above (e^-4: what the search leaves of the range still costs
// the start of its blocks), at most 2^30.
uint64_t pow_launch_nonces(uint32_t bits) {
    return 1ull << std::min(30u, std::max(14u, std::min(bits + 4, std::max(24u, bits + 2))));
}

// Decommitment gather: out[i] = word at absolute device address addr[i].
__global__ void gather_kernel(const uint64_t* __restrict__ addr, uint64_t n, uint32_t* __restrict__ out) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = *(gcu32*)(uintptr_t)addr[i];
}
void launch_gather(Ctx& c, const uint64_t* d_addr, uint64_t n, uint32_t* d_out) {
    if (!n) return;
    hipLaunchKernelGGL(gather_kernel, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, c.stream, d_addr, n, d_out);
    SR_HIP(hipGetLastError());
}

// Field inverse per element (fields/mod.zig:16 batchInverse; the inverse is unique).
__global__ void inverse_kernel(const uint32_t* __restrict__ in, uint64_t n, uint32_t* __restrict__ out) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = minv(in[i]);
}
void launch_batch_inverse(Ctx& c, const uint32_t* d_in, uint64_t n, uint32_t* d_out) {
    if (!n) return;
    hipLaunchKernelGGL(inverse_kernel, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, c.stream, d_in, n, d_out);
    SR_HIP(hipGetLastError());
}

// In-place bit reversal of 2^log elements of `wpe` words (core/utils.zig:20-34).
__global__ void bitrev_kernel(uint32_t* __restrict__ v, uint32_t log_size, uint32_t wpe) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (1u << log_size)) return;
    uint32_t j = bitrev32(i, log_size);
    if (j <= i) return;
    for (uint32_t k = 0; k < wpe; k++) {
        uint32_t t = v[(uint64_t)i * wpe + k];
        v[(uint64_t)i * wpe + k] = v[(uint64_t)j * wpe + k];
        v[(uint64_t)j * wpe + k] = t;
    }
}
void launch_bit_reverse(Ctx& c, uint32_t* d_vals, uint32_t log_size, uint32_t wpe) {
    uint32_t n = 1u << log_size;
    hipLaunchKernelGGL(bitrev_kernel, dim3((n + 255) / 256), dim3(256), 0, c.stream, d_vals, log_size, wpe);
    SR_HIP(hipGetLastError());
}

// AccumulationOps.accumulate (backend/accumulation_ops.zig): column-wise add.
__global__ void accumulate_kernel(uint32_t* __restrict__ acc, const uint32_t* __restrict__ src, uint64_t n) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) acc[i] = madd(acc[i], src[i]);
}
void launch_accumulate(Ctx& c, uint32_t* d_acc, const uint32_t* d_src, uint64_t n_words) {
    if (!n_words) return;
    hipLaunchKernelGGL(accumulate_kernel, dim3((uint32_t)((n_words + 255) / 256)), dim3(256), 0, c.stream, d_acc,
                       d_src, n_words);
    SR_HIP(hipGetLastError());
}

__global__ void coords_kernel(const uint4* __restrict__ q, uint64_t n, uint32_t* __restrict__ c0,
                              uint32_t* __restrict__ c1, uint32_t* __restrict__ c2, uint32_t* __restrict__ c3) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint4 v = q[i];
    c0[i] = v.x;
    c1[i] = v.y;
    c2[i] = v.z;
    c3[i] = v.w;
}
void launch_qm31_to_coords(Ctx& c, const uint32_t* d_qm31, uint64_t n, uint32_t* const* coords) {
    if (!n) return;
    hipLaunchKernelGGL(coords_kernel, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, c.stream,
                       (const uint4*)d_qm31, n, coords[0], coords[1], coords[2], coords[3]);
    SR_HIP(hipGetLastError());
}

}  // namespace sr
