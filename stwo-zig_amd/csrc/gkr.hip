// GKR batch prover with the whole transcript on the device (src/prover/lookups/
// gkr_prover.zig:34-298 with sumcheck.zig:76-197 and the oracle of
// gkr_circuit.zig:231-429).
//
// The layer stacks (nextLayer), the eq tables, the sum-check rounds, the
// channel (mixFelts / drawSecureFelt on one quad of lanes, chan.hpp) and the
// masks all run on the GPU; the host only enqueues launches and reads the
// transcript back once.  Per GKR layer L (L sum-check rounds):
//   * begin: newly active instances take their output claims, the claims are
//     mixed, alpha and lambda drawn, the batched claims formed; one lane per
//     round rho precomputes what the round polynomial needs from the eq point
//     y (the eq-prefix inverse prod_{i<=rho} 1/(1-y_i), the extra Lagrange node
//     b = (1-y_rho)/(1-2y_rho) and the basis coefficients for the nodes
//     0, 1, 2, b), so no round inverts anything;
//   * rounds: fixing the previous round's variable is fused into this round's
//     sums (in place: index j < h is written by the thread that reads j and
//     j + h); rounds of more than GD_SMALL_TERMS terms are one launch over
//     many workgroups whose last workgroup (atomic counter, no waiting) turns
//     the sums into the round polynomial, mixes it and draws the challenge;
//     smaller rounds, whole small layers and the layer end (masks, challenge,
//     next claims) run in one workgroup.
// The round polynomial r(x) through (0, r0), (1, claim - r0), (2, r2), (b, 0)
// (correctSumAsPolyInFirstVariable, gkr_circuit.zig:390-429) is unique, so the
// closed-form coefficients equal the reference's Lagrange interpolation.
//
// Proof word stream (what stwo_rocm_gkr_prove_batch returns):
//   per GKR layer: n_rounds, each [len, len QM31 coefficients];
//                  n_masks, each [instance, n_columns, 2*n_columns QM31];
//   per instance: [n, output claims]; [n, ood point];
//   per instance: [n, claims to verify], n_variables; final channel digest (8 words).
#include <memory>
#include <vector>

#include "chan.hpp"
#include "prover.hpp"

namespace sr {

namespace {

// Univariate polynomial with ascending QM31 coefficients, trailing zeros trimmed
// (utils.zig:14-214).
struct Poly {
    std::vector<qm31> c;
    void trim() {
        while (!c.empty() && qiszero(c.back())) c.pop_back();
    }
    qm31 eval(qm31 x) const {
        qm31 acc = qzero();
        for (size_t i = c.size(); i > 0; i--) acc = qadd(qmul(acc, x), c[i - 1]);
        return acc;
    }
};

qm31 qdiv(qm31 a, qm31 b) { return qmul(a, qinv(b)); }

// Lagrange interpolation through 4 points (utils.zig:147-190).
Poly lagrange(const qm31 xs[4], const qm31 ys[4]) {
    Poly acc;
    for (int i = 0; i < 4; i++) {
        qm31 scale = ys[i];
        for (int j = 0; j < 4; j++)
            if (j != i) scale = qdiv(scale, qsub(xs[i], xs[j]));
        Poly term;
        term.c = {scale};
        term.trim();
        for (int j = 0; j < 4 && !term.c.empty(); j++) {
            if (j == i) continue;
            Poly nt;
            nt.c.assign(term.c.size() + 1, qzero());
            for (size_t k = 0; k < term.c.size(); k++) {
                nt.c[k] = qadd(nt.c[k], qmul(term.c[k], qneg(xs[j])));
                nt.c[k + 1] = qadd(nt.c[k + 1], term.c[k]);
            }
            nt.trim();
            term = nt;
        }
        Poly s;
        s.c.assign(std::max(acc.c.size(), term.c.size()), qzero());
        for (size_t k = 0; k < s.c.size(); k++)
            s.c[k] = qadd(k < acc.c.size() ? acc.c[k] : qzero(), k < term.c.size() ? term.c[k] : qzero());
        s.trim();
        acc = s;
    }
    return acc;
}

qm31 eq_one(qm31 x, qm31 y) { return qadd(qmul(x, y), qmul(qsub(qone(), x), qsub(qone(), y))); }

// correctSumAsPolyInFirstVariable (gkr_circuit.zig:390-429).
Poly correct_sum(qm31 f0, qm31 f2, qm31 claim, const std::vector<qm31>& y, uint32_t k) {
    SR_CHECK(k >= 1 && k <= y.size(), "gkr: invalid k");
    const size_t n = y.size();
    qm31 eq_prefix = qone();
    for (size_t i = 0; i < n - k + 1; i++) eq_prefix = qmul(eq_prefix, qsub(qone(), y[i]));
    SR_CHECK(!qiszero(eq_prefix), "gkr: division by zero");
    const qm31 a_const = qinv(eq_prefix);
    const qm31 yk = y[n - k];
    const qm31 den = qsub(qone(), qadd(yk, yk));
    SR_CHECK(!qiszero(den), "gkr: division by zero");
    const qm31 b_const = qdiv(qsub(qone(), yk), den);
    const qm31 two = qfromm(2);
    const qm31 r0 = qmul(qmul(f0, qsub(qone(), yk)), a_const);
    const qm31 r2 = qmul(qmul(f2, eq_one(two, yk)), a_const);
    const qm31 xs[4] = {qzero(), qone(), two, b_const};
    const qm31 ys[4] = {r0, qsub(claim, r0), r2, qzero()};
    return lagrange(xs, ys);
}

qm31 from_acc(const uint64_t* a) { return {{mred64(a[0]), mred64(a[1])}, {mred64(a[2]), mred64(a[3])}}; }

}  // namespace

// GkrMultivariatePolyOracle.sumAsPolyInFirstVariable (gkr_circuit.zig:261-316) for one
// layer on the device: returns the trimmed coefficients of the round polynomial.
std::vector<qm31> gkr_sum_as_poly(Ctx& c, int kind, const uint32_t* d_eq, const uint32_t* d_num,
                                  const uint32_t* d_den, uint32_t n_vars, qm31 lambda, qm31 claim,
                                  const std::vector<qm31>& y, qm31 correction) {
    SR_CHECK(n_vars >= 2, "gkr: the oracle needs at least one variable");
    SR_CHECK(n_vars - 1 <= y.size(), "gkr: eq point shorter than the oracle");
    DBuf acc(&c, 64);
    launch_zero_u64(c, acc.as<unsigned long long>(), 8);
    launch_gkr_sums(c, kind, d_eq, d_num, d_den, n_vars, lambda, acc.as<unsigned long long>());
    uint64_t* h = (uint64_t*)c.pinned(64);
    SR_HIP(hipMemcpyAsync(h, acc.p, 64, hipMemcpyDeviceToHost, c.stream));
    c.sync();
    const qm31 f0 = qmul(from_acc(h), correction), f2 = qmul(from_acc(h + 4), correction);
    return correct_sum(f0, f2, claim, y, n_vars - 1).c;
}


// ====================================================================== device-resident batch prover
namespace {

constexpr uint32_t GD_MAX_INST = 8;
constexpr uint32_t GD_MAX_VARS = 30;
// A round of at most this many terms (over its instances) runs in one workgroup.  By itself a round
// of 384 terms takes 23K cycles there, 512 25K and 768 36K, and a launch over many workgroups
// 27..29K.  Whole proofs are flat up to 512 (us at limits of 256 / 384 / 512 / 768, runs of one side
// differ by 5..50): one instance of 2^18 1507 / 1499 / 1492 / 1491, two of 2^18 and 2^16 1641 / 1643 /
// 1654 / 1650, four of 2^16 1551 / 1542 / 1567 / 1561, four of 2^18, 2^17, 2^15, 2^9 1824 / 1815 / 1810 /
// 1874.  So the limit is the middle one, the best or within 1% on each.
constexpr uint32_t GD_SMALL_TERMS = 384;
// Most rounds of one such launch: layers 0..9 of one instance (layer L has L rounds, the first of 2^(L-1)
// terms).
constexpr uint32_t gd_fused_rounds(uint32_t terms) {
    uint32_t top = 0;
    while ((1u << top) <= terms) top++;
    return top * (top + 1) / 2;
}
constexpr uint32_t GD_FUSED_ROUNDS = gd_fused_rounds(GD_SMALL_TERMS);
constexpr uint32_t GD_FT = 512;       // one-workgroup kernel: 7 summing waves + 1 for the pending update
constexpr uint32_t GD_RT = 256;       // threads per workgroup of the round and begin kernels
constexpr uint32_t GD_REC_ROUND = 17;  // [len, 4 QM31] per sum-check round
constexpr uint32_t GD_REC_MASK = 16;   // [num0, num1, den0, den1] per instance and layer

// Layer stack of one instance: layer l has l variables (2^l values); num is QM31 AoS,
// M31 for a multiplicities input layer, absent for grand products and singles.
struct GdInst {
    const uint32_t* num[GD_MAX_VARS + 1];
    const uint32_t* den[GD_MAX_VARS + 1];
    uint32_t kind[GD_MAX_VARS + 1];
    uint32_t n_vars;
    uint32_t* scr_num;  // fixed layers: 2^(n_vars-1) QM31 each
    uint32_t* scr_den;
};

struct GdState {
    uint32_t dg[8];
    uint32_t n_draws, status, pad0, pad00;
    uint32_t outputs[GD_MAX_INST][2][4];  // transcript order: [den] or [num, den]
    uint32_t claims[GD_MAX_INST][2][4];
    uint32_t sc_claim[GD_MAX_INST][4];
    uint32_t corr[GD_MAX_INST][4];
    uint32_t alpha_pow[GD_MAX_INST][4];
    uint32_t lambda[4];
    uint32_t r[4];
    uint32_t ood[GD_MAX_VARS + 1][4];  // eq point of the current layer
    uint32_t asg[GD_MAX_VARS][4];      // challenges of the current layer's rounds
    uint32_t pre[GD_MAX_VARS][3][4][4];  // per round, for coefficient q: the factors of A, B, C (see fin)
    uint32_t mask[GD_MAX_INST][4][4];
    // the last round's claim update, applied while the next round sums (or dropped at the
    // layer end, where the claims are rebuilt): its coefficients, round and instance flags
    uint32_t craw[GD_MAX_INST][4][4];
    uint32_t pend, pend_rho, pad1, pad2;
    uint32_t pend_flags[GD_MAX_INST];  // bit 0: active, bit 1: summed in that round
    // the current round's coefficient c_q of instance i as A * s0 + C * s2 + B in the round
    // sums s0, s2 (set at the round start from the claim, the correction and the round's
    // basis rows), and the instance's flags in this round (bit 0: active, bit 1: summed)
    uint32_t fin[GD_MAX_INST][4][3][4];
    uint32_t rflags[GD_MAX_INST];
};
static_assert(sizeof(GdState) % 8 == 0 && sizeof(GdInst) % 8 == 0, "copies in 8-byte words");
constexpr uint32_t GD_MAX_BX = 1024;   // workgroups per instance in a round launch
constexpr uint32_t GD_CNT_GROUPS = 16;  // completion sub-counters, one 128-byte line each
constexpr uint32_t GD_CNT_STRIDE = 32;  // words between counters

// Layers and tables are in device memory (their pointers come from a table, so the compiler is
// told: a flat access would also wait on LDS).
__device__ __forceinline__ qm31 gd_ld(const uint32_t* p, uint64_t i) {
    const u32x4 v = ((const SR_GLOBAL u32x4*)p)[i];
    return {{v.x, v.y}, {v.z, v.w}};
}
__device__ __forceinline__ void gd_st(uint32_t* p, uint64_t i, qm31 v) {
    ((SR_GLOBAL u32x4*)p)[i] = u32x4{v.c0.a, v.c0.b, v.c1.a, v.c1.b};
}
__device__ __forceinline__ qm31 gd_num(uint32_t kind, const uint32_t* num, uint64_t j) {
    if (kind == GKR_LOGUP_GENERIC) return gd_ld(num, j);
    if (kind == GKR_LOGUP_MULTIPLICITIES) return qfromm(((gcu32*)num)[j]);
    return qone();
}
__device__ __forceinline__ uint32_t gd_fixed_kind(uint32_t kind) {
    return kind == GKR_LOGUP_MULTIPLICITIES ? (uint32_t)GKR_LOGUP_GENERIC : kind;
}
__device__ __forceinline__ bool gd_has_num(uint32_t kind) {
    return kind == GKR_LOGUP_GENERIC || kind == GKR_LOGUP_MULTIPLICITIES;
}
__device__ __forceinline__ qm31 gd_shfl(qm31 v, int src) {
    return {{(uint32_t)__shfl((int)v.c0.a, src), (uint32_t)__shfl((int)v.c0.b, src)},
            {(uint32_t)__shfl((int)v.c1.a, src), (uint32_t)__shfl((int)v.c1.b, src)}};
}
__device__ __forceinline__ qm31 gd_shfl_xor(qm31 v, int m) {
    return {{(uint32_t)__shfl_xor((int)v.c0.a, m), (uint32_t)__shfl_xor((int)v.c0.b, m)},
            {(uint32_t)__shfl_xor((int)v.c1.a, m), (uint32_t)__shfl_xor((int)v.c1.b, m)}};
}
template <int CTRL>
__device__ __forceinline__ qm31 gd_qperm(qm31 v) {
    return {{quad_perm<CTRL>(v.c0.a), quad_perm<CTRL>(v.c0.b)}, {quad_perm<CTRL>(v.c1.a), quad_perm<CTRL>(v.c1.b)}};
}
// The 8 sums of a wave by recursive halving: at each exchange a lane keeps half of its values
// and adds its partner's copy of that half (lane bit 5 picks the half first, then bits 4 and
// 3), then three full exchanges.  6 dependent rounds of word exchanges where 8 separate
// reductions take 48; the rounds sit on the latency path of every round.  Afterwards lane l
// holds the total of value (l >> 3) & 7.
__device__ __forceinline__ uint64_t gd_xchg(uint64_t v, uint32_t addr) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute((int)addr, (int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute((int)addr, (int)(uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ uint64_t gd_wave_sum8(uint64_t (&x)[8], uint32_t lane) {
#pragma unroll
    for (int st = 0; st < 3; st++) {
        const uint32_t h = 4u >> st, b = 32u >> st;
        // the halves are picked with a lane mask, not a select of two elements (which the
        // compiler turns into an indexed read of the whole array)
        const uint64_t m = 0ull - (uint64_t)((lane & b) != 0);  // all ones: keep the upper half
        const uint32_t addr = (lane ^ b) << 2;
#pragma unroll
        for (uint32_t i = 0; i < h; i++) {
            const uint64_t lo = x[i], hi = x[i + h];
            const uint64_t send = (lo & m) | (hi & ~m);
            x[i] = (lo ^ hi ^ send) + gd_xchg(send, addr);
        }
    }
    uint64_t v = x[0];
    v += gd_xchg(v, (lane ^ 4) << 2);
    v += gd_xchg(v, (lane ^ 2) << 2);
    v += gd_xchg(v, (lane ^ 1) << 2);
    return v;
}
__device__ __forceinline__ void gd_qstore(uint32_t* w, qm31 v) { qstore(v, w); }

// The channel on one wave (all 64 lanes, every quad computing the same).  Message words go
// through LDS in lane order (blake2s_quad.hpp): each lane below 24 owns one word and writes
// it to its place in the 10 rounds.  Lanes 0..15 own the payload words w = 4 (t & 3) + (t >> 2),
// so that lane t takes word t >> 2 of a QM31 coefficient t & 3; lanes 16..23 own the digest.
// Boards: mix block 0 (digest || payload 0..7), mix block 1 (payload 8..15 || zeros), draw
// (digest || counter || zeros).
constexpr uint32_t GD_CHAN_WORDS = 3 * 160;
struct GdChan {
    uint32_t t, ad[10];
    QuadLane L;
    uint32_t* bd;
    uint32_t ilo, ihi;
    // All threads of the block call it; a barrier must follow.
    __device__ __forceinline__ GdChan(uint32_t* boards, uint32_t tid) : t(tid), L(tid & 3), bd(boards) {
        for (uint32_t i = tid; i < GD_CHAN_WORDS; i += blockDim.x) boards[i] = 0;
        const uint32_t w = t < 16 ? 4 * (t & 3) + (t >> 2) : 0;
        const uint32_t m = t < 16 ? (w < 8 ? 8 + w : w - 8) : t & 7, blk = t < 16 && w >= 8 ? 160u : 0u;
#pragma unroll
        for (int r = 0; r < 10; r++) ad[r] = blk + 16 * r + ((uint32_t)(b2q_places(r) >> (4 * m)) & 15);
        ilo = L.sel(SR_B2_IV0 ^ 0x01010020u, SR_B2_IV1, SR_B2_IV2, SR_B2_IV3);
        ihi = L.sel(SR_B2_IV4, SR_B2_IV5, SR_B2_IV6, SR_B2_IV7);
    }
    __device__ __forceinline__ uint32_t pay_index() const { return 4 * (t & 3) + (t >> 2); }
    // This lane's digest word of a hash in the quads (meant in lanes 16..23).
    __device__ __forceinline__ uint32_t digest_word(uint32_t hlo, uint32_t hhi) const { return (t & 4) ? hhi : hlo; }

    // dv <- Blake2s(digest || payload[0..n_words)), n_words <= 16 and uniform; pv = this lane's
    // payload word (zero beyond n_words), dv = its digest word.
    __device__ __forceinline__ void mix(uint32_t& dv, uint32_t pv, uint32_t n_words) const {
        if (t < 24) {
            const uint32_t v = t < 16 ? pv : dv;
#pragma unroll
            for (int r = 0; r < 10; r++) bd[ad[r]] = v;
        }
        qboard_wave_fence();
        uint32_t hlo = ilo, hhi = ihi;
        const uint32_t len = 32 + 4 * n_words;
#pragma unroll 1
        for (uint32_t b = 0; b < (len > 64 ? 2u : 1u); b++) {
            const bool last = 64 * (b + 1) >= len;
            qboard_compress<1>(L, hlo, hhi, bd + 160 * b, 16 * (t & 3), last ? len : 64, last);
        }
        dv = digest_word(hlo, hhi);
    }

    // One secure felt of the digest: words = Blake2s(digest || LE32(n_draws) || 0x00),
    // n_draws += 1, redrawn until all 8 are < 2p; st = 1 after 64 rejections.
    __device__ __forceinline__ qm31 draw(uint32_t dv, uint32_t& n_draws, uint32_t& st) const {
#pragma unroll 1
        for (uint32_t k = 0; k < 64; k++) {
            qboard_wave_fence();
            if (t == 0 || (t >= 16 && t < 24)) {  // lane 0's word is message word 8
                const uint32_t v = t == 0 ? n_draws : dv;
#pragma unroll
                for (int r = 0; r < 10; r++) bd[320 + ad[r]] = v;
            }
            qboard_wave_fence();
            uint32_t olo = ilo, ohi = ihi;
            qboard_compress<1>(L, olo, ohi, bd + 320, 16 * (t & 3), 37, true);
            n_draws++;
            uint32_t bad = (olo >= 2u * P || ohi >= 2u * P) ? 1u : 0u;
            bad |= quad_perm<QP_ROT1>(bad);
            bad |= quad_perm<QP_ROT2>(bad);
            if (!__builtin_amdgcn_readfirstlane(bad))
                return {{mred64(quad_bcast<0>(olo)), mred64(quad_bcast<1>(olo))},
                        {mred64(quad_bcast<2>(olo)), mred64(quad_bcast<3>(olo))}};
        }
        st = 1;
        return qzero();
    }
};

// Instance view at GKR layer L: active once n_vars + L >= n_layers; its oracle layer has
// onv + 1 variables, onv = L + n_vars - n_layers.
struct GdView {
    bool active;
    uint32_t onv;
};
__device__ __forceinline__ GdView gd_view(const GdInst& in, uint32_t n_layers, uint32_t L) {
    GdView v;
    v.active = in.n_vars + L >= n_layers;
    v.onv = v.active ? in.n_vars + L - n_layers : 0;
    return v;
}

// Sum-check term k of one instance at round rho (nt = 2^(rem-1) terms): the four values
// of the current layer at rows 2k, 2k+1, 2(nt+k), 2(nt+k)+1, fixed on the fly from the
// previous layer (2x as long) when `fix`, then the terms at x = 0 and x = 2
// (gkr_circuit.zig:505-643), each multiplied by eq[k].
// The term is spread over a quad (all four lanes active, same k): lane j fixes and
// stores value j and, for fractions, forms m_j = n_j + lambda d_j, so that the term
// (d1 n0 + d0 n1) + lambda d0 d1 is d1 m0 + d0 n1 (at x = 2 the values are 2 v_{2,3} - v_{0,1},
// and m follows them).  The values are exchanged with DPP, every lane forms one product chosen
// by its lane index (branch-free) and the pairs add up: a quad's lanes pass through 5 products
// (6 with lambda as a factor of the sum).  Lanes 0 and 2 end with t0 and t2.
// Returns e * t in lanes 0 (x = 0) and 2 (x = 2), zero elsewhere.
__device__ __forceinline__ qm31 gd_term_quad(bool fix, uint32_t kind, const uint32_t* num, const uint32_t* den,
                                             uint32_t* dnum, uint32_t* dden, qm31 r, uint64_t nt, uint64_t k,
                                             qm31 lambda, const uint32_t* eq, uint32_t j) {
    const uint64_t jj = j < 2 ? 2 * k + j : 2 * (nt + k) + (j - 2);
    const uint64_t h = 4 * nt;
    const bool has_num = gd_has_num(kind);
    const qm31 e = gd_ld(eq, k);
    const qm31 da = gd_ld(den, jj);
    const qm31 db = fix ? gd_ld(den, jj + h) : qzero();
    const qm31 na = has_num ? gd_num(kind, num, jj) : qone();
    const qm31 nb = has_num && fix ? gd_num(kind, num, jj + h) : qone();
    const qm31 d = fix ? qadd(qmul(qsub(db, da), r), da) : da;
    const qm31 n = has_num && fix ? qadd(qmul(qsub(nb, na), r), na) : na;
    if (fix) {
        gd_st(dden, jj, d);
        if (has_num) gd_st(dnum, jj, n);
    }
    const qm31 d0 = quad_bcast_q<0>(d), d1 = quad_bcast_q<1>(d), d2 = quad_bcast_q<2>(d), d3 = quad_bcast_q<3>(d);
    const qm31 d20 = qsub(qadd(d2, d2), d0), d21 = qsub(qadd(d3, d3), d1);
    const bool l0 = j == 0, l1 = j == 1, l2 = j == 2;
    qm31 x;
    if (kind == GKR_GRAND_PRODUCT) {
        // lane 0: d0 d1 = t0; lane 2: d20 d21 = t2
        const qm31 A = l0 ? d0 : (l2 ? d20 : qzero());
        const qm31 B = l0 ? d1 : d21;
        x = qmul(A, B);
    } else {
        const qm31 m = qadd(n, qmul(d, lambda));
        const qm31 m0 = quad_bcast_q<0>(m), m2 = quad_bcast_q<2>(m);
        const qm31 n1 = quad_bcast_q<1>(n), n3 = quad_bcast_q<3>(n);
        const qm31 m20 = qsub(qadd(m2, m2), m0), n21 = qsub(qadd(n3, n3), n1);
        const qm31 A = l0 ? d1 : (l1 ? d0 : (l2 ? d21 : d20));
        const qm31 B = l0 ? m0 : (l1 ? n1 : (l2 ? m20 : n21));
        x = qmul(A, B);
        x = qadd(x, gd_qperm<QP_ROT1>(x));
    }
    return (l0 || l2) ? qmul(e, x) : qzero();
}

// Where instance `in` reads round rho of layer L from: the stack layer (no fix yet this
// layer), or the fix scratch; `fix` = the previous round's variable is fixed on the fly.
struct GdSrc {
    bool fix;
    uint32_t kind;  // kind of the values this round sums over
    uint32_t src_kind;
    const uint32_t* num;
    const uint32_t* den;
};
__device__ __forceinline__ GdSrc gd_src(const GdInst& in, uint32_t onv, uint32_t L, uint32_t rho) {
    const uint32_t lv = onv + 1;
    const uint32_t fixes = rho - (L - onv);  // fixes done before this round's sums
    GdSrc s;
    s.fix = fixes >= 1;
    const bool from_stack = fixes <= 1;
    s.src_kind = from_stack ? in.kind[lv] : gd_fixed_kind(in.kind[lv]);
    s.kind = s.fix ? gd_fixed_kind(s.src_kind) : s.src_kind;
    s.num = from_stack ? in.num[lv] : in.scr_num;
    s.den = from_stack ? in.den[lv] : in.scr_den;
    return s;
}

// Round start: the previous round's pending claim update (sc_claim_i = rp_i(r) and, for the
// instances summed in that round, corr_i *= eq(r, y_rho)), then the finishing coefficients
// of this round.  With y0 = s0 corr F0, y2 = s2 corr F2 and
// y1 = claim - y0, the round polynomial's coefficient q of an instance summed in the round is
// y0 for q = 0 and b1 y0 + b2 y1 + b3 y2 = (b1 - b2) y0 + b2 claim + b3 y2 for q = 1..3 (basis
// rows b of the round), so A, B, C depend only on values known before the sums: the claim times
// the round's B factor, the correction times its A and C factors (gd_begin).  One full
// wave; lanes 0..31 take the claims, 32..63 the corrections, lane l of each half instance l>>2,
// coefficient l&3: four dependent products.
__device__ __forceinline__ void gd_round_prep(GdState* S, const GdInst* I, uint32_t n_inst, uint32_t n_layers,
                                              uint32_t L, uint32_t rho) {
    const uint32_t t = threadIdx.x & 63;
    const uint32_t i = (t & 31) >> 2, q = t & 3;
    const bool cor = t >= 32, in_range = i < n_inst;
    // this lane's claim or correction
    uint32_t* own = cor ? S->corr[in_range ? i : 0] : S->sc_claim[in_range ? i : 0];
    qm31 val = qload(own);
    const uint32_t(*pr)[4][4] = S->pre[rho];
    const qm31 f1 = qload(pr[cor ? 0 : 1][q]), f2 = qload(pr[2][q]);
    if (S->pend) {
        const qm31 r = qload(S->r);
        const qm31 craw = qload(S->craw[in_range ? i : 0][q]), y = qload(S->ood[S->pend_rho]);
        const uint32_t fl = in_range ? S->pend_flags[i] : 0u;
        // claims: c1 r, r^2, c3 r in lanes 1, 2, 3; corrections: r y
        const qm31 m1 = qmul(cor ? y : (q == 2 ? r : craw), r);
        // eq(r, y) = r y + (1 - r)(1 - y) = 1 - r - y + 2 r y
        const qm31 e = qadd(qsub(qsub(qone(), r), y), qadd(m1, m1));
        // claims: rp(r) = (c0 + c1 r) + (c2 + c3 r) r^2; corrections: corr eq(r, y)
        const qm31 hi = qadd(quad_bcast_q<2>(craw), quad_bcast_q<3>(m1));
        const qm31 r2 = quad_bcast_q<2>(m1);
        const qm31 m2 = qmul(cor ? val : hi, cor ? e : r2);
        const qm31 lo = qadd(quad_bcast_q<0>(craw), quad_bcast_q<1>(m1));
        const bool upd = (fl & 1) && (!cor || (fl & 2));
        if (upd) {
            val = cor ? m2 : qadd(lo, m2);
            if (q == 0) gd_qstore(own, val);
        }
    }
    if (!in_range) return;
    const GdView vw = gd_view(I[i], n_layers, L);
    const bool act = vw.active, part = act && vw.onv >= L - rho;
    if (t < 32 && q == 0) S->rflags[i] = (act ? 1u : 0u) | (part ? 2u : 0u);
    if (!part) return;
    gd_qstore(S->fin[i][q][cor ? 0 : 1], qmul(val, f1));
    if (cor) gd_qstore(S->fin[i][q][2], qmul(val, f2));
}

// What the end of a round reads of the state, in LDS.
struct GdFin {
    uint32_t fin[GD_MAX_INST][4][3][4];
    uint32_t rflags[GD_MAX_INST];
    uint32_t alpha_pow[GD_MAX_INST][4];
    uint32_t sc_claim[GD_MAX_INST][4];
    uint32_t dg[8];
};

template <int N>
__device__ __forceinline__ qm31 gd_row_ror(qm31 v) {
    const auto f = [](uint32_t x) {
        return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x120 + N, 0xF, 0xF, false);
    };
    return {{f(v.c0.a), f(v.c0.b)}, {f(v.c1.a), f(v.c1.b)}};
}

// Turns the round sums (sums[8 i + c]: r(0) then r(2) coordinates before the eq
// correction, 64-bit) into the batched round polynomial, mixes it and draws the round
// challenge; the claim update is left pending.  Wave 0 only, with the previous round's
// update already applied; lane t handles instance t>>2, coefficient t&3.
__device__ __forceinline__ void gd_finish(GdState* S, const GdChan& C, const uint32_t (*fin)[4][3][4],
                                          const uint32_t* rflags, const uint32_t (*alpha_pow)[4],
                                          const uint32_t (*sc_claim)[4], const uint32_t* dg, uint32_t n_inst,
                                          uint32_t rho, const unsigned long long* sums, uint32_t* rec) {
    const uint32_t t = threadIdx.x;
    const uint32_t i = t >> 2, q = t & 3;
    uint32_t dv = dg[t & 7];
    qm31 craw = qzero(), cv = qzero();
    if (i < n_inst) {
        const uint32_t fl = rflags[i];  // set by gd_round_prep for this round
        const bool act = fl & 1, part = fl & 2;
        const qm31 ap = qload(alpha_pow[i]);
        if (part) {
            const unsigned long long* a = sums + 8 * i;
            const qm31 s0 = {{mred64(a[0]), mred64(a[1])}, {mred64(a[2]), mred64(a[3])}};
            const qm31 s2 = {{mred64(a[4]), mred64(a[5])}, {mred64(a[6]), mred64(a[7])}};
            craw = qadd(qadd(qmul(qload(fin[i][q][0]), s0), qmul(qload(fin[i][q][2]), s2)), qload(fin[i][q][1]));
        } else if (act && q == 0) {
            craw = qmulm(qload(sc_claim[i]), (P + 1) / 2);
        }
        cv = qmul(craw, ap);
    }
    // sum over the instances: lanes 4 and 8 apart within a row of 16, then the two rows
    cv = qadd(cv, gd_row_ror<8>(cv));
    cv = qadd(cv, gd_row_ror<4>(cv));
    if (n_inst > 4) cv = qadd(cv, gd_shfl_xor(cv, 16));
    const uint64_t nzmask = __ballot(t < 4 && !qiszero(cv)) & 0xFull;
    const uint32_t len = nzmask ? 64 - __clzll(nzmask) : 0;
    const uint32_t pv = i == 0 ? cv.c0.a : (i == 1 ? cv.c0.b : (i == 2 ? cv.c1.a : cv.c1.b));
    C.mix(dv, pv, 4 * len);
    uint32_t nd = 0, st = 0;
    const qm31 r = C.draw(dv, nd, st);
    if (t >= 16 && t < 24) S->dg[t & 7] = dv;
    if (t < 16) rec[1 + C.pay_index()] = pv;
    if (t == 0) {
        rec[0] = len;
        S->n_draws = nd;
        if (st) S->status = 1;
        gd_qstore(S->r, r);
        gd_qstore(S->asg[rho], r);
        S->pend = 1;
        S->pend_rho = rho;
    }
    if (i < n_inst) {
        gd_qstore(S->craw[i][q], craw);
        if (q == 0) S->pend_flags[i] = rflags[i];
    }
}

// Layer begin (all threads of the block call it; it synchronises the block).
__device__ __forceinline__ void gd_begin(GdState* S, const GdInst* I, const GdChan& C, uint32_t n_inst,
                                         uint32_t n_layers, uint32_t L) {
    const uint32_t t = threadIdx.x;
    const uint32_t remaining = n_layers - L;
    if (t < 64) {
        uint32_t dv = S->dg[t & 7], nd = S->n_draws, st = 0;
        for (uint32_t i = 0; i < n_inst; i++) {
            if (!gd_view(I[i], n_layers, L).active) continue;
            const uint32_t nw = I[i].kind[0] == GKR_GRAND_PRODUCT ? 4 : 8;
            const bool fresh = I[i].n_vars == remaining;
            const uint32_t w = C.pay_index();
            uint32_t pv = 0;
            if (w < 8) {
                pv = fresh ? (&S->outputs[i][0][0])[w] : (&S->claims[i][0][0])[w];
                if (fresh && t < 16) (&S->claims[i][0][0])[w] = pv;
            }
            C.mix(dv, w < nw ? pv : 0u, nw);
            nd = 0;
        }
        const qm31 alpha = C.draw(dv, nd, st);
        const qm31 lambda = C.draw(dv, nd, st);
        if (t >= 16 && t < 24) S->dg[t & 7] = dv;
        if (t == 0) {
            S->n_draws = nd;
            if (st) S->status = 1;
            S->pend = 0;
            gd_qstore(S->lambda, lambda);
            // the batch combines the active instances only, in order (sumcheck.zig:215-238)
            qm31 ap = qone();
            for (uint32_t i = 0; i < n_inst; i++) {
                const bool a = gd_view(I[i], n_layers, L).active;
                gd_qstore(S->alpha_pow[i], a ? ap : qzero());
                if (a) ap = qmul(ap, alpha);
            }
        }
    } else if (t < 256) {
        // round rho's constants from y = ood[0..L), L < 64: the prefix products by a scan, then wave
        // q = 1..3 the factors of coefficient q (the first also those of coefficient 0)
        const uint32_t rho = t & 63, q = t >> 6;
        qm31 pp = rho < L ? qsub(qone(), qload(S->ood[rho])) : qone();
        for (uint32_t d = 1; d < L; d <<= 1) {
            const qm31 o = gd_shfl(pp, (int)(rho - d));
            if (rho >= d) pp = qmul(pp, o);
        }
        if (rho < L) {
            const qm31 y = qload(S->ood[rho]);
            const qm31 dd = qsub(qone(), qadd(y, y));
            const qm31 pd = qmul(pp, dd);
            const qm31 ipd = qinv(pd);
            const qm31 ipp = qmul(ipd, dd), idd = qmul(ipd, pp);
            const qm31 one = qone(), two = qfromm(2), three = qfromm(3);
            const qm31 b = qmul(qsub(one, y), idd);
            const qm31 bm1 = qsub(b, one), tmb = qsub(two, b);
            const qm31 qq = qmul(qmul(b, bm1), tmb);
            const qm31 iq = qinv(qq);
            const qm31 ib = qmul(qmul(bm1, tmb), iq), ibm1 = qmul(qmul(b, tmb), iq), itmb = qmul(qmul(b, bm1), iq);
            const uint32_t inv2 = (P + 1) / 2;
            const qm31 s0 = qneg(qmulm(ib, inv2)), s1 = ibm1, s2 = qmulm(itmb, inv2);
            const qm31 F0 = qmul(qsub(one, y), ipp);                // (1-y) / prefix
            const qm31 F2 = qmul(qsub(qmul(three, y), one), ipp);  // eq(2, y) / prefix
            // basis row of x^q: s0 u0, s1 u1, s2 u2
            qm31 u0 = one, u1 = one, u2 = one;
            if (q == 1) u0 = qadd(two, qmulm(b, 3)), u1 = qadd(b, b), u2 = b;
            if (q == 2) u0 = qneg(qadd(three, b)), u1 = qneg(qadd(two, b)), u2 = qneg(qadd(one, b));
            const qm31 b1 = qmul(s0, u0), b2 = qmul(s1, u1), b3 = qmul(s2, u2);
            uint32_t(*pr)[4][4] = S->pre[rho];
            gd_qstore(pr[0][q], qmul(qsub(b1, b2), F0));
            gd_qstore(pr[1][q], b2);
            gd_qstore(pr[2][q], qmul(b3, F2));
            if (q == 1) {
                gd_qstore(pr[0][0], F0);
                gd_qstore(pr[1][0], qzero());
                gd_qstore(pr[2][0], qzero());
                if (qiszero(pd) || qiszero(qq)) S->status = 2;
            }
        }
    }
    __syncthreads();
    if (t < n_inst) {
        const GdView v = gd_view(I[t], n_layers, L);
        if (v.active) {
            const uint32_t nc = I[t].kind[0] == GKR_GRAND_PRODUCT ? 1 : 2;
            const qm31 lambda = qload(S->lambda);
            qm31 cl = qzero();
            for (uint32_t c = nc; c > 0; c--) cl = qadd(qmul(cl, lambda), qload(S->claims[t][c - 1]));
            gd_qstore(S->sc_claim[t], qmulm(cl, 1u << (L - v.onv)));
            gd_qstore(S->corr[t], qone());
        }
    }
    __syncthreads();
}

// eq table of layer L: eq[i] = (1 - y_0) prod_{j < L-1} (bit_{L-2-j}(i) ? y_{j+1} : 1 - y_{j+1})
// (EqEvals.generate(ood) = genEqEvals(ood[1..], 1 - ood[0]), gkr_circuit.zig:651-674).
__device__ __forceinline__ void gd_eq_entry(const GdState* S, uint32_t L, uint64_t i, uint32_t* eq) {
    qm31 acc = qsub(qone(), qload(S->ood[0]));
    for (uint32_t j = 0; j + 1 < L; j++) {
        const qm31 y = qload(S->ood[j + 1]);
        acc = qmul(acc, ((i >> (L - 2 - j)) & 1) ? y : qsub(qone(), y));
    }
    gd_st(eq, i, acc);
}

// Layer end: masks of every active instance, mixed in order; challenge; next claims and
// eq point (gkr_prover.zig:232-276, gkr_circuit.zig:341-388).
__device__ __forceinline__ void gd_end(GdState* S, const GdInst* I, const GdChan& C, uint32_t n_inst,
                                       uint32_t n_layers, uint32_t L, uint32_t* rec_mask) {
    const uint32_t t = threadIdx.x;
    if (t < n_inst) {
        const GdView v = gd_view(I[t], n_layers, L);
        if (v.active) {
            const GdInst& in = I[t];
            const uint32_t lv = v.onv + 1;
            qm31 n0, n1, d0, d1;
            if (v.onv == 0) {
                const uint32_t k = in.kind[lv];
                d0 = gd_ld(in.den[lv], 0);
                d1 = gd_ld(in.den[lv], 1);
                n0 = k == GKR_GRAND_PRODUCT ? qzero() : gd_num(k, in.num[lv], 0);
                n1 = k == GKR_GRAND_PRODUCT ? qzero() : gd_num(k, in.num[lv], 1);
            } else {
                const qm31 r = qload(S->r);
                const bool stack = v.onv == 1;
                const uint32_t k = stack ? in.kind[lv] : gd_fixed_kind(in.kind[lv]);
                const uint32_t* dn = stack ? in.den[lv] : in.scr_den;
                const uint32_t* nn = stack ? in.num[lv] : in.scr_num;
                qm31 a = gd_ld(dn, 0), b = gd_ld(dn, 2);
                d0 = qadd(qmul(r, qsub(b, a)), a);
                a = gd_ld(dn, 1), b = gd_ld(dn, 3);
                d1 = qadd(qmul(r, qsub(b, a)), a);
                if (gd_has_num(k)) {
                    a = gd_num(k, nn, 0), b = gd_num(k, nn, 2);
                    n0 = qadd(qmul(r, qsub(b, a)), a);
                    a = gd_num(k, nn, 1), b = gd_num(k, nn, 3);
                    n1 = qadd(qmul(r, qsub(b, a)), a);
                } else {
                    n0 = k == GKR_GRAND_PRODUCT ? qzero() : qone();
                    n1 = n0;
                }
            }
            gd_qstore(S->mask[t][0], n0);
            gd_qstore(S->mask[t][1], n1);
            gd_qstore(S->mask[t][2], d0);
            gd_qstore(S->mask[t][3], d1);
            uint32_t* rm = rec_mask + (uint64_t)t * GD_REC_MASK;
            gd_qstore(rm, n0);
            gd_qstore(rm + 4, n1);
            gd_qstore(rm + 8, d0);
            gd_qstore(rm + 12, d1);
        }
    }
    __syncthreads();
    if (t < 64) {
        uint32_t dv = S->dg[t & 7], nd = S->n_draws, st = 0;
        for (uint32_t i = 0; i < n_inst; i++) {
            if (!gd_view(I[i], n_layers, L).active) continue;
            const bool gp = I[i].kind[0] == GKR_GRAND_PRODUCT;
            const uint32_t w = C.pay_index();
            const uint32_t pv = t < 16 && (!gp || w < 8) ? (&S->mask[i][gp ? 2 : 0][0])[w] : 0u;
            C.mix(dv, pv, gp ? 8 : 16);
            nd = 0;
        }
        const qm31 ch = C.draw(dv, nd, st);
        if (t >= 16 && t < 24) S->dg[t & 7] = dv;
        // next claims: lane 2 i + c for column c of instance i
        if (t < 2 * n_inst) {
            const uint32_t i = t >> 1, c = t & 1;
            const bool gp = I[i].kind[0] == GKR_GRAND_PRODUCT;
            if (gd_view(I[i], n_layers, L).active && !(gp && c)) {
                const uint32_t col = gp ? 1 : c;  // mask column: den (GP) or num, den
                const qm31 m0 = qload(S->mask[i][2 * col]), m1 = qload(S->mask[i][2 * col + 1]);
                gd_qstore(S->claims[i][c], qadd(qmul(ch, qsub(m1, m0)), m0));
            }
        }
        if (t < L)
            for (int k = 0; k < 4; k++) S->ood[t][k] = S->asg[t][k];
        if (t == 0) {
            S->n_draws = nd;
            if (st) S->status = 1;
            S->pend = 0;  // the last round's claim update is not needed: the claims come from the masks
            gd_qstore(S->ood[L], ch);
        }
    }
    __syncthreads();
}

// One workgroup: whole layers [L0, L1), the first one starting at round rho0 (its begin
// already done when rho0 > 0); every layer ends here.  The state lives in LDS meanwhile.
__global__ __launch_bounds__(GD_FT) void gkr_fused_kernel(GdState* __restrict__ gS, const GdInst* __restrict__ gI,
                                                          uint32_t n_inst, uint32_t n_layers, uint32_t L0, uint32_t L1,
                                                          uint32_t rho0, uint32_t* __restrict__ eq,
                                                          uint32_t* __restrict__ rec) {
    __shared__ GdState S;
    __shared__ GdInst I[GD_MAX_INST];
    __shared__ __align__(16) uint32_t boards[GD_CHAN_WORDS];
    // round records, written out at the end: a store of the first wave in a round's finish would
    // hold up its loads of the next round
    __shared__ uint32_t recs[GD_FUSED_ROUNDS * GD_REC_ROUND];
    // round sums, double-buffered by round parity: the pending-update wave clears the other
    // buffer while a round accumulates into its own (LDS atomics, one add per term and word)
    __shared__ unsigned long long red[2][GD_MAX_INST][8];
    const uint32_t t = threadIdx.x;
    const uint32_t wv = t >> 6, ln = t & 63;
    {
        const uint64_t* src = (const uint64_t*)gS;
        uint64_t* dst = (uint64_t*)&S;
        for (uint32_t k = t; k < sizeof(GdState) / 8; k += GD_FT) dst[k] = src[k];
        for (uint32_t k = t; k < 2 * GD_MAX_INST * 8; k += GD_FT) (&red[0][0][0])[k] = 0;
        const uint64_t* is = (const uint64_t*)gI;
        for (uint32_t k = t; k < n_inst * (sizeof(GdInst) / 8); k += GD_FT) ((uint64_t*)I)[k] = is[k];
    }
    const GdChan C(boards, t);
    __syncthreads();
    if (L0 == 0 && rho0 == 0 && t < n_inst) {
        // output layer (gkr_circuit.zig:162-190)
        const GdInst& in = I[t];
        const qm31 d = gd_ld(in.den[0], 0);
        if (in.kind[0] == GKR_GRAND_PRODUCT) {
            gd_qstore(S.outputs[t][0], d);
        } else {
            gd_qstore(S.outputs[t][0], gd_num(in.kind[0], in.num[0], 0));
            gd_qstore(S.outputs[t][1], d);
        }
    }
    __syncthreads();
    const uint32_t total_rounds = n_layers * (n_layers - 1) / 2;
    uint32_t rc = 0;  // rounds run by this launch (sum buffer parity)
    for (uint32_t L = L0; L < L1; L++) {
        const uint32_t rb = L == L0 ? rho0 : 0;
        if (rb == 0) {
            gd_begin(&S, I, C, n_inst, n_layers, L);
            if (L >= 1)
                for (uint32_t k = t; k < (1u << (L - 1)); k += GD_FT) gd_eq_entry(&S, L, k, eq);
            __syncthreads();
        }
        for (uint32_t rho = rb; rho < L; rho++, rc++) {
            const uint32_t rem = L - rho;
            const uint64_t nt = 1ull << (rem - 1);
            const uint32_t b = rc & 1;
            if (wv == 7) {
                gd_round_prep(&S, I, n_inst, n_layers, L, rho);
                (&red[b ^ 1][0][0])[ln] = 0;
            } else {
                // (instance, term) pairs over the 112 quads of waves 0..6; pair x = p * nt + k for
                // the p-th instance summed in this round
                const qm31 lambda = qload(S.lambda), r = qload(S.r);
                uint32_t n_part = 0;
                for (uint32_t i = 0; i < n_inst; i++) {
                    const GdView v = gd_view(I[i], n_layers, L);
                    n_part += v.active && v.onv >= rem;
                }
                const uint32_t j = t & 3;
                for (uint64_t x = t >> 2; x < (uint64_t)n_part * nt; x += 7 * 16) {
                    const uint32_t p = (uint32_t)(x >> (rem - 1));
                    const uint64_t k = x & (nt - 1);
                    uint32_t i = 0;
                    for (uint32_t ii = 0, cnt = 0; ii < n_inst; ii++) {
                        const GdView v = gd_view(I[ii], n_layers, L);
                        if (!(v.active && v.onv >= rem)) continue;
                        if (cnt++ == p) {
                            i = ii;
                            break;
                        }
                    }
                    const GdView v = gd_view(I[i], n_layers, L);
                    const GdSrc s = gd_src(I[i], v.onv, L, rho);
                    const qm31 y = gd_term_quad(s.fix, s.src_kind, s.num, s.den, I[i].scr_num, I[i].scr_den, r, nt, k,
                                                lambda, eq, j);
                    if (j == 0 || j == 2) {
                        unsigned long long* dst = &red[b][i][j == 0 ? 0 : 4];
                        atomicAdd(dst + 0, (unsigned long long)y.c0.a);
                        atomicAdd(dst + 1, (unsigned long long)y.c0.b);
                        atomicAdd(dst + 2, (unsigned long long)y.c1.a);
                        atomicAdd(dst + 3, (unsigned long long)y.c1.b);
                    }
                }
            }
            __syncthreads();
            if (t < 64)
                gd_finish(&S, C, S.fin, S.rflags, S.alpha_pow, S.sc_claim, S.dg, n_inst, rho, &red[b][0][0],
                          recs + rc * GD_REC_ROUND);
            __syncthreads();
        }
        gd_end(&S, I, C, n_inst, n_layers, L,
               rec + (uint64_t)total_rounds * GD_REC_ROUND + (uint64_t)L * n_inst * GD_REC_MASK);
    }
    {
        uint32_t* out = rec + (uint64_t)(L0 * (L0 - 1) / 2 + rho0) * GD_REC_ROUND;  // consecutive rounds
        for (uint32_t k = t; k < rc * GD_REC_ROUND; k += GD_FT) out[k] = recs[k];
        const uint64_t* src = (const uint64_t*)&S;
        uint64_t* dst = (uint64_t*)gS;
        for (uint32_t k = t; k < sizeof(GdState) / 8; k += GD_FT) dst[k] = src[k];
    }
}

// Layer begin of a large layer plus its eq table over many workgroups (block 0 also runs the begin).
__global__ __launch_bounds__(GD_RT) void gkr_begin_eq_kernel(GdState* __restrict__ S, const GdInst* __restrict__ I,
                                                             uint32_t n_inst, uint32_t n_layers, uint32_t L,
                                                             uint32_t* __restrict__ eq) {
    const uint64_t k = (uint64_t)blockIdx.x * GD_RT + threadIdx.x;
    if (L >= 1 && k < (1ull << (L - 1))) gd_eq_entry(S, L, k, eq);
    if (blockIdx.x == 0) {
        __shared__ __align__(16) uint32_t boards[GD_CHAN_WORDS];
        const GdChan C(boards, threadIdx.x);
        __syncthreads();
        gd_begin(S, I, C, n_inst, n_layers, L);
    }
}

// One large sum-check round: grid (x: terms, y: instance).  Every workgroup stores its
// sums in its own slot of `part` and counts itself done on one of 16 sub-counters (separate
// cache lines; the workgroup completing a sub-counter counts on the top counter), so no
// address takes more than ~nb/16 atomics; the last workgroup adds the slots up and finishes
// the round.  Workgroup (x = last, y = 0) sums nothing: it applies the previous round's pending
// claim update and sets this round's finishing coefficients (gd_round_prep) while the others
// sum; the release fence before its count (the only one) publishes them to the last workgroup.
__global__ __launch_bounds__(GD_RT) void gkr_round_kernel(GdState* __restrict__ S, const GdInst* __restrict__ I,
                                                          uint32_t n_inst, uint32_t n_layers, uint32_t L, uint32_t rho,
                                                          const uint32_t* __restrict__ eq, uint32_t* __restrict__ rec,
                                                          unsigned long long* __restrict__ part, uint32_t* __restrict__ cnt) {
    __shared__ unsigned long long red[GD_RT / 64][8];
    __shared__ unsigned long long sums[GD_MAX_INST][8], rows[GD_MAX_INST][GD_RT / 64][8];
    __shared__ __align__(16) uint32_t boards[GD_CHAN_WORDS];
    __shared__ GdFin F;
    __shared__ uint32_t last;
    const uint32_t t = threadIdx.x;
    const uint32_t rem = L - rho;
    const uint64_t nt = 1ull << (rem - 1);
    // blockIdx.y = rank among the instances summed in this round
    uint32_t i = 0;
    for (uint32_t ii = 0, cnt_p = 0; ii < n_inst; ii++) {
        const GdView vi = gd_view(I[ii], n_layers, L);
        if (!(vi.active && vi.onv >= rem)) continue;
        if (cnt_p++ == blockIdx.y) {
            i = ii;
            break;
        }
    }
    // the last workgroup column runs the round-start prep (instance row 0) instead of sums, so
    // the prep overlaps the sums rather than delaying one summing workgroup
    const uint32_t nsb = gridDim.x - 1;
    const bool prep_blk = blockIdx.x == nsb;
    if (prep_blk && blockIdx.y == 0 && t < 64) gd_round_prep(S, I, n_inst, n_layers, L, rho);
    const GdView v = gd_view(I[i], n_layers, L);
    uint64_t a[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (!prep_blk) {
        const GdSrc s = gd_src(I[i], v.onv, L, rho);
        const qm31 lambda = qload(S->lambda), r = qload(S->r);
        const uint32_t j = t & 3;
        for (uint64_t k = (uint64_t)blockIdx.x * (GD_RT / 4) + (t >> 2); k < nt; k += (uint64_t)nsb * (GD_RT / 4)) {
            const qm31 y = gd_term_quad(s.fix, s.src_kind, s.num, s.den, I[i].scr_num, I[i].scr_den, r, nt, k, lambda,
                                        eq, j);
            if (j == 0) {
                a[0] += y.c0.a, a[1] += y.c0.b, a[2] += y.c1.a, a[3] += y.c1.b;
            } else if (j == 2) {
                a[4] += y.c0.a, a[5] += y.c0.b, a[6] += y.c1.a, a[7] += y.c1.b;
            }
        }
    }
    {
        const uint64_t w = gd_wave_sum8(a, t & 63);
        if ((t & 7) == 0) red[t >> 6][(t & 63) >> 3] = w;
    }
    __syncthreads();
    // The slot is written with device-coherent stores (agent-scope atomic stores) by wave 0,
    // which waits for their acknowledgement before thread 0 counts the workgroup: no L2
    // writeback per workgroup.  The prep workgroup wrote the state with plain stores and
    // publishes it with one release; the last workgroup acquires.
    if (t < 8) {
        uint64_t w = 0;
        for (uint32_t k = 0; k < GD_RT / 64; k++) w += red[k][t];
        __hip_atomic_store(&part[((uint64_t)blockIdx.y * gridDim.x + blockIdx.x) * 8 + t], (unsigned long long)w,
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (t < 64) {
        __builtin_amdgcn_s_waitcnt(0);
        if (t == 0) {
            if (prep_blk && blockIdx.y == 0) __threadfence();
            const uint32_t nb = gridDim.x * gridDim.y, b = blockIdx.y * gridDim.x + blockIdx.x;
            const uint32_t g = b % GD_CNT_GROUPS, ng = nb < GD_CNT_GROUPS ? nb : GD_CNT_GROUPS;
            const uint32_t gsize = (nb - g + GD_CNT_GROUPS - 1) / GD_CNT_GROUPS;
            uint32_t lst = 0;
            if (atomicAdd(&cnt[GD_CNT_STRIDE * g], 1u) == gsize - 1)
                lst = atomicAdd(&cnt[GD_CNT_STRIDE * GD_CNT_GROUPS], 1u) == ng - 1 ? 1u : 0u;
            last = lst;
        }
    }
    __syncthreads();
    if (!last) return;
    // acquire: the slots came with device-coherent stores and the prep's state with its
    // workgroup's release; this workgroup has nothing of its own to write back
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    if (t <= GD_CNT_GROUPS) atomicExch(&cnt[GD_CNT_STRIDE * t], 0u);
    // the state the finish reads, and the slots of every summed instance, in one round trip: the
    // waves share the rows
    const GdChan C(boards, t);
    for (uint32_t k = t; k < 48 * n_inst; k += GD_RT) (&F.fin[0][0][0][0])[k] = (&S->fin[0][0][0][0])[k];
    if (t < 4 * n_inst) {
        (&F.alpha_pow[0][0])[t] = (&S->alpha_pow[0][0])[t];
        (&F.sc_claim[0][0])[t] = (&S->sc_claim[0][0])[t];
    }
    if (t < n_inst) F.rflags[t] = S->rflags[t];
    if (t < 8) F.dg[t] = S->dg[t];
    const uint32_t n_rows = gridDim.y, wpr = n_rows >= 3 ? 1 : (n_rows == 2 ? 2 : 4), wv = t >> 6;
    for (uint32_t row = wv / wpr; row < n_rows; row += 4 / wpr) {
        uint64_t b8[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        for (uint32_t x = (wv % wpr) * 64 + (t & 63); x < gridDim.x; x += 64 * wpr) {
            unsigned long long* pp = part + ((uint64_t)row * gridDim.x + x) * 8;
#pragma unroll
            for (int c = 0; c < 8; c++) b8[c] += __hip_atomic_load(&pp[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        const uint64_t w = gd_wave_sum8(b8, t & 63);
        if ((t & 7) == 0) rows[row][wv % wpr][(t & 63) >> 3] = w;
    }
    __syncthreads();
    if (t >= 64) return;
    if (t < 8 * n_inst) {
        // instance t / 8 is the row of its rank among the summed ones
        uint32_t row = 0;
        for (uint32_t ii = 0; ii < (t >> 3); ii++) row += (F.rflags[ii] >> 1) & 1;
        uint64_t w = 0;
        if (F.rflags[t >> 3] & 2)
            for (uint32_t k = 0; k < wpr; k++) w += rows[row][k][t & 7];
        sums[t >> 3][t & 7] = w;
    }
    qboard_wave_fence();
    gd_finish(S, C, F.fin, F.rflags, F.alpha_pow, F.sc_claim, F.dg, n_inst, rho, &sums[0][0],
              rec + (uint64_t)(L * (L - 1) / 2 + rho) * GD_REC_ROUND);
}

}  // namespace

// The state starts from a device channel (every other word zero) and hands its digest and
// draw counter back at the end; a failed draw or a zero division sets the channel status.
__global__ void gkr_chan_in_kernel(GdState* __restrict__ S, const DevChannel* __restrict__ ch) {
    uint32_t* w = (uint32_t*)S;
    constexpr uint32_t NW = sizeof(GdState) / 4;
    for (uint32_t i = threadIdx.x; i < NW; i += blockDim.x) {
        uint32_t v = 0;
        if (i < 8) v = ch->digest[i];
        else if (i == 8) v = ch->n_draws;
        w[i] = v;
    }
}
__global__ void gkr_chan_out_kernel(DevChannel* __restrict__ ch, const GdState* __restrict__ S) {
    const uint32_t t = threadIdx.x;
    if (t < 8) ch->digest[t] = S->dg[t];
    if (t == 8) ch->n_draws = S->n_draws;
    if (t == 9 && S->status != 0) ch->status = S->status;
}

struct GkrRun {
    std::vector<GkrInstance> inst;
    uint32_t n_inst = 0, n_layers = 0;
    uint64_t rec_words = 0;
    std::vector<DBuf> bufs;
    DBuf d_inst, d_state, d_rec, d_eq, d_part, d_cnt;
};

GkrRun* gkr_launch_on_channel(Ctx& c, DevChannel* d_ch, const std::vector<GkrInstance>& inst) {
    SR_CHECK(d_ch, "gkr: device channel");
    SR_CHECK(!inst.empty(), "gkr: empty batch");
    SR_CHECK(inst.size() <= GD_MAX_INST, "gkr: at most 8 instances per batch");
    std::unique_ptr<GkrRun> run(new GkrRun());
    run->inst = inst;
    const uint32_t n_inst = (uint32_t)inst.size();
    uint32_t n_layers = 0;
    for (auto& in : inst) {
        SR_CHECK(in.kind >= 0 && in.kind <= 3, "gkr: layer kind");
        SR_CHECK(in.n_vars >= 1 && in.n_vars <= GD_MAX_VARS, "gkr: an instance needs 1..30 variables");
        SR_CHECK(in.d_den && (in.kind == GKR_GRAND_PRODUCT || in.kind == GKR_LOGUP_SINGLES || in.d_num),
                 "gkr: missing layer columns");
        n_layers = std::max(n_layers, in.n_vars);
    }
    run->n_inst = n_inst;
    run->n_layers = n_layers;
    // Layer stacks (buildLayers, gkr_circuit.zig:431-447) and fix scratch.
    std::vector<GdInst> h_inst(n_inst);
    std::vector<DBuf>& bufs = run->bufs;
    for (uint32_t k = 0; k < n_inst; k++) {
        GdInst& g = h_inst[k];
        memset(&g, 0, sizeof(g));
        const uint32_t nv = inst[k].n_vars;
        const bool gp = inst[k].kind == GKR_GRAND_PRODUCT;
        g.n_vars = nv;
        for (uint32_t l = 0; l < nv; l++) g.kind[l] = gp ? GKR_GRAND_PRODUCT : GKR_LOGUP_GENERIC;
        g.kind[nv] = (uint32_t)inst[k].kind;
        g.num[nv] = inst[k].d_num;
        g.den[nv] = inst[k].d_den;
        for (uint32_t l = 0; l < nv; l++) {
            if (!gp) {
                bufs.emplace_back(&c, 16ull << l);
                g.num[l] = bufs.back().as<uint32_t>();
            }
            bufs.emplace_back(&c, 16ull << l);
            g.den[l] = bufs.back().as<uint32_t>();
        }
        for (int32_t l = (int32_t)nv - 1; l >= 0; l--)
            launch_gkr_next_layer(c, (int)g.kind[l + 1], g.num[l + 1], g.den[l + 1], (uint32_t)l + 1,
                                  (uint32_t*)g.num[l], (uint32_t*)g.den[l]);
        bufs.emplace_back(&c, 16ull << (nv - 1));
        g.scr_den = bufs.back().as<uint32_t>();
        // every LogUp stack layer below the input is generic (QM31 numerators), singles included
        if (!gp) {
            bufs.emplace_back(&c, 16ull << (nv - 1));
            g.scr_num = bufs.back().as<uint32_t>();
        }
    }
    run->d_inst = upload(c, h_inst.data(), h_inst.size());
    run->d_state = DBuf(&c, sizeof(GdState));
    hipLaunchKernelGGL(gkr_chan_in_kernel, dim3(1), dim3(256), 0, c.stream, run->d_state.as<GdState>(),
                       (const DevChannel*)d_ch);
    SR_HIP(hipGetLastError());
    const uint32_t total_rounds = n_layers * (n_layers - 1) / 2;
    run->rec_words = (uint64_t)total_rounds * GD_REC_ROUND + (uint64_t)n_layers * n_inst * GD_REC_MASK;
    run->d_rec = DBuf(&c, 4 * run->rec_words);
    run->d_eq = DBuf(&c, n_layers >= 2 ? (16ull << (n_layers - 2)) : 16);
    run->d_part = DBuf(&c, 64ull * n_inst * GD_MAX_BX);
    run->d_cnt = DBuf(&c, 4ull * GD_CNT_STRIDE * (GD_CNT_GROUPS + 1));
    launch_fill_u32(c, run->d_cnt.as<uint32_t>(), GD_CNT_STRIDE * (GD_CNT_GROUPS + 1), 0);
    GdState* S = run->d_state.as<GdState>();
    const GdInst* I = run->d_inst.as<GdInst>();
    uint32_t* eq = run->d_eq.as<uint32_t>();
    uint32_t* rec = run->d_rec.as<uint32_t>();
    // the instances summed in round rho of layer L: active, with onv >= L - rho
    auto parts = [&](uint32_t L, uint32_t rho) {
        uint32_t n_part = 0;
        for (uint32_t k = 0; k < n_inst; k++)
            n_part += inst[k].n_vars + L >= n_layers && inst[k].n_vars + L - n_layers >= L - rho;
        return n_part;
    };
    // algorithmic bytes of one sum-check round: 96 B per term (four values read, two fixed
    // values written, one eq entry) for every instance summed in it
    auto round_bytes = [&](uint32_t L, uint32_t rho) {
        return 96.0 * (double)(1ull << (L - rho - 1)) * parts(L, rho);
    };
    // first round of layer L from which every round is a one-workgroup one
    auto first_small = [&](uint32_t L) {
        uint32_t rho = L;
        while (rho > 0 && ((uint64_t)parts(L, rho - 1) << (L - rho)) <= GD_SMALL_TERMS) rho--;
        return rho;
    };
    uint32_t n_small = 0;  // layers below run whole in one workgroup
    while (n_small < n_layers && first_small(n_small) == 0) n_small++;
    SR_CHECK(n_small * (n_small ? n_small - 1 : 0) / 2 <= GD_FUSED_ROUNDS, "gkr: rounds of one launch");
    {
        double bytes = 0;
        for (uint32_t L = 1; L < n_small; L++)
            for (uint32_t rho = 0; rho < L; rho++) bytes += round_bytes(L, rho);
        KTimer kt(c, "gkr_small_layers", bytes);
        hipLaunchKernelGGL(gkr_fused_kernel, dim3(1), dim3(GD_FT), 0, c.stream, S, I, n_inst, n_layers, 0u, n_small, 0u,
                           eq, rec);
        SR_HIP(hipGetLastError());
    }
    for (uint32_t L = n_small; L < n_layers; L++) {
        // > 0: the instances of a round depend on rho alone, so its terms double from one layer to the next,
        // and a layer after the first one with a large round has one too
        const uint32_t small = first_small(L);
        SR_CHECK(small > 0 && L - small <= GD_FUSED_ROUNDS, "gkr: rounds of one launch");
        {
            KTimer kt(c, "gkr_begin_eq", 16.0 * (double)(1ull << (L - 1)));
            const uint64_t blocks = ((1ull << (L - 1)) + GD_RT - 1) / GD_RT;
            hipLaunchKernelGGL(gkr_begin_eq_kernel, dim3((uint32_t)blocks), dim3(GD_RT), 0, c.stream, S, I, n_inst,
                               n_layers, L, eq);
            SR_HIP(hipGetLastError());
        }
        for (uint32_t rho = 0; rho < small; rho++) {
            const uint64_t nt = 1ull << (L - rho - 1);
            // summing workgroups per instance, plus one column for the round-start prep
            const uint64_t bx = std::min<uint64_t>((nt + GD_RT / 4 - 1) / (GD_RT / 4), GD_MAX_BX - 1) + 1;
            KTimer kt(c, "gkr_round", round_bytes(L, rho));
            hipLaunchKernelGGL(gkr_round_kernel, dim3((uint32_t)bx, parts(L, rho)), dim3(GD_RT), 0, c.stream, S, I,
                               n_inst, n_layers, L, rho, (const uint32_t*)eq, rec,
                               run->d_part.as<unsigned long long>(), run->d_cnt.as<uint32_t>());
            SR_HIP(hipGetLastError());
        }
        double bytes = 0;
        for (uint32_t r2 = small; r2 < L; r2++) bytes += round_bytes(L, r2);
        KTimer kt(c, "gkr_small_rounds", bytes);
        hipLaunchKernelGGL(gkr_fused_kernel, dim3(1), dim3(GD_FT), 0, c.stream, S, I, n_inst, n_layers, L, L + 1, small,
                           eq, rec);
        SR_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(gkr_chan_out_kernel, dim3(1), dim3(64), 0, c.stream, d_ch, (const GdState*)S);
    SR_HIP(hipGetLastError());
    return run.release();
}

void gkr_release(GkrRun* run) { delete run; }

// Reads the proof back (one synchronisation) and assembles the word stream; ch_out (optional)
// receives the final channel state.
static std::vector<uint32_t> gkr_collect_into(Ctx& c, GkrRun* run, Channel* ch_out) {
    std::unique_ptr<GkrRun> own(run);
    const std::vector<GkrInstance>& inst = run->inst;
    const uint32_t n_inst = run->n_inst, n_layers = run->n_layers;
    const uint32_t total_rounds = n_layers * (n_layers - 1) / 2;
    std::vector<uint32_t> hrec(run->rec_words);
    GdState* hs = (GdState*)c.pinned(sizeof(GdState));
    SR_HIP(hipMemcpyAsync(hs, run->d_state.p, sizeof(GdState), hipMemcpyDeviceToHost, c.stream));
    SR_HIP(hipMemcpyAsync(hrec.data(), run->d_rec.p, 4 * run->rec_words, hipMemcpyDeviceToHost, c.stream));
    c.sync();
    SR_CHECK(hs->status != 1, "gkr: channel draw rejected 64 times");
    SR_CHECK(hs->status == 0, "gkr: division by zero in a round polynomial");
    // Assemble the proof word stream.
    std::vector<uint32_t> w;
    auto ncols = [&](uint32_t k) { return inst[k].kind == GKR_GRAND_PRODUCT ? 1u : 2u; };
    for (uint32_t L = 0; L < n_layers; L++) {
        w.push_back(L);
        for (uint32_t rho = 0; rho < L; rho++) {
            const uint32_t* rr = &hrec[(uint64_t)(L * (L - 1) / 2 + rho) * GD_REC_ROUND];
            SR_CHECK(rr[0] <= 4, "gkr: round record");
            w.push_back(rr[0]);
            w.insert(w.end(), rr + 1, rr + 1 + 4 * rr[0]);
        }
        uint32_t n_act = 0;
        for (uint32_t k = 0; k < n_inst; k++) n_act += inst[k].n_vars + L >= n_layers;
        w.push_back(n_act);
        for (uint32_t k = 0; k < n_inst; k++) {
            if (inst[k].n_vars + L < n_layers) continue;
            const uint32_t* rm = &hrec[(uint64_t)total_rounds * GD_REC_ROUND + ((uint64_t)L * n_inst + k) * GD_REC_MASK];
            w.push_back(k);
            w.push_back(ncols(k));
            if (ncols(k) == 1)
                w.insert(w.end(), rm + 8, rm + 16);
            else
                w.insert(w.end(), rm, rm + 16);
        }
    }
    for (uint32_t k = 0; k < n_inst; k++) {
        w.push_back(ncols(k));
        w.insert(w.end(), &hs->outputs[k][0][0], &hs->outputs[k][0][0] + 4 * ncols(k));
    }
    w.push_back(n_layers);
    w.insert(w.end(), &hs->ood[0][0], &hs->ood[0][0] + 4 * n_layers);
    for (uint32_t k = 0; k < n_inst; k++) {
        w.push_back(ncols(k));
        w.insert(w.end(), &hs->claims[k][0][0], &hs->claims[k][0][0] + 4 * ncols(k));
        w.push_back(inst[k].n_vars);
    }
    w.insert(w.end(), hs->dg, hs->dg + 8);
    if (ch_out) {
        memcpy(ch_out->digest, hs->dg, 32);
        ch_out->n_draws = hs->n_draws;
    }
    return w;
}

std::vector<uint32_t> gkr_collect(Ctx& c, GkrRun* run) { return gkr_collect_into(c, run, nullptr); }

std::vector<uint32_t> gkr_prove_batch(Ctx& c, Channel& ch, const std::vector<GkrInstance>& inst) {
    DBuf d_ch(&c, sizeof(DevChannel));
    DevChannel hc{};
    memcpy(hc.digest, ch.digest, 32);
    hc.n_draws = ch.n_draws;
    SR_HIP(hipMemcpyAsync(d_ch.p, c.stage(&hc, sizeof(hc)), sizeof(hc), hipMemcpyHostToDevice, c.stream));
    GkrRun* run = gkr_launch_on_channel(c, d_ch.as<DevChannel>(), inst);
    return gkr_collect_into(c, run, &ch);
}

}  // namespace sr
