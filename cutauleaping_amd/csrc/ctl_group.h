// ctl_group.h -- the group kernel: G lanes of a wavefront (G = 2..64, a
// power of two) cooperate on one simulation, for networks whose per-lane
// working set does not fit on chip.  Included by ctl_sim.hip.
//
// Work split: reaction j belongs to lane j mod G; species go to lanes in
// rounds of G, longest var/fear lists first (the round streams).  A group's
// simulation state lives in LDS for the whole launch:
//     X   int32 [2][S]   state and trial state (parity bit swaps them)
//     A   uint32[Rp]     propensity (FP32 bits) | critical flag << 31; zero
//                        past R (Rp = R + 1 rounded up to a multiple of G)
//     Kc  int32 [Rp]     counts drawn for the current leap attempt
//     Q   uint16[R]      reactions queued for a Poisson draw (lambda >= 1), in
//                        the trial-state half of X while it is free
//     F   uint32[2S+1]   reactant factors of the current state (reactions of
//                        at most two reactant entries of multiplicity <= 2):
//                        F[s] = x_s, F[S+s] = x_s (x_s - 1) / 2 as FP32 bits,
//                        each with its criticality in bit 31, F[2S] = 1.0; in
//                        the Kc region, which is free outside the leap's
//                        count and update phases
// so every table-driven access is an LDS access instead of a dependent HBM
// load.  Group-wide values (a0, tau, the chosen reaction) are computed with
// DPP row operations and lane reads and are identical in every lane of the
// group, so the group's control flow is uniform.
//
// Two widths: G is the algorithm's (whose partial sums and lane streams fix a
// trajectory's bits), W >= G the lanes that execute one simulation.  With
// W > G, lane l stands for the algorithm's lane l mod G (W / G lanes hold the
// same partial sums and streams); the work whose result does not depend on the
// lane that does it -- a reaction's propensity, a species' tau' and update, a
// queued Poisson draw, a sample, a dependent -- is spread over all W.  A run
// whose simulations do not fill the chip takes a larger W (gwidth), down to
// one simulation per wavefront.
//
// Algorithm (restated lane by lane by the oracle's group mode):
//  * propensities and criticality per reaction as in the one-lane kernel;
//  * a0 and every cumulative selection use the lane partial sums (each
//    lane's reactions in ascending order) combined by an inclusive scan over
//    the G lanes (Hillis-Steele inside rows of 16 lanes, then the row totals
//    carried across rows; see gscan); a selection takes the first lane with
//    a positive partial whose inclusive sum reaches the threshold (else the
//    last lane with a positive partial), then walks that lane's reactions;
//  * tau' per species as in the one-lane kernel, minimum across lanes;
//  * group-wide draws (tau'', critical pick, SSA uniforms) come from the
//    event's Philox stream with counter word 3 = 0; lane l's small-lambda
//    Poisson process from the stream with word 3 = 1 + l (first gap drawn at
//    the start of the attempt); the count of a reaction with lambda >= 1
//    from the reaction's own stream (word 3 = 2^31 | j), so those draws can
//    be queued and spread over the group's lanes;
//  * the leap update and its negativity / int32 test run per species over
//    the species-major fear entries in ascending reaction order, which
//    rejects exactly when the reaction-major order of test_update
//    (2phase_n-tau-leaping.cu:1300-1351) would.
#pragma once

#include "ctl_kernels.h"

#pragma clang fp contract(off)

namespace ctl {

// LDS ordering between lanes of one wavefront (a group never spans two).
__device__ __forceinline__ void gsync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------------------
// Phase clock, compiled only into the profiling build of the library
// (CTL_PHASE_CLOCK=1: libctl_phases.so, ctl_phase_clock): the time the
// wavefronts spend in each phase of the group kernel, from s_memtime read at
// phase boundaries and summed over the launch's wavefronts.  The segment
// between two consecutive marks of a wavefront is added to the phase of the
// later mark by the wavefront's lowest active lane (the last mark's time is
// kept per wavefront, so the two sides of a divergent branch count once
// each).  The normal build compiles the marks to nothing.
// ---------------------------------------------------------------------------
enum : int {
    PH_PROPS = 0, PH_TAU1, PH_PICK, PH_COUNTS, PH_POISSON, PH_UPDATE, PH_SAMPLE,
    PH_SSA_OPEN, PH_SSA_SELECT, PH_SSA_UPDATE, PH_SSA_DEPS,
    PH_PRE_LEAP, PH_PRE_SSA, PH_LOOP, PH_REGROUP, PH_PARK, PH_COUNT
};
#if CTL_PHASE_CLOCK
static __device__ unsigned long long phase_total[PH_COUNT];
static __shared__ unsigned long long phase_row[4][PH_COUNT + 1];    // per wavefront; last: time of the last mark
__device__ __forceinline__ bool phase_leader() {
    return (int)(threadIdx.x & 63u) == __builtin_ffsll((long long)__ballot(1)) - 1;
}
// The clock read is a volatile asm with a memory clobber, so that the
// compiler neither merges the reads of two branches nor moves the row
// updates across them (a predicated if/else would interleave both sides).
__device__ __forceinline__ unsigned long long phase_now() {
    unsigned long long t;
    asm volatile("s_memtime %0\n\ts_waitcnt lgkmcnt(0)" : "=s"(t) : : "memory");
    return t;
}
__device__ __forceinline__ void phase_start() {
    if (phase_leader()) {
        unsigned long long* r = phase_row[threadIdx.x >> 6];
        for (int k = 0; k < PH_COUNT; ++k) r[k] = 0ull;
        r[PH_COUNT] = phase_now();
    }
}
__device__ __forceinline__ void phase_mark(int k) {
    const unsigned long long t = phase_now();
    if (phase_leader()) {
        unsigned long long* r = phase_row[threadIdx.x >> 6];
        r[k] += t - r[PH_COUNT];
        r[PH_COUNT] = t;
    }
}
__device__ __forceinline__ void phase_flush() {
    if (phase_leader()) {
        unsigned long long* r = phase_row[threadIdx.x >> 6];
        for (int k = 0; k < PH_COUNT; ++k)
            if (r[k]) {
                atomicAdd(&phase_total[k], r[k]);
                r[k] = 0ull;
            }
    }
}
#define CTL_PHASE_START() phase_start()
#define CTL_PHASE(k) phase_mark(k)
#define CTL_PHASE_FLUSH() phase_flush()
#else
#define CTL_PHASE_START() ((void)0)
#define CTL_PHASE(k) ((void)0)
#define CTL_PHASE_FLUSH() ((void)0)
#endif

// How propensities are computed (KParams::pfast): 0 from the reactant
// entries (any multiplicity), 1 as two entries of the LDS factor table, 2 as
// two entries computed from the state (models with at most two reactant
// entries of multiplicity <= 2, 1 when the table fits in the Kc region).
// PFM 0..2 fixes the mode at compile time (the simulation kernels: one
// instance per mode, so none keeps another's registers live); PFM 3 reads
// p.pfast (the batch kernels, whose models differ).
template <int PFM>
__device__ __forceinline__ int pmode(int pfast) {
    if constexpr (PFM == 3) return pfast;
    else return PFM;
}

// Two reactant entries (multiplicity 0, 1 or 2) from the state: the
// arithmetic and the criticality test of greactant, in the same order.
__device__ __forceinline__ void gtwo(float& a, bool& c, int32_t x0, uint32_t v0, int32_t x1, uint32_t v1,
                                     uint32_t nc) {
    const int32_t xs[2] = {x0, x1};
    const uint32_t vs[2] = {v0, v1};
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int32_t x = xs[k];
        const uint32_t v = vs[k];
        const float xf = (float)x;
        const float f2 = (x < 2) ? 0.0f : (0.5f * xf) * (float)(x - 1);
        a = a * (v == 1u ? xf : (v == 2u ? f2 : 1.0f));
        c = c || ((uint32_t)x >= v && (uint32_t)x < nc * v);
    }
}

// A kernel parameter read at its point of use: the compiler may not hoist a
// test of it out of the main loop, where it would hold a 64-bit lane mask in
// scalar registers for the whole kernel (and spill others).
static __device__ __forceinline__ int kuse(int v) {
#if CTL_UNIFORM_PARAMS
    v = __builtin_amdgcn_readfirstlane(v);         // uniform; a no-op when already scalar
    asm volatile("" : "+s"(v));
#endif
    return v;
}

template <int G>
__device__ __forceinline__ uint64_t gballot(bool pred) {
    const uint64_t b = __ballot(pred);
    if (G == 64) return b;
    const int base = (int)(threadIdx.x & 63u) & ~(G - 1);
    return (b >> base) & ((1ull << G) - 1ull);
}

// Cross-lane moves inside a row of 16 lanes through DPP (a VALU operand
// modifier, no LDS round trip).  Lanes whose source is outside the row read 0.
template <int CTRL>
__device__ __forceinline__ float dppf(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
enum : int {
    DPP_QP_1133 = 0xF5,       // quad_perm [1,1,3,3]
    DPP_QP_3333 = 0xFF,       // quad_perm [3,3,3,3]
    DPP_QP_1032 = 0xB1,       // quad_perm [1,0,3,2]  (xor 1)
    DPP_QP_2301 = 0x4E,       // quad_perm [2,3,0,1]  (xor 2)
    DPP_ROW_SHL4 = 0x104,
    DPP_ROW_SHR1 = 0x111,
    DPP_ROW_SHR2 = 0x112,
    DPP_ROW_SHR4 = 0x114,
    DPP_ROW_SHR8 = 0x118,
    DPP_ROW_MIRROR = 0x140,
    DPP_ROW_HALF_MIRROR = 0x141,
    DPP_ROW_NEWBCAST15 = 0x15F,   // lane 15 of each row to the whole row
    DPP_WAVE_SHR1 = 0x138,        // lane l reads lane l - 1 across rows
    DPP_ROW_BCAST15 = 0x142,      // lane 15 of each row to the next row
    DPP_ROW_BCAST31 = 0x143,      // lane 31 to rows 2 and 3
};

// Inclusive scan over the group.  Inside each DPP row of 16 lanes (the whole
// group when G <= 16) a Hillis-Steele scan, v_l <- v_{l-d} + v_l for
// d = 1, 2, 4, 8; wider groups then add the previous row's total to rows 1
// and 3 (row_bcast:15) and, for G = 64, the first two rows' total to rows 2
// and 3 (row_bcast:31).
template <int G>
__device__ __forceinline__ float gscan(float v, int l) {
    float t;
    if (G == 16) {
        // the group is the DPP row: a shifted-in lane reads 0, and 0 + v = v
        // (v is a sum of non-negative terms started from +0, never -0)
        v = dppf<DPP_ROW_SHR1>(v) + v;
        v = dppf<DPP_ROW_SHR2>(v) + v;
        v = dppf<DPP_ROW_SHR4>(v) + v;
        v = dppf<DPP_ROW_SHR8>(v) + v;
    } else if (G < 16) {
        if (G >= 2) { t = dppf<DPP_ROW_SHR1>(v); if (l >= 1) v = t + v; }
        if (G >= 4) { t = dppf<DPP_ROW_SHR2>(v); if (l >= 2) v = t + v; }
        if (G >= 8) { t = dppf<DPP_ROW_SHR4>(v); if (l >= 4) v = t + v; }
        if (G >= 16) { t = dppf<DPP_ROW_SHR8>(v); if (l >= 8) v = t + v; }
    } else {
        v = dppf<DPP_ROW_SHR1>(v) + v;              // a shifted-in lane reads 0
        v = dppf<DPP_ROW_SHR2>(v) + v;
        v = dppf<DPP_ROW_SHR4>(v) + v;
        v = dppf<DPP_ROW_SHR8>(v) + v;
        v = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), DPP_ROW_BCAST15, 0xa, 0xf, false)) + v;
        if (G == 64)
            v = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), DPP_ROW_BCAST31, 0xc, 0xf, false)) + v;
    }
    return v;
}

__device__ __forceinline__ float rdlane(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// The value of the group's last lane, in every lane of the group.
template <int G>
__device__ __forceinline__ float gbcast_last(float v, int l) {
    if (G == 2) return dppf<DPP_QP_1133>(v);
    if (G == 4) return dppf<DPP_QP_3333>(v);
    if (G == 8) {
        const float t = dppf<DPP_QP_3333>(v);
        const float u = dppf<DPP_ROW_SHL4>(t);
        return l < 4 ? u : t;
    }
    const int wl = (int)(threadIdx.x & 63u);
    if (G == 16) return dppf<DPP_ROW_NEWBCAST15>(v);
    if (G == 32) {
        const float r0 = rdlane(v, 31), r1 = rdlane(v, 63);
        return wl < 32 ? r0 : r1;
    }
    return rdlane(v, 63);
}

// Minimum over the group (exact in any order).
template <int G>
__device__ __forceinline__ float gmin(float v) {
    float o;
    if (G >= 2) { o = dppf<DPP_QP_1032>(v); v = o < v ? o : v; }
    if (G >= 4) { o = dppf<DPP_QP_2301>(v); v = o < v ? o : v; }
    if (G >= 8) { o = dppf<DPP_ROW_HALF_MIRROR>(v); v = o < v ? o : v; }
    if (G >= 16) { o = dppf<DPP_ROW_MIRROR>(v); v = o < v ? o : v; }
    if (G >= 32) {                                  // combine the rows' minima
        const float r0 = rdlane(v, 15), r1 = rdlane(v, 31), r2 = rdlane(v, 47), r3 = rdlane(v, 63);
        const float m01 = r1 < r0 ? r1 : r0, m23 = r3 < r2 ? r3 : r2;
        if (G == 64) v = m23 < m01 ? m23 : m01;
        else v = (threadIdx.x & 32u) ? m23 : m01;
    }
    return v;
}

template <int CTRL>
__device__ __forceinline__ uint64_t dppu64(uint64_t v) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, 0xf, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), CTRL, 0xf, 0xf, false);
    return ((uint64_t)hi << 32) | lo;
}

template <int G>
__device__ __forceinline__ uint64_t gsum64(uint64_t v) {
    if constexpr (G <= 16) {
        // butterfly inside the DPP row (the pairings of gmin); integer sums are exact in any order
        if (G >= 2) v += dppu64<DPP_QP_1032>(v);
        if (G >= 4) v += dppu64<DPP_QP_2301>(v);
        if (G >= 8) v += dppu64<DPP_ROW_HALF_MIRROR>(v);
        if (G >= 16) v += dppu64<DPP_ROW_MIRROR>(v);
        return v;
    }
#pragma unroll
    for (int m = G / 2; m >= 1; m >>= 1) {
        const uint32_t lo = __shfl_xor((uint32_t)v, m, G);
        const uint32_t hi = __shfl_xor((uint32_t)(v >> 32), m, G);
        v += ((uint64_t)hi << 32) | lo;
    }
    return v;
}

// Sum of uint32 over the group (the caller knows that it fits).
template <int G>
__device__ __forceinline__ uint32_t gsum32(uint32_t v) {
    auto step = [&](int o) { v += (uint32_t)o; };
    if (G >= 2) step(__builtin_amdgcn_update_dpp(0, (int)v, DPP_QP_1032, 0xf, 0xf, false));
    if (G >= 4) step(__builtin_amdgcn_update_dpp(0, (int)v, DPP_QP_2301, 0xf, 0xf, false));
    if (G >= 8) step(__builtin_amdgcn_update_dpp(0, (int)v, DPP_ROW_HALF_MIRROR, 0xf, 0xf, false));
    if (G >= 16) step(__builtin_amdgcn_update_dpp(0, (int)v, DPP_ROW_MIRROR, 0xf, 0xf, false));
    if (G >= 32) {                                  // add the rows' sums
        const uint32_t r0 = __builtin_amdgcn_readlane(v, 15), r1 = __builtin_amdgcn_readlane(v, 31);
        const uint32_t r2 = __builtin_amdgcn_readlane(v, 47), r3 = __builtin_amdgcn_readlane(v, 63);
        if (G == 64) v = (r0 + r1) + (r2 + r3);
        else v = (threadIdx.x & 32u) ? r2 + r3 : r0 + r1;
    }
    return v;
}

// Group state: the scalars are identical in every lane of the group; the
// Poisson / gap counters are per lane and summed when the simulation ends.
// The group's stream (counter word 3 = 0) with its Philox blocks spread over
// the group: lane i holds block cb + i of the current event, so 4G words (2G
// SSA steps) cost each lane one Philox evaluation where a per-lane buffer
// costs one per 4 words, and the groups of a wavefront, at different points
// of their streams, seldom make the wavefront evaluate Philox for one of them
// alone.  A word is read from the lane that holds its block; the words and
// their order are those of a per-lane stream (rng_u32).
struct GRng {
    uint32_t k0, k1;             // key
    uint32_t sim;                // global simulation index
    uint32_t ev;                 // current event
    uint32_t wc;                 // words of the event consumed
    uint32_t cb;                 // first block held by the group (GRNG_NONE: none)
    uint32_t c0, c1, c2, c3;     // this lane's block, cb + lane
};
constexpr uint32_t GRNG_NONE = 0x80000000u;   // b - cb >= 2^31 for every block b of an event

__device__ __forceinline__ void grng_event(GRng& g, uint32_t ev) {
    g.ev = ev;
    g.wc = 0u;
    g.cb = GRNG_NONE;
}

template <int W>
__device__ __forceinline__ uint32_t grng_u32(GRng& g, int l) {
    const uint32_t b = g.wc >> 2;
    if (b - g.cb >= (uint32_t)W) {
        g.cb = b;
        philox_block(b + (uint32_t)l, g.ev, g.sim, 0u, g.k0, g.k1, g.c0, g.c1, g.c2, g.c3);
    }
    // the four words as values: a select between loads of the struct's fields
    // would become a load through a selected address, which keeps the whole
    // lane state in scratch memory
    uint32_t c0 = g.c0, c1 = g.c1, c2 = g.c2, c3 = g.c3;
    asm volatile("" : "+v"(c0), "+v"(c1), "+v"(c2), "+v"(c3));
    const uint32_t k = g.wc & 3u;
    const uint32_t lo = (k & 1u) ? c1 : c0;
    const uint32_t hi = (k & 1u) ? c3 : c2;
    const uint32_t mine = (k & 2u) ? hi : lo;
    const int src = (int)(b - g.cb);
    g.wc += 1u;
    return __shfl(mine, src, W);
}

// Two consecutive words of one block (an SSA step's: an event's steps consume
// two words each, so a pair never spans blocks).
template <int W>
__device__ __forceinline__ void grng_pair(GRng& g, int l, uint32_t& w0, uint32_t& w1) {
    const uint32_t b = g.wc >> 2;
    if (b - g.cb >= (uint32_t)W) {
        g.cb = b;
        philox_block(b + (uint32_t)l, g.ev, g.sim, 0u, g.k0, g.k1, g.c0, g.c1, g.c2, g.c3);
    }
    uint32_t c0 = g.c0, c1 = g.c1, c2 = g.c2, c3 = g.c3;      // values: see grng_u32
    asm volatile("" : "+v"(c0), "+v"(c1), "+v"(c2), "+v"(c3));
    const bool hi = (g.wc & 2u) != 0u;
    const int src = (int)(b - g.cb);
    g.wc += 2u;
    w0 = __shfl(hi ? c2 : c0, src, W);
    w1 = __shfl(hi ? c3 : c1, src, W);
}

struct GLane {
    int slot;                // group slot
    int sim;                 // local index, -1 none, -2 queue exhausted
    double t;
    uint32_t cursor, evc, xb;
    uint64_t firings, ssa_steps;
    uint32_t leaps, rejections, switches, absorbed;
    uint64_t poisson, gaps;
    const float* crate;      // the simulation's rate constants (HBM, cached)
    const uint32_t* fvrow;   // the simulation's feed values (when the model has feeds)
    GRng gg;                 // group stream (word 3 = 0)
    Rng lg;                  // this lane's stream (word 3 = 1 + lane)
    double tacc;             // clock advance of the SSA burst in progress
    int ssa_left;            // steps left in the SSA burst in progress (0: none)
    int ssa_mode;            // 1 once a leap attempt switched, until its burst has run
};

struct GView {
    int32_t* Xb;             // [2][S]
    uint32_t* A;             // [Rp] (entries R .. Rp-1 stay 0)
    int32_t* Kc;             // [Rp]
    uint16_t* Qx;            // [R] own queue region, or null: the queue lives in the trial state
    uint32_t* F;             // [2S+1] reactant factors, in the Kc region (used only when 2S + 1 <= Rp)
    uint32_t* qn;            // length of the Poisson queue (LDS atomic counter)
};

// Padded reaction count of the LDS arrays: R + 1 rounded up to a multiple of
// G.  The entries past R stay zero in A, so a loop over a lane's rounds needs
// no per-lane bounds test and A[R] is a zero propensity that padding entries
// of the tau' stream point at.
__host__ __device__ __forceinline__ int group_rpad(int R, int G) { return (R + G) / G * G; }

// LDS words of one group's simulation: X[2][S], A[Rp], Kc[Rp], then one
// region shared by the queue of lambda >= 1 reactions (16-bit indices; it
// lives in the trial-state half of X, free until the update writes it, when
// R/2 <= S) and the factor table F[2S+1] (in Kc when 2S+1 <= Rp): the queue
// is used only by the count phase, the table only before it and in SSA;
// last, the queue's length.
__host__ __device__ __forceinline__ size_t group_lds_words(int S, int R, int G) {
    const size_t Rp = (size_t)group_rpad(R, G);
    const size_t q = ((size_t)R + 1) / 2;
    const size_t qx = q > (size_t)S ? q : 0;
    return (size_t)2 * S + 2 * Rp + qx + 1;
}

__device__ __forceinline__ GView group_view(uint32_t* base, int S, int R, int G) {
    GView V;
    const int Rp = group_rpad(R, G);
    V.Xb = (int32_t*)base;
    V.A = (uint32_t*)(V.Xb + 2 * S);
    V.Kc = (int32_t*)(V.A + Rp);
    V.Qx = ((size_t)R + 1) / 2 > (size_t)S ? (uint16_t*)(V.Kc + Rp) : nullptr;
    V.F = (uint32_t*)V.Kc;              // factor table (only when 2S + 1 <= Rp: see pfast)
    V.qn = base + group_lds_words(S, R, G) - 1;
    return V;
}

// The reactant factors of species s from its count x (the arithmetic and the
// criticality test of greactant for multiplicities 1 and 2): x and
// x (x - 1) / 2 as FP32, bit 31 set when v <= x < nc v.
__device__ __forceinline__ void gfactor(uint32_t* F, int S, int s, int32_t x, uint32_t nc) {
    const float xf = (float)x;
    const float f2 = (x < 2) ? 0.0f : (0.5f * xf) * (float)(x - 1);
    const bool c1 = (uint32_t)x >= 1u && (uint32_t)x < nc;
    const bool c2 = (uint32_t)x >= 2u && (uint32_t)x < nc * 2u;
    F[s] = __float_as_uint(xf) | (c1 ? 0x80000000u : 0u);
    F[S + s] = __float_as_uint(f2) | (c2 ? 0x80000000u : 0u);
}

// The whole factor table of state X; F[2S] = 1.0 is the factor of a padding
// entry (multiplicity 0), never critical.
template <int W>
__device__ __forceinline__ void gfactors(const KParams& p, const int32_t* X, uint32_t* F, int l) {
    const uint32_t nc = (uint32_t)p.nc;
    for (int s = l; s < p.S; s += W) gfactor(F, p.S, s, X[s], nc);
    if (l == 0) F[2 * p.S] = 0x3f800000u;
}

// Zeroes a group's A padding (R .. Rp-1); done when the group's model is set.
template <int G, int W>
__device__ __forceinline__ void gzero_pad(const GView& V, int R, int l) {
    for (int j = R + l; j < group_rpad(R, G); j += W) V.A[j] = 0u;
}

// Propensity of reaction j from the group's LDS state; the arithmetic of
// prop_one (CalculatePropensity, T.cu:1443-1470, in FP32).
__device__ __forceinline__ void greactant(float& a, bool& c, int32_t x, int v, uint32_t nc) {
    if (v == 1) {
        a = a * (float)x;
    } else if (v == 2) {
        a = a * ((x < 2) ? 0.0f : (0.5f * (float)x) * (float)(x - 1));
    } else if (x < v) {
        a = a * 0.0f;
    } else {
        for (int q = 1; q <= v; ++q) a = a * ((float)(x - q + 1) / (float)q);
    }
    // 0 < floor(x / v) < nc, as compares: v <= x < nc * v
    c = c || ((uint32_t)x >= (uint32_t)v && (uint64_t)(uint32_t)x < (uint64_t)nc * (uint32_t)v);
}

// Reaction j from its own reactant list (the SSA dependents).
__device__ __forceinline__ float gprop(const KParams& p, const int32_t* X, const float* crate, int j, bool& crit) {
    float a = crate[j];
    bool c = false;
    const uint32_t h1 = p.T[p.oLp + j + 1];
    for (uint32_t h = p.T[p.oLp + j]; h < h1; ++h) {
        const uint32_t e = p.T[p.oLe + h];
        greactant(a, c, X[e & 0xffffu], (int)(e >> 16), (uint32_t)p.nc);
    }
    crit = c;
    return a;
}

// gprops with W > G lanes per simulation: lane l computes reactions l, l + W,
// ..., so a round of W lanes covers W / G of the algorithm's rounds; then every
// algorithm lane's partial sums are added from LDS in ascending round order
// (the W / G lanes that stand for one algorithm lane do so redundantly).  The
// propensities are the same values, the sums the same additions.
template <int G, int W, int PFM>
__device__ __forceinline__ void gprops_wide(const KParams& p, const int32_t* X, const uint32_t* F, const float* crate,
                                            uint32_t* A, int l, float& P, float& PC) {
    const int pm = pmode<PFM>(kuse(p.pfast));
    const uint32_t nc = (uint32_t)p.nc;
    const int a0 = l & (G - 1);
    if (pm != 0) {
        const uint32_t* E = p.T + p.oPRe;
        for (int j0 = l; j0 < p.R; j0 += 4 * W) {
            float cr[4];
            uint32_t e0[4], e1[4], u0[4], u1[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int j = j0 + q * W;
                cr[q] = 0.0f;
                e0[q] = e1[q] = pm == 1 ? (uint32_t)(2 * p.S) : 0u;
                if (j < p.R) {
                    const uint32_t* Er = E + (2 * (j / G)) * G + a0;
                    e0[q] = Er[0];
                    e1[q] = Er[G];
                    cr[q] = crate[j];
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                u0[q] = pm == 1 ? F[e0[q]] : (uint32_t)X[e0[q] & 0xffffu];
                u1[q] = pm == 1 ? F[e1[q]] : (uint32_t)X[e1[q] & 0xffffu];
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int j = j0 + q * W;
                if (j < p.R) {
                    float a = cr[q];
                    uint32_t cbit;
                    if (pm == 1) {
                        a = a * __uint_as_float(u0[q] & 0x7fffffffu);
                        a = a * __uint_as_float(u1[q] & 0x7fffffffu);
                        cbit = (u0[q] | u1[q]) & 0x80000000u;
                    } else {
                        bool c = false;
                        gtwo(a, c, (int32_t)u0[q], e0[q] >> 16, (int32_t)u1[q], e1[q] >> 16, nc);
                        cbit = c ? 0x80000000u : 0u;
                    }
                    A[j] = __float_as_uint(a) | cbit;
                }
            }
        }
    } else {
        for (int j = l; j < p.R; j += W) {
            bool c;
            const float a = gprop(p, X, crate, j, c);
            A[j] = __float_as_uint(a) | (c ? 0x80000000u : 0u);
        }
    }
    gsync();
    P = 0.0f;
    PC = 0.0f;
    const int nrp = group_rpad(p.R, G) / G;
    constexpr int D = W > 16 ? 16 : 4;                 // reads in flight
    for (int r0 = 0; r0 < nrp; r0 += D) {
        uint32_t u[D];
#pragma unroll
        for (int q = 0; q < D; q += 4)
            if (r0 + q < nrp) {
#pragma unroll
                for (int i = q; i < q + 4; ++i) u[i] = A[a0 + (r0 + i < nrp ? r0 + i : nrp - 1) * G];
            }
#pragma unroll
        for (int q = 0; q < D; q += 4)
            if (r0 + q < nrp) {
#pragma unroll
                for (int i = q; i < q + 4; ++i) {
                    const float a = r0 + i < nrp ? aval(u[i]) : 0.0f;
                    P = P + a;
                    PC = PC + ((u[i] & 0x80000000u) ? a : 0.0f);
                }
            }
    }
}

// Every reaction of lane l (j = l, l + G, ...) from the reactant round
// stream: the table addresses do not depend on loaded data, so the loads of a
// round issue together.  Writes A[j] (propensity bits | critical << 31) and
// returns the lane's partial sums of all and of the critical propensities.
// With pfast the two entries of a reaction are indices into the factor table
// F of the state (built by gfactors), so a reaction costs two multiplies:
// the same factors in the same order as greactant, hence the same bits.
template <int G, int W, int PFM = 3>
__device__ __forceinline__ void gprops(const KParams& p, const int32_t* X, const uint32_t* F, const float* crate,
                                       uint32_t* A, int l, float& P, float& PC) {
    if constexpr (W > G) {
        gprops_wide<G, W, PFM>(p, X, F, crate, A, l, P, PC);
        return;
    }
    const int nr = (p.R + G - 1) / G;
    P = 0.0f;
    PC = 0.0f;
    const int pm = pmode<PFM>(kuse(p.pfast));
    if (pm == 2) {
        // two entries per reaction (species | multiplicity << 16) read from
        // the state; four rounds per batch of loads
        const uint32_t* E = p.T + p.oPRe + l;
        const uint32_t nc = (uint32_t)p.nc;
        for (int r0 = 0; r0 < nr; r0 += 4) {
            float cr[4];
            uint32_t e0[4], e1[4];
            int32_t x0[4], x1[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = r0 + q, j = l + r * G;
                cr[q] = 0.0f;
                e0[q] = e1[q] = 0u;
                if (r < nr) {
                    e0[q] = E[(2 * r) * G];
                    e1[q] = E[(2 * r + 1) * G];
                    if (j < p.R) cr[q] = crate[j];
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                x0[q] = X[e0[q] & 0xffffu];
                x1[q] = X[e1[q] & 0xffffu];
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = r0 + q, j = l + r * G;
                if (r < nr) {                          // past R: 0 (rate 0) into A's zero padding
                    float a = cr[q];
                    bool c = false;
                    gtwo(a, c, x0[q], e0[q] >> 16, x1[q], e1[q] >> 16, nc);
                    A[j] = __float_as_uint(a) | (c ? 0x80000000u : 0u);
                    P = P + a;
                    if (c) PC = PC + a;
                }
            }
        }
        return;
    }
    if (pm == 1) {
        // two entries per reaction; four rounds per batch of loads
        const uint32_t* E = p.T + p.oPRe + l;
        for (int r0 = 0; r0 < nr; r0 += 4) {
            float cr[4];
            uint32_t e0[4], e1[4];
            uint32_t u0[4], u1[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = r0 + q, j = l + r * G;
                cr[q] = 0.0f;
                e0[q] = e1[q] = (uint32_t)(2 * p.S);
                if (r < nr) {
                    e0[q] = E[(2 * r) * G];
                    e1[q] = E[(2 * r + 1) * G];
                    if (j < p.R) cr[q] = crate[j];
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                u0[q] = F[e0[q]];
                u1[q] = F[e1[q]];
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = r0 + q, j = l + r * G;
                if (r < nr) {                          // past R: 0 (rate 0) into A's zero padding
                    float a = cr[q];
                    a = a * __uint_as_float(u0[q] & 0x7fffffffu);
                    a = a * __uint_as_float(u1[q] & 0x7fffffffu);
                    const uint32_t c = (u0[q] | u1[q]) & 0x80000000u;
                    A[j] = __float_as_uint(a) | c;
                    P = P + a;
                    if (c) PC = PC + a;
                }
            }
        }
        return;
    }
    const ctab_u32 TC = CT_U32(p.T);
    const uint32_t* E = p.T + p.oPRe + l;
    for (int r = 0, j = l; r < nr; ++r, j += G) {
        const uint32_t len = TC[p.oPRm + r];
        if (j < p.R) {
            float a = crate[j];
            bool c = false;
            for (uint32_t k = 0; k < len; ++k) {
                const uint32_t e = E[k * G];
                const int v = (int)(e >> 16);
                if (v != 0) greactant(a, c, X[e & 0xffffu], v, (uint32_t)p.nc);
            }
            A[j] = __float_as_uint(a) | (c ? 0x80000000u : 0u);
            P = P + a;
            if (c) PC = PC + a;
        }
        E += len * G;
    }
}

// Selection: among the lanes with a positive own partial (Pown), the first
// whose inclusive sum P reaches w, else the last such lane; then the walk
// through that lane's reactions from the previous lane's inclusive sum
// (the critical ones plus reaction 0: the reference's pick walk starts from
// a_0, T.cu:1993-2006).  Lanes
// with a zero partial are skipped: the scan associates differently per lane,
// so such a lane's inclusive sum can round above its predecessor's.  Only a
// reaction with a positive propensity is chosen.  Returns the chosen
// reaction (group-uniform) or -1 when no lane has a positive partial.
template <int G, int W>
__device__ __forceinline__ int gselect(const KParams& p, const uint32_t* A, float Pown, float P, float w, int l) {
    const uint64_t cand = gballot<G>(Pown > 0.0f);
    if (cand == 0) return -1;
    const uint64_t hit = gballot<G>(Pown > 0.0f && P >= w);
    const int sel = hit ? __builtin_ctzll(hit) : 63 - __builtin_clzll(cand);
    const float excl = G <= 16 ? dppf<DPP_ROW_SHR1>(P) : dppf<DPP_WAVE_SHR1>(P);   // lane 0's value is unused
    // The walk through lane sel's reactions sel + i*G, spread over the first
    // N lanes of the team (a row of 16 at most): lane i holds the i-th
    // propensity and the sequential sums excl + a_0 + ... + a_i are built by
    // N-1 row shifts (after k shifts lanes 0..k hold their final sum; a
    // shifted-in 0 or a skipped entry adds an exact 0), so every sum is
    // rounded as in the one-lane walk.  Lane sel's reactions number at most
    // 16 per round; wider teams leave their other rows idle.
    constexpr int N = W <= 16 ? W : 16;
    const int nj = (p.R - sel + G - 1) / G;
    float carry = __shfl(excl, sel, G);
    if (sel == 0) carry = 0.0f;
    int last = -1;
    for (int c = 0; c < nj; c += N) {
        const int i = c + l;
        const bool in = l < N && i < nj;
        const int j = sel + i * G;
        const uint32_t u = in ? A[j] : 0u;
        const bool use = (u & 0x80000000u) || j == 0;
        const float a = use ? aval(u) : 0.0f;
        const float a1 = l == 0 ? carry + a : a;
        float x = a1;
#pragma unroll
        for (int k = 1; k < N; ++k) {
            const float t = dppf<DPP_ROW_SHR1>(x) + a1;
            x = (N == 16 || l > 0) ? t : a1;
        }
        const uint64_t pos = gballot<W>(in && a > 0.0f);
        const uint64_t hm = gballot<W>(in && a > 0.0f && w <= x);
        if (hm) return sel + (c + __builtin_ctzll(hm)) * G;
        if (pos) last = sel + (c + 63 - __builtin_clzll(pos)) * G;
        carry = W <= 16 ? gbcast_last<W>(x, l) : __shfl(x, N - 1, W);
    }
    return last;
}

// Minimum of an int over N lanes (N <= 16).
template <int N>
__device__ __forceinline__ int gmini(int v) {
    auto step = [&](int o) { v = o < v ? o : v; };
    if (N >= 2) step(__builtin_amdgcn_update_dpp(v, v, DPP_QP_1032, 0xf, 0xf, false));
    if (N >= 4) step(__builtin_amdgcn_update_dpp(v, v, DPP_QP_2301, 0xf, 0xf, false));
    if (N >= 8) step(__builtin_amdgcn_update_dpp(v, v, DPP_ROW_HALF_MIRROR, 0xf, 0xf, false));
    if (N >= 16) step(__builtin_amdgcn_update_dpp(v, v, DPP_ROW_MIRROR, 0xf, 0xf, false));
    return v;
}

// The same over all reactions for the SSA step, without branches
// that depend on the simulation: a taken branch costs about 20 ns, and
// straight-line code lets the step's exponential run between the row shifts.
// cand: the lanes with a positive partial (not 0).  Teams narrower than 16
// fold in chunks of N reactions, each lane keeping the first of its own that
// reaches w.
template <int G, int W>
__device__ __forceinline__ int gselect_ssa(const uint32_t* A, uint64_t cand, float Pown, float P, float w, int l,
                                           int nrp) {
    const uint64_t hit = gballot<G>(Pown > 0.0f && P >= w);
    const int sel = hit ? __builtin_ctzll(hit) : 63 - __builtin_clzll(cand);
    const float excl = G <= 16 ? dppf<DPP_ROW_SHR1>(P) : dppf<DPP_WAVE_SHR1>(P);   // lane 0's value is unused
    constexpr int N = W <= 16 ? W : 16;
    float carry = __shfl(excl, sel, G);
    if (sel == 0) carry = 0.0f;
    if (N == 16 && nrp <= 16) {              // the usual case: at most 16 reactions per lane
        const uint32_t u = A[sel + (l < nrp ? l : 0) * G];
        const float a = l < nrp ? aval(u) : 0.0f;
        const float a1 = l == 0 ? carry + a : a;
        float x = a1;
#pragma unroll
        for (int k = 1; k < 16; ++k) x = dppf<DPP_ROW_SHR1>(x) + a1;
        const uint64_t pos = gballot<W>(l < 16 && a > 0.0f);
        const uint64_t hm = gballot<W>(l < 16 && a > 0.0f && w <= x);
        return sel + (hm ? __builtin_ctzll(hm) : 63 - __builtin_clzll(pos)) * G;
    }
    constexpr int NONE = 0x7fffffff;
    int first = NONE;
    for (int c0 = 0; c0 < nrp; c0 += 4 * N) {
        uint32_t u[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int i = c0 + q * N + l;
            u[q] = A[sel + (i < nrp ? i : nrp - 1) * G];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (c0 + q * N >= nrp) break;
            const int i = c0 + q * N + l;
            const float a = (W == N || l < N) && i < nrp ? aval(u[q]) : 0.0f;
            const float a1 = l == 0 ? carry + a : a;
            float x = a1;
#pragma unroll
            for (int k = 1; k < N; ++k) {
                const float t = dppf<DPP_ROW_SHR1>(x) + a1;
                x = (N == 16 || l > 0) ? t : a1;
            }
            const int f = a > 0.0f && w <= x ? i : NONE;
            first = f < first ? f : first;
            carry = W <= 16 ? gbcast_last<W>(x, l) : __shfl(x, N - 1, W);
        }
    }
    first = gmini<N>(first);
    if (W > 16) first = __shfl(first, 0, W);             // the other rows hold no reactions
    if (first == NONE) {                                 // rounding left w above every sum: the last positive one
        int last = -1;
        for (int i = l; i < nrp; i += W) last = aval(A[sel + i * G]) > 0.0f ? i : last;
        for (int d = W / 2; d > 0; d >>= 1) {
            const int o = __shfl_xor(last, d, W);
            last = o > last ? o : last;
        }
        first = last;
    }
    return sel + first * G;
}

template <int W>
__device__ __forceinline__ void gabsorb(const KParams& p, GLane& L, const int32_t* X, int l) {
    uint32_t* out = p.storage + (size_t)L.sim * p.K * p.SS;
    if (L.cursor == 0) {
        for (int sk = l; sk < p.SS; sk += W) out[sk] = (uint32_t)X[p.T[p.oCs + sk]];
        L.cursor = 1;
    }
    const uint32_t* last = out + (size_t)(L.cursor - 1) * p.SS;
    for (int i = (int)L.cursor; i < p.K; ++i)
        for (int sk = l; sk < p.SS; sk += W) out[(size_t)i * p.SS + sk] = last[sk];
    L.t = p.tmax + (double)0.1f;
    L.cursor = (uint32_t)p.K;
    L.absorbed = 1;
}

// Four entries of a lane's round list from entry k on, one batch ahead of
// their use: without the barrier the compiler moves the loads back there.
// Taken by teams of more than 16 lanes, which wait for the L1 / L2 and not
// for issue slots: 200 reactions, 1000 simulations at W = 64 67.9 -> 66.9 ms,
// 300 reactions at G = W = 64 66.8 -> 64.7 ms; at W = 16, full chip, the four
// more registers cost 79.1 -> 82.3 ms.
template <int W>
__device__ __forceinline__ void gentries(const uint32_t* E, uint32_t k, uint32_t (&e)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) e[i] = E[(k + i) * W];
    asm volatile("" ::: "memory");
}

constexpr int LEAP_ATTEMPTS = 300;       // halvings after which a rejected leap gives up

// One adaptive leap attempt (PreCalculations, T.cu:1568-2093).
template <int G, int W, int PFM = 3>
__device__ __forceinline__ int gleap(const KParams& p, GLane& L, const GView& V, int l,
                                     const float* __restrict__ recip) {
    if (L.t >= p.tmax) return LEAP_DONE;
    const int la = l & (G - 1);              // the algorithm's lane this one stands for
    const bool own = l < G;                  // one lane per algorithm lane counts
    constexpr bool kAhead = W > 16 && (W > G || W == 64);    // see gentries
    int32_t* X = V.Xb + (L.xb ? p.S : 0);
    int32_t* X1 = V.Xb + (L.xb ? 0 : p.S);
    float P, PC;
    if (pmode<PFM>(kuse(p.pfast)) == 1) {
        gfactors<W>(p, X, V.F, l);
        gsync();
    }
    gprops<G, W, PFM>(p, X, V.F, L.crate, V.A, l, P, PC);
    gsync();
    P = gscan<G>(P, la);
    PC = gscan<G>(PC, la);
    const float a0 = gbcast_last<G>(P, la);
    const float a0c = gbcast_last<G>(PC, la);
    CTL_PHASE(PH_PROPS);
    if (a0 == 0.0f) { gabsorb<W>(p, L, X, l); return LEAP_ABSORB; }
    // tau' (T.cu:1860-1922): the one-lane kernel's per-species values, min over lanes
    float tau1 = 3.40282347e+38f;
    const ctab_u32 TC = CT_U32(p.T);
    const int nrs = (p.S + W - 1) / W;
    const uint32_t* E = p.T + p.oVRe + l;
    const uint32_t* SPI = p.T + p.oSPI + l;
    for (int r = 0; r < nrs; ++r) {
        const uint32_t len = TC[p.oVRm + r];
        const uint32_t spw = SPI[r * W];             // species | HOR << 16 | HORtype << 24
        float mu = 0.0f, sg = 0.0f;
        if (kuse(p.vhalf) == 2) {
            // every coefficient is 0 or a power of two: v a and v (v a) are
            // exact, so the fused additions round as the separate ones do
            const char* Ab = reinterpret_cast<const char*>(V.A);
            uint32_t en[4];
            if (kAhead && len > 0) gentries<W>(E, 0u, en);
            for (uint32_t k = 0; k < len; k += 4) {  // len is a multiple of 4
                uint32_t e[4];
                int32_t u[4];
                if (kAhead) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) e[i] = en[i];
                    gentries<W>(E, k + 4 < len ? k + 4 : k, en);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) e[i] = E[(k + i) * W];
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) u[i] = *reinterpret_cast<const int32_t*>(Ab + (e[i] & 0xffffu));
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float v = (float)__builtin_bit_cast(_Float16, (uint16_t)(e[i] >> 16));
                    const float a = __int_as_float(u[i] > 0 ? u[i] : 0);     // critical: 0, see below
                    mu = fmaf(v, a, mu);
                    sg = fmaf(v, v * a, sg);
                }
            }
        } else if (kuse(p.vhalf)) {
            // entries (coefficient as FP16 << 16 | byte offset of A[reaction]):
            // both halves are read as operand selects, and v * v in FP32 is exact
            const char* Ab = reinterpret_cast<const char*>(V.A);
            uint32_t en[4];
            if (kAhead && len > 0) gentries<W>(E, 0u, en);
            for (uint32_t k = 0; k < len; k += 4) {  // len is a multiple of 4
                uint32_t e[4];
                int32_t u[4];
                if (kAhead) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) e[i] = en[i];
                    gentries<W>(E, k + 4 < len ? k + 4 : k, en);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) e[i] = E[(k + i) * W];
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) u[i] = *reinterpret_cast<const int32_t*>(Ab + (e[i] & 0xffffu));
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float v = (float)__builtin_bit_cast(_Float16, (uint16_t)(e[i] >> 16));
                    // a critical propensity has bit 31 set: as an integer it is
                    // negative and the maximum with 0 gives +0; padding (A[R] = 0)
                    // adds an exact zero too
                    const float a = __int_as_float(u[i] > 0 ? u[i] : 0);
                    mu = mu + v * a;
                    sg = sg + (v * v) * a;
                }
            }
        } else {
            for (uint32_t k = 0; k < len; k += 4) {  // len is a multiple of 4
                uint32_t e[4], u[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) e[i] = E[(k + i) * W];
#pragma unroll
                for (int i = 0; i < 4; ++i) u[i] = V.A[e[i] & 0xffffu];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int v = (int)(int16_t)(e[i] >> 16);
                    // critical reactions and padding (A[R] = 0) add an exact zero
                    const float a = (u[i] & 0x80000000u) ? 0.0f : __uint_as_float(u[i]);
                    mu = mu + (float)v * a;
                    sg = sg + (float)(v * v) * a;
                }
            }
        }
        E += len * W;
        if (mu == 0.0f || sg == 0.0f) continue;      // no var entries (no species included)
        const int32_t x = X[spw & 0xffffu];
        const float ex = p.eps * (float)x;
        // g is 1 or 2 unless some species has HOR 3 or HOR 2 of type 2: then
        // the division by 2 is the exact scaling by 0.5
        const float tmp2 = kuse(p.gsimple) ? (((spw >> 16) & 0xffu) == 2u ? ex * 0.5f : ex)
                                           : ex / gfun(spw >> 16, x);
        const float macs = tmp2 > 1.0f ? tmp2 : 1.0f;
        const float t3 = macs / fabsf(mu);
        const float t4 = (macs * macs) / sg;
        const float tmp = t3 < t4 ? t3 : t4;
        if (tmp < tau1) tau1 = tmp;
    }
    tau1 = gmin<W>(tau1);
    CTL_PHASE(PH_TAU1);
    if (tau1 < p.ssa_factor / a0) { L.switches++; return LEAP_SWITCH; }      // T.cu:1935-1941
    uint32_t e = L.evc++;
    grng_event(L.gg, e);
    float tau2 = 3.40282347e+38f;
    if (a0c > 0.0f) tau2 = u32_exp(grng_u32<W>(L.gg, l)) / a0c;                                // T.cu:1962-1965
    float tau = tau1 < tau2 ? tau1 : tau2;
    int pick = -1;
    if (tau1 > tau2) {                                                         // T.cu:1993-2006
        const float w = u32_oc(grng_u32<W>(L.gg, l)) * a0c;
        float Q = 0.0f;
        for (int j = la; j < p.R; j += G) {
            const uint32_t u = V.A[j];
            if ((u & 0x80000000u) || j == 0) Q = Q + aval(u);
        }
        const float Qown = Q;
        Q = gscan<G>(Q, la);
        pick = gselect<G, W>(p, V.A, Qown, Q, w, l);
    }
    CTL_PHASE(PH_PICK);
    uint64_t fired = 0;
    for (int attempt = 0;; ++attempt) {                                        // T.cu:2011-2050
        if (attempt > 0) { e = L.evc++; L.rejections++; }
        // counts: critical reactions (the pick), the small-lambda process of
        // this lane (its first gap drawn up front), and a queue of the
        // reactions with lambda >= 1, drawn afterwards by the group's lanes in
        // parallel, each from the reaction's own stream (word 3 = 2^31 | j)
        rng_event(L.lg, e);
        uint32_t fk = 0;                         // counts of this loop: process events and the pick
        uint16_t* Q = V.Qx ? V.Qx : (uint16_t*)X1;
        if (l == 0) *V.qn = 0u;
        gsync();
        double cum = 0.0, pos = (double)exp_rv(L.lg);
        if (own) L.gaps++;
        // The lane's second event position is drawn now, with the first, by
        // every lane at once; drawn inside the loop below it would cost the
        // wavefront a divergent draw for almost every reaction round.  It is
        // the same value from the same stream (the lane stream serves only
        // these gaps), counted as a gap when it is used.
        double pos2 = pos + (double)exp_rv(L.lg);
        bool have2 = true;
        // Rounds in batches of four: their reads are in flight together, and
        // the events in the batch's span of the running sum are walked by one
        // loop (one turn per event of the busiest lane) instead of a loop per
        // reaction.
        const int nit = (p.R + G - 1) / G;
        for (int i0 = 0; i0 < nit; i0 += 4) {
            uint32_t u[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) u[q] = V.A[la + (i0 + q < nit ? i0 + q : nit - 1) * G];
            double cs[4];
            int32_t k[4];
            bool need[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {              // past R: the zero padding of A
                const int j = la + (i0 + q) * G;
                const bool in = i0 + q < nit;
                const bool crit = (u[q] & 0x80000000u) != 0u;
                const float lam = tau * __uint_as_float(u[q]);
                need[q] = in && !crit && !(lam < 1.0f);
                const bool small = in && !crit && lam < 1.0f && lam > 0.0f;
                k[q] = (crit && attempt == 0 && j == pick) ? 1 : 0;
                cum = small ? cum + (double)lam : cum;
                cs[q] = cum;
            }
            // pos >= cum held before this batch; an event belongs to the first
            // reaction whose running sum lies above it
            while (pos < cum) {
#pragma unroll
                for (int q = 0; q < 4; ++q) k[q] += pos < cs[q] && (q == 0 || !(pos < cs[q - 1])) ? 1 : 0;
                if (have2) {
                    pos = pos2;
                    have2 = false;
                } else {
                    pos = pos + (double)exp_rv(L.lg);
                }
                if (own) L.gaps++;
            }
            if (own) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (i0 + q < nit) {
                        V.Kc[la + (i0 + q) * G] = k[q];      // a queued reaction's count is drawn below
                        fk += (uint32_t)k[q];
                    }
            }
            // the queue's order is free: each count comes from its reaction's own stream
            if (own && (need[0] || need[1] || need[2] || need[3])) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (need[q]) Q[atomicAdd(V.qn, 1u)] = (uint16_t)(la + (i0 + q) * G);
            }
        }
        gsync();
        CTL_PHASE(PH_COUNTS);
        const uint32_t nq = *V.qn;
        uint64_t f = fk;
        for (uint32_t qi = (uint32_t)l; qi < nq; qi += W) {
            const int j = Q[qi];
            const float lam = tau * __uint_as_float(V.A[j]);
            Rng gr{};
            gr.k0 = L.gg.k0;
            gr.k1 = L.gg.k1;
            gr.sim = L.gg.sim;
            gr.tag = 0x80000000u | (uint32_t)j;
            rng_event(gr, e);
            const int32_t k = poisson(gr, lam, recip);
            V.Kc[j] = k;
            f += (uint64_t)k;
            L.poisson++;
        }
        gsync();
        CTL_PHASE(PH_POISSON);
        bool bad = false;
        const uint32_t* F = p.T + p.oFRe + l;
        const char* Kb = reinterpret_cast<const char*>(V.Kc);
        // While every lane drew fewer than flim / W firings, the counts are
        // below 2^23 and no partial sum leaves (-2^30, 2^31 + 2^30): bit 31 of
        // the sum modulo 2^32 says that it left [0, 2^31) (a 64-bit
        // multiply-add issues at a quarter of the rate).  The sums are
        // unsigned: a signed one beyond 2^31 - 1 has no defined value.
        if (__ballot(f >= (uint64_t)(p.flim / (uint32_t)W)) == 0) {
            for (int r = 0; r < nrs; ++r) {
                const uint32_t len = TC[p.oFRm + r];
                const uint32_t sp = SPI[r * W] & 0xffffu;
                if (sp < (uint32_t)p.S) {
                    uint32_t x = (uint32_t)X[sp], any = 0u;
                    uint32_t en[4];
                    if (kAhead && len > 0) gentries<W>(F, 0u, en);
                    for (uint32_t k = 0; k < len; k += 4) {   // len is a multiple of 4; padding adds 0
                        uint32_t e[4];
                        int32_t kc[4];
                        if (kAhead) {
#pragma unroll
                            for (int i = 0; i < 4; ++i) e[i] = en[i];
                            gentries<W>(F, k + 4 < len ? k + 4 : k, en);
                        } else {
#pragma unroll
                            for (int i = 0; i < 4; ++i) e[i] = F[(k + i) * W];
                        }
#pragma unroll
                        for (int i = 0; i < 4; ++i) kc[i] = *reinterpret_cast<const int32_t*>(Kb + (e[i] & 0xffffu));
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            x = (uint32_t)__mul24((int)(int16_t)(e[i] >> 16), kc[i]) + x;
                            any |= x;
                        }
                    }
                    X1[sp] = (int32_t)x;
                    bad = bad || (any >> 31) != 0u;
                }
                F += len * W;
            }
            if (W > 16) fired = gsum32<W>((uint32_t)f);
        } else {
            if (W > 16) fired = gsum64<W>(f);
            for (int r = 0; r < nrs; ++r) {
                const uint32_t len = TC[p.oFRm + r];
                const uint32_t sp = SPI[r * W] & 0xffffu;
                if (sp < (uint32_t)p.S) {
                    int64_t x = X[sp];
                    bool bs = false;
                    for (uint32_t k = 0; k < len; k += 4) {
                        uint32_t e[4];
                        int32_t kc[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i) e[i] = F[(k + i) * W];
#pragma unroll
                        for (int i = 0; i < 4; ++i) kc[i] = *reinterpret_cast<const int32_t*>(Kb + (e[i] & 0xffffu));
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            x += (int64_t)(int16_t)(e[i] >> 16) * (int64_t)kc[i];
                            bs = bs || x < 0 || x > 2147483647LL;
                        }
                    }
                    X1[sp] = (int32_t)x;
                    bad = bad || bs;
                }
                F += len * W;
            }
        }
        if (W <= 16) fired = gsum64<W>(f);
        const bool any_bad = gballot<W>(bad) != 0;
        gsync();
        CTL_PHASE(PH_UPDATE);
        if (!any_bad) break;
        // 277 halvings bring any tau to 0, which draws nothing, so counts within
        // [0, 2^31) pass by then.  A species that wrapped in an SSA step, or
        // was given as 2^31 or more, fails whatever is drawn: only an SSA burst
        // moves on.  (Counting this as a switch here cost 2 % at W = 64.)
        if (__builtin_expect(attempt == LEAP_ATTEMPTS, 0)) return LEAP_SWITCH;
        tau = tau * 0.5f;
    }
    // check_time_instant (T.cu:1507-1562), per sampled species
    {
        uint32_t i = L.cursor;
        const double tn = L.t + (double)tau;
        if (i < (uint32_t)p.K && tn >= p.ts[i]) {
            uint32_t* out = p.storage + (size_t)L.sim * p.K * p.SS;
            while (i < (uint32_t)p.K && tn >= p.ts[i]) {
                const double ti = p.ts[i];
                for (int sk = l; sk < p.SS; sk += W) {
                    const int sp = (int)p.T[p.oCs + sk];
                    const int32_t d = X1[sp] - X[sp];
                    uint32_t val = (uint32_t)X[sp];
                    if (d > 0) {
                        const double delta = ((double)d * (ti - L.t)) / (double)tau;
                        val += (uint32_t)rint(delta);
                    }
                    out[(size_t)i * p.SS + sk] = val;
                }
                ++i;
            }
            L.cursor = i;
        }
    }
    L.xb ^= 1u;
    if (kuse(p.nfs) > 0) {               // feeds (T.cu:2072-2079)
        int32_t* Xn = V.Xb + (L.xb ? p.S : 0);
        for (int u = l; u < p.nfs; u += W) Xn[p.fs[u]] = (int32_t)L.fvrow[u];
        gsync();
    }
    L.t = L.t + (double)tau;
    L.firings += fired;
    L.leaps++;
    CTL_PHASE(PH_SAMPLE);
    return LEAP_OK;
}

// The sampled species of state X to row (four reads in flight).
template <int W>
__device__ __forceinline__ void gsample(const KParams& p, const int32_t* X, uint32_t* row, int l) {
    for (int s0 = l; s0 < p.SS; s0 += 4 * W) {
        uint32_t sp[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) sp[i] = p.T[p.oCs + (s0 + i * W < p.SS ? s0 + i * W : s0)];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (s0 + i * W < p.SS) row[s0 + i * W] = (uint32_t)X[sp[i]];
    }
}

// Up to nmax steps of an SSA burst (EventualSSASteps T.cu:2099-2273 /
// LightweightSSA T.cu:2280-2454), opening the burst when none is in progress:
// a burst of p.ssa_steps steps may run in several calls, its clock advance,
// propensities and factor table kept meanwhile (L.tacc, L.ssa_left, the
// group's LDS), so the steps and their draws are those of one call.  After
// the fired reaction only its dependent propensities are recomputed (same
// values as recomputing all).  Returns true on absorption.
template <int G, int W, int PFM = 3>
__device__ __forceinline__ bool gssa_run(const KParams& p, GLane& L, const GView& V, int l, int nmax) {
    int32_t* X = V.Xb + (L.xb ? p.S : 0);
    const int la = l & (G - 1);              // the algorithm's lane this one stands for
    if (L.ssa_left == 0) {
        grng_event(L.gg, L.evc++);
        L.tacc = 0.0;
        L.ssa_left = p.ssa_steps;
        if (pmode<PFM>(kuse(p.pfast)) == 1) {
            gfactors<W>(p, X, V.F, l);
            gsync();
        }
        float P, PC;
        gprops<G, W, PFM>(p, X, V.F, L.crate, V.A, l, P, PC);
        gsync();
    }
    CTL_PHASE(PH_SSA_OPEN);
    double tacc = L.tacc;
    const int n = nmax < L.ssa_left ? nmax : L.ssa_left;
    const int pm = pmode<PFM>(kuse(p.pfast));
    const bool fac = pm == 1;
    const uint4* SR = reinterpret_cast<const uint4*>(p.T + p.oSR);
    const uint4* DR = reinterpret_cast<const uint4*>(p.T + p.oDR);
    double tnext = L.cursor < (uint32_t)p.K ? p.ts[L.cursor] : 0.0;        // the next sample time
    constexpr int SB = W > G || G <= 4 ? 16 : 4;
    for (int step = 0; step < n; ++step) {
        float P = 0.0f;
        const int nrp = group_rpad(p.R, G) / G;        // rounds over A with its zero padding
        for (int r0 = 0; r0 < nrp; r0 += SB) {         // padding adds an exact 0
            uint32_t u[SB];
#pragma unroll
            for (int q = 0; q < SB; q += 4)            // SB reads in flight
                if (SB == 4 || r0 + q < nrp) {
#pragma unroll
                    for (int i = q; i < q + 4; ++i) u[i] = V.A[la + (r0 + i < nrp ? r0 + i : nrp - 1) * G];
                }
#pragma unroll
            for (int q = 0; q < SB; q += 4)
                if (SB == 4 || r0 + q < nrp) {
#pragma unroll
                    for (int i = q; i < q + 4; ++i) P = P + (r0 + i < nrp ? aval(u[i]) : 0.0f);
                }
        }
        const float Pown = P;
        P = gscan<G>(P, la);
        const float a0 = gbcast_last<G>(P, la);
        const uint64_t cand = gballot<G>(Pown > 0.0f);
        if (a0 == 0.0f || cand == 0) { gabsorb<W>(p, L, X, l); L.ssa_left = 0; return true; }   // no lane: only with a NaN
        uint32_t w0, w1;
        grng_pair<W>(L.gg, l, w0, w1);
        const int j = gselect_ssa<G, W>(V.A, cand, Pown, P, u32_oc(w0) * a0, l, nrp);
        const uint4 sr = SR[j];              // {first change entry, count, first dependent, count}
        const float dt = u32_exp(w1) / a0;
        CTL_PHASE(PH_SSA_SELECT);
        tacc = tacc + (double)dt;
        const double tn = L.t + tacc;
        // this lane's first change entry and dependent: one latency for both
        uint32_t ent = 0u;
        uint4 rec = make_uint4(0u, 0u, 0u, 0u);
        const bool hasf = (uint32_t)l < sr.y, hasd = (uint32_t)l < sr.w;
        if (hasf) ent = p.T[sr.x + (uint32_t)l];
        if (pm != 0 && hasd) rec = DR[sr.z + (uint32_t)l];
        if (L.cursor < (uint32_t)p.K && tn > tnext) {                          // T.cu:2213-2236
            uint32_t i = L.cursor;
            uint32_t* out = p.storage + (size_t)L.sim * p.K * p.SS;
            while (i < (uint32_t)p.K && tn > p.ts[i]) {
                gsample<W>(p, X, out + (size_t)i * p.SS, l);
                ++i;
            }
            L.cursor = i;
            tnext = i < (uint32_t)p.K ? p.ts[i] : 0.0;
            gsync();
        }
        float c = 0.0f;
        if (pm != 0 && hasd) c = p.drate ? __uint_as_float(rec.w) : L.crate[rec.x];
        auto change = [&](uint32_t e) {      // a species occurs once per reaction
            const int s = (int)(e & 0xffffu);
            const int32_t x = (int32_t)((uint32_t)X[s] + (uint32_t)(int)(int16_t)(e >> 16));
            X[s] = x;
            if (fac) gfactor(V.F, p.S, s, x, (uint32_t)p.nc);
        };
        if (hasf) change(ent);
        for (uint32_t h = (uint32_t)l + W; h < sr.y; h += W) change(p.T[sr.x + h]);
        gsync();
        CTL_PHASE(PH_SSA_UPDATE);
        L.ssa_steps++;
        if (tn <= p.tmax) L.firings++;
        if (pm != 0) {
            auto depend = [&](const uint4& d, float a) {
                if (fac) {                   // {r, factor index 0, factor index 1, rate}
                    const uint32_t u0 = V.F[d.y], u1 = V.F[d.z];
                    a = a * __uint_as_float(u0 & 0x7fffffffu);
                    a = a * __uint_as_float(u1 & 0x7fffffffu);
                    V.A[d.x] = __float_as_uint(a) | ((u0 | u1) & 0x80000000u);
                } else {                     // {r, reactant entry 0, entry 1, rate} read from the state
                    bool crit = false;
                    gtwo(a, crit, X[d.y & 0xffffu], d.y >> 16, X[d.z & 0xffffu], d.z >> 16, (uint32_t)p.nc);
                    V.A[d.x] = __float_as_uint(a) | (crit ? 0x80000000u : 0u);
                }
            };
            if (hasd) depend(rec, c);
            for (uint32_t d = (uint32_t)l + W; d < sr.w; d += W) {
                const uint4 q = DR[sr.z + d];
                depend(q, p.drate ? __uint_as_float(q.w) : L.crate[q.x]);
            }
        } else {
            for (uint32_t d = (uint32_t)l; d < sr.w; d += W) {
                const int r = (int)p.T[p.oDe + sr.z + d];
                bool crit;
                const float a = gprop(p, X, L.crate, r, crit);
                V.A[r] = __float_as_uint(a) | (crit ? 0x80000000u : 0u);
            }
        }
        gsync();
        CTL_PHASE(PH_SSA_DEPS);
    }
    L.ssa_left -= n;
    L.tacc = tacc;
    if (L.ssa_left == 0) {
        L.t = L.t + tacc;
        L.tacc = 0.0;
    }
    return false;
}

// One whole SSA burst.
template <int G, int W, int PFM = 3>
__device__ __forceinline__ bool gssa(const KParams& p, GLane& L, const GView& V, int l) {
    L.ssa_left = 0;
    return gssa_run<G, W, PFM>(p, L, V, l, p.ssa_steps);
}

__device__ __forceinline__ const float* grates(const KParams& p, int sim) {
    return p.c_bcast ? p.c_bcast : p.c_sims + (size_t)(sim / p.c_div) * p.R;
}

// Next simulation from the queue (PrepareVariables, T.cu:1269-1297).
template <int W>
__device__ __forceinline__ bool gfetch(const KParams& p, GLane& L, const GView& V, int l) {
    uint32_t q = 0;
    if (l == 0) q = atomicAdd(p.next_sim, 1u);
    q = __shfl(q, 0, W);
    if (q >= (uint32_t)p.n) { L.sim = -2; return false; }
    L.sim = (int)q;
    L.t = 0.0;
    L.tacc = 0.0;
    L.ssa_left = 0;
    L.ssa_mode = kuse(p.force_ssa);
    L.cursor = 0;
    L.evc = 0;
    L.xb = 0;
    L.firings = L.ssa_steps = 0;
    L.leaps = L.rejections = L.switches = L.absorbed = 0;
    L.poisson = L.gaps = 0;
    L.gg.sim = L.lg.sim = p.sim_base + q;
    L.gg.cb = GRNG_NONE;
    L.lg.pos = 4;
    for (int s = l; s < p.S; s += W)
        V.Xb[s] = (int32_t)(p.x0_bcast ? p.x0_bcast[s] : p.x0_sims[(size_t)(q / (uint32_t)p.x0_div) * p.S + s]);
    L.crate = grates(p, (int)q);
    L.fvrow = p.nfs > 0 ? p.fv + (size_t)(q / (uint32_t)p.fv_div) * p.nfs : nullptr;
    gsync();
    return true;
}

template <int W>
__device__ __forceinline__ void gfinish(const KParams& p, GLane& L, const GView& V, int l) {
    const int32_t* X = V.Xb + (L.xb ? p.S : 0);
    const uint64_t pois = gsum64<W>(L.poisson);
    const uint64_t gaps = gsum64<W>(L.gaps);
    for (int s = l; s < p.S; s += W) p.xfinal[(size_t)L.sim * p.S + s] = X[s];
    if (l == 0) {
        ctl_sim_stat st;
        st.firings = L.firings;
        st.ssa_steps = L.ssa_steps;
        st.poisson = pois;
        st.gaps = gaps;
        st.t_end = L.t;
        st.leaps = L.leaps;
        st.rejections = L.rejections;
        st.switches = L.switches;
        st.events = L.evc;
        st.absorbed = L.absorbed;
        st.reserved = 0;
        p.simstat[L.sim] = st;
        p.tfinal[L.sim] = L.t;
        atomicAdd(p.done, 1u);
    }
    L.sim = -1;
}

// Longest a switched group waits for the bursts of the wavefront's other
// groups (leap iterations).  A burst of 100 steps idles every group that is
// not in one, so they gather: when one has waited this long, or all have
// switched, all that have switched run theirs.  Going as soon as two had
// switched cost more the more groups share the wavefront.  Kernel times in ms,
// two or 24 / all or 4 / 6 / 10 / 16 / 28:
//   100x200 network, 4 groups, t = 50      1250 / 1206 / 1184 / 1161 / 1176 / 1247
//   50x100 network, 8 groups, t = 0.2       417 /  284 /  268 /  258 /  267 /  288
//   50x100 sweep network, 8 groups          408 /  325 /  320 /  318 /  316 /  318
//   20-stage cascade, 16 groups            20.2 / 18.5 / 18.4 / 18.5 / 18.5 / 18.5
constexpr int GBURST_WAIT = 10;

// ---------------------------------------------------------------------------
// Regrouping groups by mode.  The groups of a wavefront run in lockstep: while
// one group runs SSA steps the wavefront's leaping groups wait, and the
// other way round.  With p.compact > 0 a workgroup's group slots ("regions":
// a simulation's LDS state and its global slot) are reassigned to the
// workgroup's wavefronts every p.compact iterations, leap-mode regions first,
// SSA-mode ones next, regions without a simulation last, so that each
// wavefront runs one mode.  SSA bursts then run in chunks of p.ssa_chunk steps
// per iteration, comparable to a leap.  A region's simulation keeps its LDS
// state; its registers travel
// through the slot arrays in global memory (the parking format).  No event of
// any simulation changes: only which lanes run it.
// ---------------------------------------------------------------------------

// Writes the group's registers to the slot arrays of its region's slot s0.
template <int W>
__device__ __forceinline__ void gstage_put(const KParams& p, const GLane& L, int s0, int l) {
    p.st->poisson[(size_t)s0 * W + l] = L.poisson;
    p.st->gaps[(size_t)s0 * W + l] = L.gaps;
    if (l == 0) {
        p.st->sim[s0] = L.sim;
        p.st->t[s0] = L.t;
        p.st->tacc[s0] = L.tacc;
        p.st->cursor[s0] = L.cursor;
        p.st->ssa_left[s0] = L.ssa_left;
        p.st->mode[s0] = L.ssa_mode;
        p.st->evc[s0] = L.evc;
        p.st->xb[s0] = L.xb;
        p.st->firings[s0] = L.firings;
        p.st->ssa_steps[s0] = L.ssa_steps;
        p.st->leaps[s0] = L.leaps;
        p.st->rejections[s0] = L.rejections;
        p.st->switches[s0] = L.switches;
        p.st->ev[s0] = L.gg.ev;
        p.st->blk[s0] = L.gg.wc;      // words of the event consumed
    }
}

// Takes over the simulation of slot s0: its registers, rate and feed rows and
// the position in its group stream.
template <int W>
__device__ __forceinline__ void gstage_get(const KParams& p, GLane& L, int s0, int l) {
    L.sim = p.st->sim[s0];
    L.poisson = p.st->poisson[(size_t)s0 * W + l];
    L.gaps = p.st->gaps[(size_t)s0 * W + l];
    L.absorbed = 0;
    if (L.sim < 0) return;
    L.t = p.st->t[s0];
    L.tacc = p.st->tacc[s0];
    L.cursor = p.st->cursor[s0];
    L.ssa_left = p.st->ssa_left[s0];
    L.ssa_mode = p.st->mode[s0];
    L.evc = p.st->evc[s0];
    L.xb = p.st->xb[s0];
    L.firings = p.st->firings[s0];
    L.ssa_steps = p.st->ssa_steps[s0];
    L.leaps = p.st->leaps[s0];
    L.rejections = p.st->rejections[s0];
    L.switches = p.st->switches[s0];
    L.gg.ev = p.st->ev[s0];
    L.gg.wc = p.st->blk[s0];
    L.gg.cb = GRNG_NONE;                 // the blocks are regenerated at the next word
    L.gg.sim = L.lg.sim = p.sim_base + (uint32_t)L.sim;
    L.crate = grates(p, L.sim);
    L.fvrow = p.nfs > 0 ? p.fv + (size_t)(L.sim / p.fv_div) * p.nfs : nullptr;
}

// Stable partition of the workgroup's regions by key (0 leap, 1 SSA, 2
// none); cnt: 3 words per wavefront, perm: one word per region.  Every lane
// of the workgroup must call it.  Returns false, with no other effect, when
// no region of the workgroup holds a simulation; else the new region of
// this lane's group in *next and whether any region moves to other lanes in
// *moves (the same for the whole workgroup).
template <int W>
__device__ __forceinline__ bool gregroup(int key, int reg, uint32_t* cnt, uint32_t* perm, int l, int* next,
                                         bool* moves) {
    const int lane = (int)(threadIdx.x & 63u), wave = (int)(threadIdx.x >> 6), nw = (int)(blockDim.x >> 6);
    const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    uint32_t rank = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const uint64_t b = __ballot(l == 0 && key == k);      // one bit per group (its lane 0)
        if (key == k) rank = (uint32_t)__popcll(b & lt);
        if (lane == 0) cnt[wave * 3 + k] = (uint32_t)__popcll(b);
    }
    __syncthreads();
    uint32_t active = 0, pos = 0;
    for (int w = 0; w < nw; ++w) active += cnt[w * 3] + cnt[w * 3 + 1];
    if (active == 0) return false;
    for (int k = 0; k < key; ++k)
        for (int w = 0; w < nw; ++w) pos += cnt[w * 3 + k];
    for (int w = 0; w < wave; ++w) pos += cnt[w * 3 + key];
    if (l == 0) perm[pos + rank] = (uint32_t)reg;
    __syncthreads();
    const int nreg = (int)(blockDim.x / W);
    bool mv = false;
    for (int q = 0; q < nreg; ++q) mv = mv || perm[q] != (uint32_t)q;
    *moves = mv;
    *next = (int)perm[threadIdx.x / W];
    return true;
}

// Waves per SIMD the group kernels are compiled for.  W = G: G = 8, 16 and 32
// for four (128 VGPRs, a few bytes of scratch), measured +9 % at G = 16 and
// +4 % at G = 32 on the 100x200 network, +24 % at G = 8 on the 50x100 sweep
// network; G = 64 would spill heavily.  G = 2 and 4 hold three by themselves
// except in mode 1 (174 VGPRs, where three waves have 168 each) and, with
// regrouping, in mode 2 (170): up to two spilled registers there give the
// third wave back (mode 1, 14 species and 40 reactions, 262144 simulations,
// two / three: adaptive 35.6 / 26.4 ms, force-SSA 29.6 / 21.0; mode 2 with
// regrouping every 8, 22 species and 24 reactions, G = 4: 8.4 / 6.5, 97 / 72;
// larger models are bounded by LDS).  W > G serves runs that leave the chip
// short of wavefronts.
__host__ __device__ constexpr int gwaves(int G, int W, int PFM = 3, bool RG = false) {
    const bool spill = PFM == 1 || (PFM == 2 && RG);
    return W > G ? (W == 64 ? 2 : 4) : (G == 8 || G == 16 || G == 32 ? 4 : (G <= 4 && spill ? 3 : 1));
}

// Persistent group kernel: p.ns lanes = p.ns / W group slots, each pulling
// simulations from the queue; a launch runs up to p.iters iterations per
// group (a leap attempt, or SSA steps), then parks the group's state in the
// slot arrays for the next launch.  Without regrouping (RG false: W = 64, or
// p.compact = 0) a group that switched to SSA holds its whole burst until one
// has waited GBURST_WAIT iterations or every group of the wavefront still
// running has switched, so that bursts run side by side.  Either way each simulation's events and draws are its own;
// only the order in which the lanes serve the simulations moves.
template <int G, int W, bool RG, int PF>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(gwaves(G, W, PF, RG)))) void group_kernel(KParams p) {
    extern __shared__ uint32_t smem[];
    __shared__ float recip[64];
    __shared__ uint32_t rg_cnt[12];
    __shared__ uint32_t rg_perm[256 / W];
    for (int i = threadIdx.x; i < 64; i += blockDim.x) recip[i] = c_recip[i];
    __syncthreads();
    const int l = (int)(threadIdx.x & (unsigned)(W - 1));
    const int nreg = (int)(blockDim.x / W);
    int gib = (int)(threadIdx.x / W);
    const size_t gw = group_lds_words(p.S, p.R, G);
    constexpr bool rg = RG && W < 64;     // the host launches RG only with p.compact > 0 and several wavefronts
    GLane L;
    L.slot = (int)blockIdx.x * nreg + gib;
    CTL_PHASE_START();
    if (L.slot * W >= p.ns) return;                  // whole workgroups when regrouping
    GView V = group_view(smem + (size_t)gib * gw, p.S, p.R, G);
    gzero_pad<G, W>(V, p.R, l);
    L.gg.k0 = L.lg.k0 = p.key0;
    L.gg.k1 = L.lg.k1 = p.key1;
    L.lg.tag = 1u + (uint32_t)(l & (G - 1));
    L.tacc = 0.0;
    L.ssa_left = 0;
    L.ssa_mode = 0;
    L.sim = p.st->sim[L.slot];
    if (L.sim == -2 && !rg) {
        CTL_PHASE(PH_PARK);
        CTL_PHASE_FLUSH();
        return;
    }
    if (L.sim >= 0) {                    // resume a parked simulation
        const int s0 = L.slot;
        L.t = p.st->t[s0];
        L.cursor = p.st->cursor[s0];
        L.evc = p.st->evc[s0];
        L.xb = 0;
        L.firings = p.st->firings[s0];
        L.ssa_steps = p.st->ssa_steps[s0];
        L.leaps = p.st->leaps[s0];
        L.rejections = p.st->rejections[s0];
        L.switches = p.st->switches[s0];
        L.absorbed = 0;
        L.ssa_mode = kuse(p.force_ssa);
        L.poisson = p.st->poisson[(size_t)s0 * W + l];
        L.gaps = p.st->gaps[(size_t)s0 * W + l];
        L.gg.sim = L.lg.sim = p.sim_base + (uint32_t)L.sim;
        L.gg.cb = GRNG_NONE;
        L.lg.pos = 4;
        for (int s = l; s < p.S; s += W) V.Xb[s] = p.X[(size_t)s0 * p.S + s];
        L.crate = grates(p, L.sim);
        L.fvrow = p.nfs > 0 ? p.fv + (size_t)(L.sim / p.fv_div) * p.nfs : nullptr;
        gsync();
    }
    bool pend = false;
    int waited = 0;
    for (int it = 0; it < p.iters; ++it) {
        CTL_PHASE(PH_LOOP);
        if (rg) {
            if (it % p.compact == 0) {
                // 0: leap (or about to take a simulation), 1: SSA, 2: no simulation left
                const int key = L.sim == -2 ? 2 : (L.sim >= 0 ? L.ssa_mode : kuse(p.force_ssa));
                int ng;
                bool moves;
                if (!gregroup<W>(key, gib, rg_cnt, rg_perm, l, &ng, &moves)) break;
                // a group whose region stays on its lanes keeps its registers;
                // the others hand their state over through the slot arrays
                if (moves) {
                    const bool move = ng != gib;
                    if (move) gstage_put<W>(p, L, L.slot, l);
                    __syncthreads();
                    if (move) {
                        gib = ng;
                        L.slot = (int)blockIdx.x * nreg + gib;
                        gstage_get<W>(p, L, L.slot, l);
                        V = group_view(smem + (size_t)gib * gw, p.S, p.R, G);
                    }
                }
                CTL_PHASE(PH_REGROUP);
            }
            if (L.sim == -2) continue;
            if (L.sim < 0 && !gfetch<W>(p, L, V, l)) continue;
            if (L.ssa_mode) {
                CTL_PHASE(PH_PRE_SSA);
                if (kuse(p.force_ssa) && L.ssa_left == 0 && L.t >= p.tmax) {
                    gfinish<W>(p, L, V, l);
                } else if (gssa_run<G, W, PF>(p, L, V, l, p.ssa_chunk)) {
                    gfinish<W>(p, L, V, l);
                } else if (L.ssa_left == 0 && !kuse(p.force_ssa)) {
                    L.ssa_mode = 0;
                }
            } else {
                CTL_PHASE(PH_PRE_LEAP);
                const int r = gleap<G, W, PF>(p, L, V, l, recip);
                if (r == LEAP_DONE || r == LEAP_ABSORB) {
                    gfinish<W>(p, L, V, l);
                } else if (r == LEAP_SWITCH) {
                    L.ssa_mode = 1;
                }
            }
            continue;
        }
        if (L.sim < 0 && !gfetch<W>(p, L, V, l)) break;
        if (kuse(p.force_ssa)) {
            if (L.t >= p.tmax || gssa<G, W, PF>(p, L, V, l)) gfinish<W>(p, L, V, l);
            continue;
        }
        if (!pend) {
            CTL_PHASE(PH_PRE_LEAP);
            const int r = gleap<G, W, PF>(p, L, V, l, recip);
            if (r == LEAP_DONE || r == LEAP_ABSORB) {
                gfinish<W>(p, L, V, l);
            } else if (r == LEAP_SWITCH) {
                pend = true;
                waited = 0;
            }
        } else {
            ++waited;
        }
        bool go = pend;
        if (W < 64) {
            const uint64_t lead = __ballot(l == 0);            // groups still in the loop
            const uint64_t pm = __ballot(pend && l == 0);       // ... waiting for a burst
            go = pm != 0 && (pm == lead || __ballot(pend && waited >= GBURST_WAIT) != 0);
        }
        if (go && pend) {
            pend = false;
            CTL_PHASE(PH_PRE_SSA);
            if (gssa<G, W, PF>(p, L, V, l)) gfinish<W>(p, L, V, l);
        }
    }
    // before parking: the burst of a switched simulation runs to its end (a
    // parked simulation resumes with a leap attempt, or with a new burst in
    // force-SSA mode)
    if (rg) {
        if (L.sim >= 0 && (L.ssa_left > 0 || (L.ssa_mode && !kuse(p.force_ssa))) &&
            gssa_run<G, W, PF>(p, L, V, l, L.ssa_left > 0 ? L.ssa_left : p.ssa_steps))
            gfinish<W>(p, L, V, l);
    } else if (pend && gssa<G, W, PF>(p, L, V, l)) {
        gfinish<W>(p, L, V, l);
    }
    const int s0 = L.slot;
    if (L.sim >= 0) {                    // park: state to the slot arrays
        const int32_t* X = V.Xb + (L.xb ? p.S : 0);
        for (int s = l; s < p.S; s += W) p.X[(size_t)s0 * p.S + s] = X[s];
        p.st->poisson[(size_t)s0 * W + l] = L.poisson;
        p.st->gaps[(size_t)s0 * W + l] = L.gaps;
        if (l == 0) {
            p.st->t[s0] = L.t;
            p.st->cursor[s0] = L.cursor;
            p.st->evc[s0] = L.evc;
            p.st->firings[s0] = L.firings;
            p.st->ssa_steps[s0] = L.ssa_steps;
            p.st->leaps[s0] = L.leaps;
            p.st->rejections[s0] = L.rejections;
            p.st->switches[s0] = L.switches;
        }
    }
    if (l == 0) p.st->sim[s0] = L.sim;
    CTL_PHASE(PH_PARK);
    CTL_PHASE_FLUSH();
}

// Host: propensity mode (pmode) of a model at G lanes: with at most two
// reactant entries of multiplicity <= 2 per reaction, two table entries per
// reaction -- factor indices (1) when the factor table fits in the Kc region,
// free outside the count and update phases, else species | multiplicity read
// from the state (2): a separate table would enlarge every group's LDS and
// cost occupancy (the enzyme cascade, 61 species and 60 reactions at G = 4,
// ran 20 % slower with one).
inline int group_pmode(const Model& m, int G) {
    bool two = true;
    for (int j = 0; j < m.R; ++j) {
        if (m.Lptr[j + 1] - m.Lptr[j] > 2) two = false;
        for (uint32_t h = m.Lptr[j]; h < m.Lptr[j + 1]; ++h)
            if ((m.Lent[h] >> 16) > 2) two = false;
    }
    return !two ? 0 : (2 * m.S + 1 <= group_rpad(m.R, G) ? 1 : 2);
}

// Host: appends the lane-interleaved round streams (KParams::oPRm ..) of a
// group kernel with G lanes to the packed table buffer T.
inline void append_group_streams(std::vector<uint32_t>& T, KParams& p, int G, int W, const Model& m,
                                 const std::vector<uint32_t>& FSptr, const std::vector<uint32_t>& FSent,
                                 const std::vector<uint32_t>& Dptr, const std::vector<uint32_t>& Dent) {
    // Item order[r * B + l] (-1: none) goes to lane l of round r of B lanes.  fixed > 0:
    // every round has exactly that many entries per lane; else the round's
    // longest list rounded up to a multiple of quantum.
    auto rounds = [&](int B, const std::vector<int>& order, const std::vector<uint32_t>& ptr,
                      const std::vector<uint32_t>& ent, int& om, int& oe, uint32_t quantum, uint32_t fixed,
                      uint32_t pad) {
        const int nr = (int)(order.size() / (size_t)B);
        auto cnt = [&](int i) { return i < 0 ? 0u : ptr[i + 1] - ptr[i]; };
        std::vector<uint32_t> len((size_t)nr, 0u), e;
        for (int r = 0; r < nr; ++r) {
            uint32_t mx = 0;
            for (int l = 0; l < B; ++l) mx = std::max(mx, cnt(order[(size_t)r * B + l]));
            mx = fixed ? fixed : (mx + quantum - 1) / quantum * quantum;
            len[r] = mx;
            for (uint32_t k = 0; k < mx; ++k)
                for (int l = 0; l < B; ++l) {
                    const int i = order[(size_t)r * B + l];
                    e.push_back(k < cnt(i) ? ent[ptr[i] + k] : pad);
                }
        }
        om = (int)T.size();
        T.insert(T.end(), len.begin(), len.end());
        oe = (int)T.size();
        T.insert(T.end(), e.begin(), e.end());
    };
    p.pfast = group_pmode(m, G);
    std::vector<int> rorder((size_t)((m.R + G - 1) / G) * G, -1);
    for (int j = 0; j < m.R; ++j) rorder[j] = j;          // reaction j: lane j mod G (the selection's partials)
    // pfast: a reactant entry becomes its index in the factor table F
    // (multiplicity 1: s, 2: S + s; padding: 2S, the constant 1.0)
    const uint32_t one = (uint32_t)(2 * m.S);
    auto findex = [&](uint32_t e) { const uint32_t v = e >> 16, sp = e & 0xffffu;
                                    return v == 1u ? sp : (v == 2u ? (uint32_t)m.S + sp : one); };
    if (p.pfast == 1) {
        std::vector<uint32_t> fent(m.Lent.size());
        for (size_t h = 0; h < m.Lent.size(); ++h) fent[h] = findex(m.Lent[h]);
        rounds(G, rorder, m.Lptr, fent, p.oPRm, p.oPRe, 1, 2, one);
    } else {
        rounds(G, rorder, m.Lptr, m.Lent, p.oPRm, p.oPRe, 1, p.pfast == 2 ? 2 : 0, 0u);
    }
    while (T.size() % 4) T.push_back(0u);   // per reaction {first change entry, count, first dependent, count}
    p.oSR = (int)T.size();
    for (int j = 0; j < m.R; ++j) {
        T.push_back((uint32_t)p.oFe + m.Fptr[j]);
        T.push_back(m.Fptr[j + 1] - m.Fptr[j]);
        T.push_back(Dptr[j]);
        T.push_back(Dptr[j + 1] - Dptr[j]);
    }
    p.oDR = p.oSR;
    p.drate = m.c_rows == 1;
    if (p.pfast) {                        // dependent records
        p.oDR = (int)T.size();
        for (uint32_t r : Dent) {       // factor indices (mode 1) or the entries themselves (mode 2)
            const uint32_t n = m.Lptr[r + 1] - m.Lptr[r];
            const uint32_t e0 = n > 0 ? m.Lent[m.Lptr[r]] : 0u, e1 = n > 1 ? m.Lent[m.Lptr[r] + 1] : 0u;
            T.push_back(r);
            T.push_back(p.pfast == 1 ? (n > 0 ? findex(e0) : one) : e0);
            T.push_back(p.pfast == 1 ? (n > 1 ? findex(e1) : one) : e1);
            T.push_back(p.drate ? __builtin_bit_cast(uint32_t, (float)m.c[r]) : 0u);
        }
    }
    // species by entry count, longest first, so that a round's lanes carry
    // lists of similar length (tau' is a minimum and the update is per
    // species, so the species-to-lane map is free)
    std::vector<int> sorder((size_t)((m.S + W - 1) / W) * W, -1);
    for (int i = 0; i < m.S; ++i) sorder[i] = i;
    std::stable_sort(sorder.begin(), sorder.begin() + m.S, [&](int a, int b) {
        return std::max(m.Vptr[a + 1] - m.Vptr[a], FSptr[a + 1] - FSptr[a]) >
               std::max(m.Vptr[b + 1] - m.Vptr[b], FSptr[b + 1] - FSptr[b]);
    });
    p.oSPI = (int)T.size();
    p.gsimple = 1;
    for (int i = 0; i < m.S; ++i)
        if (m.hor[i] >= 3 || (m.hor[i] == 2 && m.hort[i] == 2)) p.gsimple = 0;
    for (int i : sorder)
        T.push_back(i < 0 ? 0xffffffffu
                          : (uint32_t)i | ((uint32_t)m.hor[i] << 16) | ((uint32_t)m.hort[i] << 24));
    // var entries: with every |coefficient| <= 2048 (exact in FP16, v * v exact
    // in FP32) and A's byte offsets below 2^16, as FP16 coefficient << 16 |
    // byte offset of A[reaction]; else reaction | v << 16
    p.vhalf = 4 * (m.R + 1) <= 0xffff ? 2 : 0;
    for (uint32_t e : m.Vent) {
        const int v = (int)(int16_t)(e >> 16);
        if (v > 2048 || v < -2048) p.vhalf = 0;
        else if ((v & -v) != v && ((-v) & v) != -v && p.vhalf) p.vhalf = 1;
    }
    if (p.vhalf) {
        std::vector<uint32_t> vent(m.Vent.size());
        for (size_t h = 0; h < m.Vent.size(); ++h) {
            const _Float16 hv = (_Float16)(float)(int16_t)(m.Vent[h] >> 16);
            vent[h] = (uint32_t)__builtin_bit_cast(uint16_t, hv) << 16 | (m.Vent[h] & 0xffffu) * 4u;
        }
        rounds(W, sorder, m.Vptr, vent, p.oVRm, p.oVRe, 4, 0, (uint32_t)m.R * 4u);   // padding: A[R] = 0
    } else {
        rounds(W, sorder, m.Vptr, m.Vent, p.oVRm, p.oVRe, 4, 0, (uint32_t)m.R);       // padding: the zero slot A[R]
    }
    // change entries as byte offset of Kc[reaction] (R <= 8191: a group's LDS
    // holds 16384 words) | change << 16; flim: firings of a leap below which
    // the update's sums fit 32 bits (0: never, a count may be negative)
    std::vector<uint32_t> fent(FSent.size());
    int vmax = 1;
    for (size_t h = 0; h < FSent.size(); ++h) {
        vmax = std::max(vmax, std::abs((int)(int16_t)(FSent[h] >> 16)));
        fent[h] = (FSent[h] & 0xffff0000u) | (FSent[h] & 0xffffu) * 4u;
    }
    p.flim = plain_values(m) ? std::min(1u << 23, (1u << 30) / (uint32_t)vmax) : 0u;
    rounds(W, sorder, FSptr, fent, p.oFRm, p.oFRe, 4, 0, 0u);
}

}  // namespace ctl
