// ctl_small.h -- the one-lane kernel for small models: one lane runs one
// simulation with everything a step reads in LDS.  Included by ctl_sim.hip.
//
// A simulation is one chain of dependent steps, so a run is bound by the
// latency of a step: a read of LDS takes 26 ns, a global load at a per-lane
// index 50 to 60 ns, a taken branch about 20 ns, a dependent FP32 operation
// 2.7 ns (measured; one wavefront).  Hence
//   * the tables that are read at per-lane indices (the fired reaction's
//     change list and dependents, the dependents' reactants) are copied to
//     LDS, species and propensities already as byte offsets of the lane's
//     words;
//   * a propensity is a product of table entries: F1 = x, F2 = x (x - 1) / 2,
//     G2 = (x - 1) / 2 and G3 = (x - 2) / 3 per species (0 where the count is
//     below the multiplicity), F1, F2 and G3 with the criticality of
//     multiplicity 1, 2 and 3 in bit 31.  Multiplicity 1 is F1, 2 is F2, 3 is
//     P1 (x without the bit), G2, G3 in turn: prop_one's factors in its order.  A step rebuilds the entries of the one
//     to three species it changed;
//   * the reads of four dependents, or of a batch of terms of a sum, are in
//     flight together, and the arithmetic selects instead of branching;
//   * few simulations are spread over many wavefronts (KParams::lpw lanes of
//     each hold one): lanes of one wavefront in different modes run one after
//     the other.
// Every value, draw and sum is the one of leap / ssa_steps.  Schlogl, one
// wavefront: 2.8 us an SSA step with global tables, 1.36 us with these; 1024
// adaptive simulations to t = 10: 119 -> 52 ms.
//
// Table (words from T[oST]): R records {factor 0 | factor 1 << 16, factor 2 |
// factor 3 << 16, change list | length << 16, dependents | padded length << 16};
// the change entries (species | change << 16); the dependents, each list padded
// with its last reaction to a multiple of 4.  A factor is an index into the
// lane's factor words (kind * S + species; snf * S: the constant 1).  The copy
// in LDS holds byte offsets instead of indices: a dependent as record offset |
// propensity offset << 16.
//
// LDS of a workgroup (one wavefront, B = lpw lanes): the table, the shared
// rates (R words), then [word][lane]: X S, X1 S, A Rp (R rounded up to the
// batch RB, zero past R), factors snf S + 1, and the rates R when they differ.
#pragma once

#include "ctl_kernels.h"

#pragma clang fp contract(off)

namespace ctl {

typedef __attribute__((address_space(3))) uint32_t lds_word;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) u32x2 lds_word2;
typedef __attribute__((address_space(3))) u32x4 lds_word4;

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(size_t)(const lds_word*)p;
}
__device__ __forceinline__ uint32_t lget(uint32_t a) { return *(const lds_word*)(size_t)a; }
__device__ __forceinline__ u32x2 lget2(uint32_t a) { return *(const lds_word2*)(size_t)a; }
__device__ __forceinline__ u32x4 lget4(uint32_t a) { return *(const lds_word4*)(size_t)a; }
__device__ __forceinline__ void lput(uint32_t a, uint32_t v) { *(lds_word*)(size_t)a = v; }

// Batch of terms of a sum, to which R is padded.
__host__ __device__ constexpr int small_batch(int R) { return R <= 4 ? 4 : 8; }
__host__ __device__ inline int small_words(int S, int R, int snf, bool shared_rates) {
    const int b = small_batch(R);
    return 2 * S + (R + b - 1) / b * b + snf * S + 1 + (shared_rates ? 0 : R);
}

// LDS byte addresses of one lane's arrays.
struct SmallView {
    uint32_t tab, rates;     // table; rates: shared, or the lane's own
    uint32_t x, a, f;        // state buffer 0, propensities, factors
    uint32_t st;             // bytes between consecutive words of a lane (4 B)
    uint32_t sx;             // bytes between the two state buffers
    bool shared;             // one rate row for every simulation
};

// The factor words of one species with count x.
__device__ __forceinline__ void small_factor(const KParams& p, const SmallView& Z, uint32_t f, int32_t x) {
    const uint32_t ncm1 = p.nc > 0 ? (uint32_t)(p.nc - 1) : 0u;
    const float xf = (float)x;
    const float xm = (float)(x - 1);
    const float f2 = (x < 2) ? 0.0f : (0.5f * xf) * xm;
    // critical at multiplicity v: v <= x < nc v
    const uint32_t c1 = (uint32_t)(x - 1) < ncm1 ? 0x80000000u : 0u;
    const uint32_t c2 = (uint32_t)(x - 2) < 2u * ncm1 ? 0x80000000u : 0u;
    lput(f, __float_as_uint(xf) | c1);
    lput(f + Z.sx, __float_as_uint(f2) | c2);
    if (p.snf > 2) {                         // P1, G2, G3
        const uint32_t c3 = (uint32_t)(x - 3) < 3u * ncm1 ? 0x80000000u : 0u;
        const float g2 = x < 1 ? 0.0f : 0.5f * xm;
        // (x - 2) / 3, correctly rounded: one Newton step on the remainder
        // (equal to the division for every FP32 significand)
        const float n = x < 3 ? 0.0f : (float)(x - 2);
        const float q = n * 0x1.555556p-2f;
        const float g3 = fmaf(fmaf(-3.0f, q, n), 0x1.555556p-2f, q);
        lput(f + 2 * Z.sx, __float_as_uint(xf));
        lput(f + 3 * Z.sx, __float_as_uint(g2));
        lput(f + 4 * Z.sx, __float_as_uint(g3) | c3);
    }
}

// The propensity bits (| critical << 31) of four reactions: record addresses
// rec, rate addresses ra.
__device__ __forceinline__ void small_props(const KParams& p, const SmallView& Z, const uint32_t (&rec)[4],
                                            const uint32_t (&ra)[4], uint32_t (&u)[4]) {
    u32x2 e[4];
    uint32_t f0[4], f1[4], f2[4], f3[4], c[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        e[i] = lget2(rec[i]);
        c[i] = lget(ra[i]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f0[i] = lget(Z.f + (e[i].x & 0xffffu));
        f1[i] = lget(Z.f + (e[i].x >> 16));
        if (p.snf > 2) {
            f2[i] = lget(Z.f + (e[i].y & 0xffffu));
            f3[i] = lget(Z.f + (e[i].y >> 16));
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float a = __uint_as_float(c[i]);
        a = a * aval(f0[i]);
        a = a * aval(f1[i]);
        uint32_t s = f0[i] | f1[i];
        if (p.snf > 2) {
            a = a * aval(f2[i]);
            a = a * aval(f3[i]);
            s |= f2[i] | f3[i];
        }
        u[i] = __float_as_uint(a) | (s & 0x80000000u);
    }
}

// One adaptive leap attempt (leap): propensities and tau' from the tables, the
// rest as every one-lane kernel does it.
__device__ __forceinline__ int leap_small(const KParams& p, Lane& L, const View& V, const SmallView& Z,
                                          const float* __restrict__ recip) {
    if (L.t >= p.tmax) return LEAP_DONE;
    const uint32_t x = Z.x + (L.xb ? Z.sx : 0u);
    for (int s = 0; s < p.S; ++s) small_factor(p, Z, Z.f + s * Z.st, (int32_t)lget(x + s * Z.st));
    float a0 = 0.0f, a0c = 0.0f;
    for (int r0 = 0; r0 < p.R; r0 += 4) {
        uint32_t rec[4], ra[4], u[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t r = (uint32_t)(r0 + i < p.R ? r0 + i : p.R - 1);
            rec[i] = Z.tab + 16u * r;
            ra[i] = Z.rates + r * (Z.shared ? 4u : Z.st);
        }
        small_props(p, Z, rec, ra, u);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t r = (uint32_t)(r0 + i < p.R ? r0 + i : p.R - 1);
            lput(Z.a + r * Z.st, u[i]);
            const float a = r0 + i < p.R ? aval(u[i]) : 0.0f;
            a0 = a0 + a;
            a0c = a0c + ((u[i] & 0x80000000u) ? a : 0.0f);
        }
    }
    int32_t* X = xcur(V, L);
    if (a0 == 0.0f) { absorb(p, L, V, X); return LEAP_ABSORB; }
    float tau1 = 3.40282347e+38f;            // T.cu:1860-1922, as in leap
    for (int sp = 0; sp < p.S; ++sp) {
        const uint32_t h0 = CT_U32(p.Vptr)[sp], h1 = CT_U32(p.Vptr)[sp + 1];
        if (h0 == h1) continue;
        float mu = 0.0f, sg = 0.0f;
        for (uint32_t h = h0; h < h1; h += 4) {
            uint32_t e[4], u[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) e[i] = CT_U32(p.Vent)[h + i < h1 ? h + i : h1 - 1];
#pragma unroll
            for (int i = 0; i < 4; ++i) u[i] = lget(Z.a + (e[i] & 0xffffu) * Z.st);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int v = (int)(int16_t)(e[i] >> 16);
                // a critical reaction and the filling add an exact zero
                const float a = (u[i] & 0x80000000u) || h + i >= h1 ? 0.0f : __uint_as_float(u[i]);
                mu = mu + (float)v * a;
                sg = sg + (float)(v * v) * a;
            }
        }
        const int32_t xs = (int32_t)lget(x + sp * Z.st);
        const float gg = gfun(CT_U32(p.horw)[sp], xs);
        const float tmp2 = (p.eps * (float)xs) / gg;
        const float macs = tmp2 > 1.0f ? tmp2 : 1.0f;
        const float t3 = macs / fabsf(mu);
        const float t4 = (macs * macs) / sg;
        const float tmp = t3 < t4 ? t3 : t4;
        if (mu != 0.0f && sg != 0.0f && tmp < tau1) tau1 = tmp;
    }
    return leap_from_tau(p, L, V, recip, X, tau1, a0, a0c);
}

// Running sums of the propensities in reaction order: the first RB in s, the
// total returned (the zero padding adds an exact 0).
template <int RB>
__device__ __forceinline__ float small_prefix(const KParams& p, const SmallView& Z, float (&s)[RB]) {
    uint32_t u[RB];
    float acc = 0.0f;
#pragma unroll
    for (int i = 0; i < RB; ++i) u[i] = lget(Z.a + i * Z.st);
#pragma unroll
    for (int i = 0; i < RB; ++i) {
        acc = acc + aval(u[i]);
        s[i] = acc;
    }
    if constexpr (RB > 4)
        for (int r0 = RB; r0 < p.R; r0 += RB) {
#pragma unroll
            for (int i = 0; i < RB; ++i) u[i] = lget(Z.a + (r0 + i) * Z.st);
#pragma unroll
            for (int i = 0; i < RB; ++i) acc = acc + aval(u[i]);
        }
    return acc;
}

// Up to `steps` steps of the current burst (ssa_steps).  fresh: factors and
// propensities in LDS are not those of the state (a chunk of a burst leaves
// them current for the next one).
template <int RB>
__device__ __forceinline__ bool ssa_small(const KParams& p, Lane& L, const View& V, const SmallView& Z, int steps,
                                          bool fresh) {
    const uint32_t x = Z.x + (L.xb ? Z.sx : 0u);
    if (fresh) {
        for (int s = 0; s < p.S; ++s) small_factor(p, Z, Z.f + s * Z.st, (int32_t)lget(x + s * Z.st));
        for (int r0 = 0; r0 < p.R; r0 += 4) {
            uint32_t rec[4], ra[4], u[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t r = (uint32_t)(r0 + i < p.R ? r0 + i : p.R - 1);
                rec[i] = Z.tab + 16u * r;
                ra[i] = Z.rates + r * (Z.shared ? 4u : Z.st);
            }
            small_props(p, Z, rec, ra, u);
#pragma unroll
            for (int i = 0; i < 4; ++i) lput(Z.a + (uint32_t)(r0 + i < p.R ? r0 + i : p.R - 1) * Z.st, u[i]);
        }
    }
    float s[RB];
    float a0 = small_prefix<RB>(p, Z, s);
    double tnext = L.cursor < (uint32_t)p.K ? p.ts[L.cursor] : 0.0;      // the next sample time
    for (int st = 0; st < steps; ++st) {
        if (a0 == 0.0f) { absorb(p, L, V, xcur(V, L)); return true; }
        const float r1 = rng_oc(L.g) * a0;
        const uint32_t w2 = rng_u32(L.g);
        // the first reaction whose running sum reaches r1, else the last: the
        // sums never decrease and the last one, a0, is not below r1, so it is
        // the number of sums below r1
        int j = 0;
#pragma unroll
        for (int i = 0; i < RB; ++i) j += r1 > s[i] ? 1 : 0;
        if constexpr (RB > 4) {
            float acc = s[RB - 1];
            for (int r0 = RB; r0 < p.R; r0 += RB) {
                uint32_t u[RB];
#pragma unroll
                for (int i = 0; i < RB; ++i) u[i] = lget(Z.a + (r0 + i) * Z.st);
#pragma unroll
                for (int i = 0; i < RB; ++i) {
                    acc = acc + aval(u[i]);
                    j += r1 > acc ? 1 : 0;
                }
            }
        }
        const u32x4 rj = lget4(Z.tab + 16u * (uint32_t)j);
        const float dt = u32_exp(w2) / a0;
        L.tacc = L.tacc + (double)dt;
        const double tn = L.t + L.tacc;
        if (L.cursor < (uint32_t)p.K && tn > tnext) {                    // T.cu:2213-2236
            uint32_t i = L.cursor;
            uint32_t* out = p.storage + (size_t)L.sim * p.K * p.SS;
            while (i < (uint32_t)p.K && tn > p.ts[i]) {
                for (int sk = 0; sk < p.SS; ++sk)
                    out[(size_t)i * p.SS + sk] = lget(x + (uint32_t)CT_I32(p.cs)[sk] * Z.st);
                ++i;
            }
            L.cursor = i;
            tnext = i < (uint32_t)p.K ? p.ts[i] : 0.0;
        }
        const uint32_t F = Z.tab + (rj.z & 0xffffu), nf = rj.z >> 16;
        for (uint32_t h = 0; h < nf; ++h) {
            const uint32_t e = lget(F + 4u * h), o = e & 0xffffu;
            const int32_t xs = (int32_t)(lget(x + o) + (uint32_t)(int)(int16_t)(e >> 16));
            lput(x + o, (uint32_t)xs);
            small_factor(p, Z, Z.f + o, xs);
        }
        L.ssa_steps++;
        if (tn <= p.tmax) L.firings++;
        const uint32_t D = Z.tab + (rj.w & 0xffffu), nd = rj.w >> 16;
        for (uint32_t d = 0; d < nd; d += 4u) {
            const u32x4 q = lget4(D + 4u * d);
            const uint32_t w[4] = {q.x, q.y, q.z, q.w};
            uint32_t rec[4], ra[4], u[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                rec[i] = Z.tab + (w[i] & 0xffffu);
                ra[i] = Z.rates + (Z.shared ? (w[i] & 0xffffu) >> 2 : w[i] >> 16);
            }
            small_props(p, Z, rec, ra, u);
#pragma unroll
            for (int i = 0; i < 4; ++i) lput(Z.a + (w[i] >> 16), u[i]);
        }
        a0 = small_prefix<RB>(p, Z, s);
    }
    return false;
}

// Persistent over slots like tau_leap_kernel<true>; one wavefront per
// workgroup, B = p.lpw of its lanes hold a slot each.
template <int RB>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void small_kernel(KParams p) {
    extern __shared__ __align__(16) uint32_t smem[];
    __shared__ float recip[64];
    recip[threadIdx.x] = c_recip[threadIdx.x];
    const uint32_t B4 = 4u * (uint32_t)p.lpw;
    // the table: change entries and dependents with byte offsets for B lanes
    for (int i = threadIdx.x; i < p.nST; i += 64) {
        const uint32_t w = p.T[p.oST + i];
        uint32_t v;
        if (i < 4 * p.R) {
            const int k = i & 3;
            v = k < 2 ? ((w & 0xffffu) * B4) | (((w >> 16) * B4) << 16) : ((w & 0xffffu) * 4u) | (w & 0xffff0000u);
        } else if (i < p.oSD) {
            v = ((w & 0xffffu) * B4) | (w & 0xffff0000u);
        } else {
            v = (w * 16u) | ((w * B4) << 16);
        }
        smem[i] = v;
    }
    const bool shared = p.c_bcast != nullptr;
    float* const rates = (float*)(smem + p.nST);
    if (shared)
        for (int i = threadIdx.x; i < p.R; i += 64) rates[i] = p.c_bcast[i];
    __syncthreads();
    const int B = p.lpw, col = (int)threadIdx.x;
    Lane L;
    L.slot = (int)blockIdx.x * B + col;
    if (col >= B || L.slot >= p.ns) return;
    const int Rp = (p.R + RB - 1) / RB * RB;
    uint32_t* const base = smem + p.nST + (shared ? p.R : 0) + col;
    View V;
    V.st = (size_t)B;
    V.xbuf = (size_t)p.S * B;
    V.X = (int32_t*)base;
    V.A = base + 2 * V.xbuf;
    uint32_t* const fac = V.A + (size_t)Rp * B;
    V.Cs = (float*)(fac + ((size_t)p.snf * p.S + 1) * B);
    SmallView Z;
    Z.tab = lds_addr(smem);
    Z.x = lds_addr(base);
    Z.st = B4;
    Z.sx = (uint32_t)p.S * B4;
    Z.a = Z.x + 2u * Z.sx;
    Z.f = Z.a + (uint32_t)Rp * B4;
    Z.shared = shared;
    Z.rates = shared ? lds_addr(rates) : Z.f + ((uint32_t)p.snf * p.S + 1u) * B4;
    for (int r = p.R; r < Rp; ++r) lput(Z.a + (uint32_t)r * B4, 0u);
    lput(Z.f + (uint32_t)p.snf * Z.sx, 0x3f800000u);
    load_lane(p, L);
    if (L.sim == -2) return;             // queue was exhausted for this slot
    if (L.sim >= 0) {                    // resume: state from the global slot arrays
        const int32_t* G = p.X + (L.xb ? (size_t)p.S * p.ns : 0) + L.slot;
        for (int s = 0; s < p.S; ++s) V.X[(size_t)s * V.st] = G[(size_t)s * p.ns];
        L.xb = 0;
        load_rates(p, V, L.sim);
    }
    bool fresh = true;
    for (int it = 0; it < p.iters; ++it) {
        if (L.sim < 0 && !fetch(p, L, V)) break;
        if (L.mode == MODE_LEAP) {
            const int r = leap_small(p, L, V, Z, recip);
            if (r == LEAP_DONE || r == LEAP_ABSORB) {
                finish(p, L, V);
            } else if (r == LEAP_SWITCH) {
                L.mode = MODE_SSA;
            }
        } else {
            if (L.ssa_left == 0) {       // open a burst
                if (p.force_ssa && L.t >= p.tmax) { finish(p, L, V); continue; }
                rng_event(L.g, L.evc++);
                L.tacc = 0.0;
                L.ssa_left = p.ssa_steps;
                fresh = true;
            }
            const int n = L.ssa_left < p.ssa_chunk ? L.ssa_left : p.ssa_chunk;
            const bool absorbed = ssa_small<RB>(p, L, V, Z, n, fresh);
            fresh = false;
            if (absorbed) {
                L.ssa_left = 0;
                finish(p, L, V);
                continue;
            }
            L.ssa_left -= n;
            if (L.ssa_left == 0) {
                L.t = L.t + L.tacc;
                L.tacc = 0.0;
                if (!p.force_ssa) L.mode = MODE_LEAP;
            }
        }
    }
    if (L.sim >= 0) {                    // suspend: current state to the global slot arrays
        const int32_t* X = xcur(V, L);
        int32_t* G = p.X + L.slot;
        for (int s = 0; s < p.S; ++s) G[(size_t)s * p.ns] = X[(size_t)s * V.st];
        L.xb = 0;
    }
    store_lane(p, L);
}

// Host: the table of a small model, or nothing when it is not eligible: a
// reaction of more than two reactant entries, of a multiplicity above 3 or of
// more than four factors.  words before the dependents in *dep, factor kinds
// per species in *kinds.
inline std::vector<uint32_t> small_table(const Model& m, const std::vector<uint32_t>& Dptr,
                                         const std::vector<uint32_t>& Dent, int* dep, int* kinds) {
    const uint32_t S = (uint32_t)m.S;
    uint32_t mmax = 0;
    for (uint32_t e : m.Lent) mmax = std::max(mmax, e >> 16);
    if (mmax > 3) return {};
    *kinds = mmax > 2 ? 5 : 2;
    const uint32_t one = (uint32_t)*kinds * S;
    std::vector<uint32_t> t((size_t)4 * m.R, 0u);
    for (int j = 0; j < m.R; ++j) {
        uint32_t f[4] = {one, one, one, one};
        int k = 0;
        if (m.Lptr[j + 1] - m.Lptr[j] > 2) return {};
        for (uint32_t h = m.Lptr[j]; h < m.Lptr[j + 1]; ++h) {
            const uint32_t s = m.Lent[h] & 0xffffu, v = m.Lent[h] >> 16;
            if (k + (v == 3u ? 3 : 1) > (mmax > 2 ? 4 : 2)) return {};
            if (v == 3u) {
                for (uint32_t q = 2; q < 5; ++q) f[k++] = q * S + s;
            } else {
                f[k++] = (v - 1u) * S + s;
            }
        }
        t[4 * j] = f[0] | (f[1] << 16);
        t[4 * j + 1] = f[2] | (f[3] << 16);
        t[4 * j + 2] = (uint32_t)t.size() | ((m.Fptr[j + 1] - m.Fptr[j]) << 16);
        t.insert(t.end(), m.Fent.begin() + m.Fptr[j], m.Fent.begin() + m.Fptr[j + 1]);
    }
    while (t.size() % 4) t.push_back(0u);
    *dep = (int)t.size();
    for (int j = 0; j < m.R; ++j) {
        const uint32_t n = Dptr[j + 1] - Dptr[j], padded = (n + 3) / 4 * 4;
        t[4 * j + 3] = (uint32_t)t.size() | (padded << 16);
        for (uint32_t k = 0; k < padded; ++k) t.push_back(Dent[Dptr[j] + std::min(k, n - 1)]);
    }
    return t;
}

}  // namespace ctl
