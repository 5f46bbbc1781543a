// ctl_mlp.hip -- the learned surrogate's MLP on gfx950: hand-written BF16
// MFMA GEMMs with FP32 accumulation for inference and training (forward,
// backward, Adam).  No counterpart in the reference (the surrogate is an
// addition of this build); the simulator is its data source, its fallback
// and the judge of its error.
//
// Network: widths w0 -> w1 -> ... -> wL, ReLU after every hidden layer,
// linear output.  Weights W_l are [w_{l-1}][w_l] row-major; activations are
// [batch][width] row-major.  Master weights, Adam moments and gradients are
// FP32; the GEMM operands (weights, activations, back-propagated errors) are
// BF16 (round to nearest even); every product accumulates in FP32.
//
// Every GEMM reads both operands contiguous along k, straight from global
// memory into MFMA fragments (gemm_frag): lane l of v_mfma_f32_32x32x16_bf16
// holds A[l%32][8*(l/32)+0..7] and B[8*(l/32)+0..7][l%32], one 16-byte load
// each, and accumulator v of lane l is C[8*(v/4) + 4*(l/32) + v%4][l%32].  So
// each BF16 array is kept in the layouts its readers need: weights as W
// [w_{l-1}][w_l] (input errors) and in fragment order (forward: packed), activations and
// errors as [batch][width] and, in training, transposed (weight gradients),
// written by the epilogue that produces them (four consecutive rows of one
// column per lane: 8 bytes).  Rows are padded to multiples of 32 elements and
// arrays to multiples of 32 rows, the padding zero, so no load needs a bounds
// check.  The products of one output accumulate in k steps of 16 in ascending
// order, whatever the tile.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "ctl_internal.h"

namespace ctl {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

enum : int { EPI_STORE_F32 = 0, EPI_BIAS_RELU, EPI_BIAS_F32, EPI_BIAS_MSE, EPI_MASK, EPI_GRAD, EPI_ADAM };

constexpr int MLAYERS = 8;               // layers of one fused launch
constexpr int MPAD = 32;                 // rows and leading dimensions are padded to multiples of this
__host__ __device__ constexpr long mpad(long w) { return (w + MPAD - 1) / MPAD * MPAD; }
// Leading dimension of the transposed arrays of B rows: never a multiple of a
// large power of two, at which the columns a wavefront writes would all fall
// on one memory channel.
__host__ __device__ constexpr long tpad(long B) { return (B + 63) / 64 * 64 + 64; }

// k padding of the weights in fragment order (and of the activations they
// meet in LDS): four steps of 16.
__host__ __device__ constexpr long kpad(long w) { return (w + 63) / 64 * 64; }

// Offset of weight (k, n) of a layer with ksteps steps of 16 in fragment
// order: the 16 x 32 fragment of a k step and a 32-column tile is 512
// consecutive elements, eight per lane, so a wavefront loads it with one
// contiguous kilobyte.
__host__ __device__ __forceinline__ long packed(long k, long n, long ksteps) {
    return ((n >> 5) * ksteps + (k >> 4)) * 512 + ((n & 31) + 32 * ((k >> 3) & 1)) * 8 + (k & 7);
}

struct AdamArgs {
    float lr, b1, b2, eps, c1, c2;
};

// One step of Adam (Kingma & Ba 2015) for one parameter.
__device__ __forceinline__ float adam_step(const AdamArgs& q, float g, float w, float& m, float& v) {
    const float mi = q.b1 * m + (1.0f - q.b1) * g;
    const float vi = q.b2 * v + (1.0f - q.b2) * g * g;
    m = mi;
    v = vi;
    return w - q.lr * (mi / q.c1) / (sqrtf(vi / q.c2) + q.eps);
}

struct GemmArgs {
    const uint16_t* A;         // [M][lda], k contiguous
    const uint16_t* B;         // [N][ldb], k contiguous; or (ldb = 0) in fragment order, bks steps a tile
    long lda, ldb;
    int bks;
    int M, N, K;               // K a multiple of 32 (zero padding)
    int tiles_n;               // column tiles (of a workgroup)
    int kchunk;                // k per split (split-K: blockIdx.y selects [y*kchunk, (y+1)*kchunk))
    const float* bias;         // [N] (EPI_BIAS_*)
    const uint16_t* maskT;     // [N][ldt] activation whose sign gates (EPI_MASK), transposed
    uint16_t* C;               // [M][ldc] bf16 out
    uint16_t* CT;              // [N][ldt] bf16 out, transposed (null: not kept); EPI_ADAM: in fragment order
    long ldc, ldt;
    float* Cf;                 // [M][N] fp32 out
    // EPI_BIAS_MSE: error against rows tidx[row] (or row) of t, and the loss
    const float* t;
    const int32_t* tidx;
    float scale;
    double* loss;              // one total per wavefront of the product, added to
    // EPI_GRAD / EPI_ADAM: weights W [M][N] (Cf: FP32 gradient or master copy)
    float *am, *av;
    AdamArgs adam;
};

__device__ __forceinline__ void store4(uint16_t* p, const uint16_t (&h)[4]) {
    *reinterpret_cast<uint2*>(p) =
        make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
}

// One 32 x 32 accumulator tile at (m0, n0): the epilogue of g.  Whatever it
// reads (targets, mask, master weights and moments) is loaded first, all of it
// in flight together.
template <int EPI>
__device__ __forceinline__ void gemm_epilogue(const GemmArgs& g, const f32x16& acc, int m0, int n0, int lane,
                                              float& sq) {
    const int col = n0 + (lane & 31);
    const bool cin = col < g.N;
    const int row0 = m0 + 4 * (lane >> 5);          // value v: row row0 + 8 (v / 4) + v % 4
    constexpr bool kBias = EPI == EPI_BIAS_RELU || EPI == EPI_BIAS_F32 || EPI == EPI_BIAS_MSE;
    const float bias = kBias && cin ? g.bias[col] : 0.0f;
    float p0[16], p1[16], p2[16];
    uint2 mk[4];
    if constexpr (EPI == EPI_BIAS_MSE) {
        long tr[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int r = row0 + 8 * (v >> 2) + (v & 3), rc = r < g.M ? r : g.M - 1;
            tr[v] = g.tidx ? g.tidx[rc] : rc;
        }
#pragma unroll
        for (int v = 0; v < 16; ++v) p0[v] = cin ? g.t[tr[v] * g.N + col] : 0.0f;
    }
    if constexpr (EPI == EPI_MASK) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            mk[q] = cin ? *reinterpret_cast<const uint2*>(g.maskT + (long)col * g.ldt + row0 + 8 * q) : make_uint2(0u, 0u);
    }
    if constexpr (EPI == EPI_ADAM) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int r = row0 + 8 * (v >> 2) + (v & 3);
            const long o = (long)r * g.N + col;
            const bool in = cin && r < g.M;
            p0[v] = in ? g.Cf[o] : 0.0f;
            p1[v] = in ? g.am[o] : 0.0f;
            p2[v] = in ? g.av[o] : 0.0f;
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int row = row0 + 8 * q;
        uint16_t h[4] = {0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int v = 4 * q + i, r = row + i;
            const bool in = cin && r < g.M;
            const long o = (long)r * g.N + col;
            const float x = acc[v];
            if constexpr (EPI == EPI_STORE_F32) {
                if (in) g.Cf[(long)blockIdx.y * g.M * g.N + o] = x;             // split y's partial
            } else if constexpr (EPI == EPI_BIAS_RELU) {
                const float y = x + bias;
                h[i] = in ? f2bf(y > 0.0f ? y : 0.0f) : (uint16_t)0;
            } else if constexpr (EPI == EPI_BIAS_F32) {
                if (in) g.Cf[o] = x + bias;
            } else if constexpr (EPI == EPI_BIAS_MSE) {
                const float e = (x + bias) - p0[v];
                if (in) {
                    sq += e * e;
                    h[i] = f2bf(2.0f * e * g.scale);
                }
            } else if constexpr (EPI == EPI_MASK) {
                const uint32_t w = i < 2 ? mk[q].x : mk[q].y;
                h[i] = in && bf2f((uint16_t)(w >> (16 * (i & 1)))) > 0.0f ? f2bf(x) : (uint16_t)0;
            } else if constexpr (EPI == EPI_GRAD) {
                if (in) g.Cf[o] = x;
            } else {
                const float w = adam_step(g.adam, x, p0[v], p1[v], p2[v]);
                if (in) {
                    g.Cf[o] = w;
                    g.am[o] = p1[v];
                    g.av[o] = p2[v];
                    h[i] = f2bf(w);
                }
            }
        }
        if constexpr (EPI == EPI_BIAS_RELU || EPI == EPI_BIAS_MSE || EPI == EPI_MASK || EPI == EPI_ADAM) {
            if (cin) {                       // rows up to the padding: zero past M
#pragma unroll
                for (int i = 0; i < 4; ++i) g.C[(long)(row + i) * g.ldc + col] = h[i];
                if (g.CT)
                    store4(EPI == EPI_ADAM ? g.CT + packed(row, col, g.ldt >> 4) : g.CT + (long)col * g.ldt + row, h);
            }
        }
    }
}

// C = A B^T by 32 x 32 tiles, one wavefront (and workgroup) each.  No LDS and
// no barrier: the fragments of eight k steps are in flight while earlier ones
// feed the matrix cores.  The small products of a training batch are bound by
// the latency of their loads: a 256 x 256 x 256 product staged through LDS in
// eight slabs, each waiting for the last, took 12 us, this way 5 us.
template <int EPI>
__device__ __forceinline__ void gemm_tile(const GemmArgs& g, int id) {
    constexpr int PF = 8;
    const int lane = threadIdx.x & 63;
    const int m0 = (id / g.tiles_n) * 32, n0 = (id % g.tiles_n) * 32;
    const int kb = (int)blockIdx.y * g.kchunk;                      // this split's k range [kb, ke)
    const int ke = kb + g.kchunk < g.K ? kb + g.kchunk : g.K;
    const int steps = ke > kb ? (ke - kb) / 16 : 0;                 // 0: a split past the end of k
    const uint16_t* pa = g.A + (long)(m0 + (lane & 31)) * g.lda + kb + 8 * (lane >> 5);
    const uint16_t* pb = g.ldb ? g.B + (long)(n0 + (lane & 31)) * g.ldb + kb + 8 * (lane >> 5)
                               : g.B + ((long)(n0 >> 5) * g.bks + (kb >> 4)) * 512 + 8 * lane;
    const int bstep = g.ldb ? 16 : 512;
    f32x16 acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
    bf16x8 fa[PF], fb[PF];
    if (steps > 0) {
#pragma unroll
        for (int q = 0; q < PF; ++q) {
            const int k = q < steps ? q : steps - 1;
            fa[q] = *reinterpret_cast<const bf16x8*>(pa + k * 16);
            fb[q] = *reinterpret_cast<const bf16x8*>(pb + (long)k * bstep);
        }
    }
    int s0 = 0;
    for (; s0 + PF <= steps; s0 += PF) {
#pragma unroll
        for (int q = 0; q < PF; ++q) {
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[q], fb[q], acc, 0, 0, 0);
            const int n = s0 + q + PF < steps ? s0 + q + PF : steps - 1;
            fa[q] = *reinterpret_cast<const bf16x8*>(pa + n * 16);
            fb[q] = *reinterpret_cast<const bf16x8*>(pb + (long)n * bstep);
            // the loads stay here: moved to their use in the next round of the
            // loop, each would be waited for
            asm volatile("" ::: "memory");
        }
    }
#pragma unroll
    for (int q = 0; q < PF; ++q)
        if (s0 + q < steps) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[q], fb[q], acc, 0, 0, 0);
    float sq = 0.0f;
    gemm_epilogue<EPI>(g, acc, m0, n0, lane, sq);
    if constexpr (EPI == EPI_BIAS_MSE) {
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) sq += __shfl_xor(sq, d);
        if (lane == 0) g.loss[id] += (double)sq;
    }
}

// XCD-aware order: consecutive workgroup ids go to different XCDs; give each
// XCD a run of consecutive tiles (same rows of A, several columns).
__device__ __forceinline__ int xcd_order() {
    const int nb = (int)gridDim.x, b = (int)blockIdx.x;
    const int full = nb / 8 * 8;
    return b < full ? (b % 8) * (full / 8) + b / 8 : b;
}

template <int EPI>
__global__ __launch_bounds__(64) void gemm_frag(GemmArgs g) {
    gemm_tile<EPI>(g, xcd_order());
}

// Products with a 128 x 128 tile for every CU (a training batch of thousands
// of rows): four wavefronts of 64 x 64, A and B staged in LDS in two slabs of
// 32 k (rows padded to 40 elements), the next slab's loads in flight during
// the products of the current one.  Fragments straight from memory are bound
// by their 32-byte rows there (us by fragments / here, rows x k x columns:
// 65536 x 2048 x 2048 2431 / 898, 612 TFLOP/s; 65536 x 288 x 1000 169 / 124;
// at the line, 256 tiles, 8192 x 512 x 512 28.1 / 22.5; at half of it 4096 x
// 512 x 512 16.7 / 20.5).  The pieces on their way are native vectors: as
// HIP's uint4 they went through scratch memory, 2452 us for the largest.
constexpr int GKP = 40;
template <int EPI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void gemm_lds(GemmArgs g) {
    __shared__ __align__(16) uint16_t As[2][128 * GKP], Bs[2][128 * GKP];
    const int id = xcd_order();
    const int m0 = (id / g.tiles_n) * 128, n0 = (id % g.tiles_n) * 128;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, tid = (int)threadIdx.x;
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    const int mrows = (int)mpad(g.M), ncols = (int)mpad(g.N);
    // this lane's two 16-byte pieces of a slab of each operand
    const uint16_t *pa[2], *pb[2];
    int sa[2];
    long bstep;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int v = tid + 256 * t, r = v >> 2, k = (v & 3) * 8;
        const int ra = m0 + r < mrows ? m0 + r : mrows - 1, rb = n0 + r < ncols ? n0 + r : ncols - 1;
        pa[t] = g.A + (long)ra * g.lda + k;
        pb[t] = g.ldb ? g.B + (long)rb * g.ldb + k : g.B + packed(k, rb, g.bks);
        sa[t] = r * GKP + k;
    }
    bstep = g.ldb ? 32 : 1024;
    f32x16 acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[a][c][v] = 0.0f;
    u32x4 ra[2], rb[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        ra[t] = *reinterpret_cast<const u32x4*>(pa[t]);
        rb[t] = *reinterpret_cast<const u32x4*>(pb[t]);
    }
    const int slabs = g.K / 32;
    for (int s = 0; s < slabs; ++s) {
        uint16_t* const A = As[s & 1];
        uint16_t* const B = Bs[s & 1];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            *reinterpret_cast<u32x4*>(A + sa[t]) = ra[t];
            *reinterpret_cast<u32x4*>(B + sa[t]) = rb[t];
        }
        __syncthreads();             // the other buffer's readers passed the previous barrier
        const int n = s + 1 < slabs ? s + 1 : s;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            ra[t] = *reinterpret_cast<const u32x4*>(pa[t] + n * 32);
            rb[t] = *reinterpret_cast<const u32x4*>(pb[t] + n * bstep);
        }
#pragma unroll
        for (int ks = 0; ks < 32; ks += 16) {
            const int kk = ks + 8 * (lane >> 5);
            bf16x8 fa[2], fb[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                fa[t] = *reinterpret_cast<const bf16x8*>(A + (wm + 32 * t + (lane & 31)) * GKP + kk);
                fb[t] = *reinterpret_cast<const bf16x8*>(B + (wn + 32 * t + (lane & 31)) * GKP + kk);
            }
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int c = 0; c < 2; ++c)
                    acc[a][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[a], fb[c], acc[a][c], 0, 0, 0);
        }
    }
    float sq = 0.0f;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int c = 0; c < 2; ++c)
            if (m0 + wm + 32 * a < g.M && n0 + wn + 32 * c < g.N)
                gemm_epilogue<EPI>(g, acc[a][c], m0 + wm + 32 * a, n0 + wn + 32 * c, lane, sq);
    if constexpr (EPI == EPI_BIAS_MSE) {
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) sq += __shfl_xor(sq, d);
        if (lane == 0) g.loss[id * 4 + wave] += (double)sq;
    }
}

// Inference of a whole network for 32 rows per workgroup: activations stay in
// LDS from the input to the output layer, weights come in fragment order from
// the L2.  Wavefront w computes columns 64 w .. 64 w + 63 of a layer (two
// accumulator tiles).  Hidden layers compute the transposed product, which
// leaves a lane four consecutive columns of one row: one 8-byte LDS store.
// Tiles of 64 and 128 rows reuse a weight fragment more but leave one or two
// wavefronts a SIMD to hide its latency (65536 rows of 32-256-256-256-1000:
// 118 / 119 / 161 us at 32 / 64 / 128; 1000 rows: 27 / 37 / 64 us).  Layer by
// layer with the activations in memory the passes took 368 us and 46 us; the
// output rows (262 MB) take 51 us at the rate of a copy.
struct FusedArgs {
    const float* x;
    float* y;
    long rows;
    int L, ldk;                              // LDS row length (elements)
    int w[MLAYERS + 1];
    const uint16_t* wt[MLAYERS];             // fragment order
    const float* bias[MLAYERS];
};

// The product of a wavefront's two tiles: pa its activations in LDS, pb its
// weight fragments, ks k steps (a multiple of 4).  Four steps of weights are in
// flight; the last loads of a tile run into the next one's fragments (or the
// slack behind the array) and are not used.
template <bool LAST>
__device__ __forceinline__ void fused_product(f32x16 (&acc)[2], const uint16_t* pa, const uint16_t* const (&pb)[2],
                                              int ks) {
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[c][v] = 0.0f;
    bf16x8 fb[4][2], fa[2];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int c = 0; c < 2; ++c) fb[q][c] = *reinterpret_cast<const bf16x8*>(pb[c] + q * 512);
    fa[0] = *reinterpret_cast<const bf16x8*>(pa);
    for (int s0 = 0; s0 < ks; s0 += 4) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int n = s0 + q + 1 < ks ? s0 + q + 1 : 0;
            fa[(q + 1) & 1] = *reinterpret_cast<const bf16x8*>(pa + n * 16);
#pragma unroll
            for (int c = 0; c < 2; ++c)
                acc[c] = LAST ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[q & 1], fb[q][c], acc[c], 0, 0, 0)
                              : __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[q][c], fa[q & 1], acc[c], 0, 0, 0);
#pragma unroll
            for (int c = 0; c < 2; ++c)
                fb[q][c] = *reinterpret_cast<const bf16x8*>(pb[c] + (long)(s0 + q + 4) * 512);
            // the loads stay here: the compiler would move them to their use
            // in the next round of the loop, and wait for each
            asm volatile("" ::: "memory");
        }
    }
}

__global__ __launch_bounds__(256) void mlp_fused(FusedArgs f) {
    extern __shared__ __align__(16) uint16_t act[];                  // [BM][ldk], then the biases
    constexpr int BM = 32;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long r0 = (long)blockIdx.x * BM;
    // input rows (64 columns at a time, eight loads in flight) and every bias
    float* const bias = reinterpret_cast<float*>(act + BM * f.ldk);
    for (int c0 = 0; c0 < f.w[0]; c0 += 64) {
        const int c = c0 + lane;
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const long r = r0 + wave + 4 * j;
            v[j] = c < f.w[0] && r < f.rows ? f.x[r * f.w[0] + c] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) act[(wave + 4 * j) * f.ldk + c] = f2bf(v[j]);
    }
    for (int l = 0, o = 0; l < f.L; ++l) {
        for (int c = threadIdx.x; c < f.w[l + 1]; c += 256) bias[o + c] = f.bias[l][c];
        o += (int)kpad(f.w[l + 1]);
    }
    __syncthreads();
    int bo = 0;
    const uint16_t* pa = act + (lane & 31) * f.ldk + 8 * (lane >> 5);
    for (int l = 0; l + 1 < f.L; ++l) {                              // hidden layers: at most 256 columns
        const int ks = (int)kpad(f.w[l]) / 16, N = f.w[l + 1], n0 = 64 * wave;
        const bool work = n0 < N;
        f32x16 acc[2];
        if (work) {
            const uint16_t* const pb[2] = {f.wt[l] + (long)(n0 >> 5) * ks * 512 + 8 * lane,
                                           f.wt[l] + (long)((n0 >> 5) + (n0 + 32 < N ? 1 : 0)) * ks * 512 + 8 * lane};
            fused_product<false>(acc, pa, pb, ks);
        }
        __syncthreads();                                             // every wavefront has read the activations
        if (work) {
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int col = n0 + 32 * c + 8 * q + 4 * (lane >> 5);
                    const float4 bv = *reinterpret_cast<const float4*>(bias + bo + col);
                    const float b[4] = {bv.x, bv.y, bv.z, bv.w};
                    uint16_t h[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float y = acc[c][4 * q + i] + b[i];
                        h[i] = col + i < N ? f2bf(y > 0.0f ? y : 0.0f) : (uint16_t)0;
                    }
                    store4(act + (lane & 31) * f.ldk + col, h);
                }
        }
        __syncthreads();
        bo += (int)kpad(N);
    }
    const int l = f.L - 1, ks = (int)kpad(f.w[l]) / 16, N = f.w[l + 1];
    for (int n0 = 64 * wave; n0 < N; n0 += 256) {
        f32x16 acc[2];
        const uint16_t* const pb[2] = {f.wt[l] + (long)(n0 >> 5) * ks * 512 + 8 * lane,
                                       f.wt[l] + (long)((n0 >> 5) + (n0 + 32 < N ? 1 : 0)) * ks * 512 + 8 * lane};
        fused_product<true>(acc, pa, pb, ks);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int col = n0 + 32 * c + (lane & 31);
            if (col >= N) continue;
            const float b = bias[bo + col];
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const long row = r0 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                if (row < f.rows) f.y[row * N + col] = acc[c][v] + b;
            }
        }
    }
}

// Column sums db[j] = sum_b d[b][j] (d in BF16, read transposed: [j][ldt]),
// FP32, in a fixed order: rows in chunks of CS_ROWS, a chunk as four sums of
// every fourth row, (s0 + s1) + (s2 + s3), the chunks added in order.
constexpr int CS_ROWS = 512;
__device__ __forceinline__ float col_chunk(const uint16_t* __restrict__ d, int b0, int b1) {
    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int b = b0; b < b1; b += 32) {                // rows past the batch are zero padding
        uint4 w[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) w[k] = *reinterpret_cast<const uint4*>(d + b + 8 * k);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t u[4] = {w[k].x, w[k].y, w[k].z, w[k].w};
#pragma unroll
            for (int i = 0; i < 8; ++i) s[i & 3] += bf2f((uint16_t)(u[i >> 1] >> (16 * (i & 1))));
        }
    }
    return (s[0] + s[1]) + (s[2] + s[3]);
}

__global__ __launch_bounds__(64) void col_sum_part(const uint16_t* __restrict__ dT, long ldt, float* __restrict__ part,
                                                   int B, int N) {
    const int j = blockIdx.x * 64 + (int)threadIdx.x;
    if (j >= N) return;
    const int b0 = blockIdx.y * CS_ROWS;
    part[(long)blockIdx.y * N + j] = col_chunk(dT + (long)j * ldt, b0, b0 + CS_ROWS < B ? b0 + CS_ROWS : B);
}

__global__ void col_sum(const float* __restrict__ part, float* __restrict__ db, int chunks, int N) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= N) return;
    float s = 0.0f;
    for (int c0 = 0; c0 < chunks; c0 += 8) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = part[(long)(c0 + k < chunks ? c0 + k : chunks - 1) * N + j];
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (c0 + k < chunks) s += v[k];
    }
    db[j] = s;
}

// The parameter step of a small batch in one launch: for up to MLAYERS layers
// the weight gradient act^T err (32 x 32 tiles, one wavefront each) with Adam
// (or the store of the gradient) as its epilogue, and the bias gradients as
// column sums of the errors, 64 columns a wavefront.
struct StepArgs {
    GemmArgs g[MLAYERS];
    float *bw[MLAYERS], *bm[MLAYERS], *bv[MLAYERS];       // bias: parameters (or gradient) and moments
    int first[MLAYERS + 1];                               // first workgroup of each layer
    int layers, rows;
};

template <int EPI>
__global__ __launch_bounds__(64) void grad_step(StepArgs a) {
    int l = 0;
    while (l + 1 < a.layers && (int)blockIdx.x >= a.first[l + 1]) ++l;
    const GemmArgs& g = a.g[l];
    const int id = (int)blockIdx.x - a.first[l];
    const int tiles = (g.M + 31) / 32 * g.tiles_n;
    if (id < tiles) {
        gemm_tile<EPI>(g, id);
        return;
    }
    const int j = (id - tiles) * 64 + (int)threadIdx.x;
    if (j >= g.N) return;
    float s = 0.0f;
    for (int b0 = 0; b0 < a.rows; b0 += CS_ROWS)
        s += col_chunk(g.B + (long)j * g.ldb, b0, b0 + CS_ROWS < a.rows ? b0 + CS_ROWS : a.rows);
    if constexpr (EPI == EPI_ADAM) a.bw[l][j] = adam_step(g.adam, s, a.bw[l][j], a.bm[l][j], a.bv[l][j]);
    else a.bw[l][j] = s;
}

// The wavefronts' loss totals, in order: total[0] = sum of part[0 .. n).
__global__ __launch_bounds__(256) void loss_sum(const double* __restrict__ part, double* __restrict__ total, long n) {
    __shared__ double red[256];
    double s = 0.0;
    for (long i0 = threadIdx.x; i0 < n; i0 += 256 * 16) {
        double v[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) v[k] = i0 + 256 * k < n ? part[i0 + 256 * k] : 0.0;
#pragma unroll
        for (int k = 0; k < 16; ++k) s += v[k];
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) total[0] = red[0];
}

// Split-K partial sums, added in split order: C[i] = sum_s part[s][i].
__global__ void ksplit_sum(const float* __restrict__ part, float* __restrict__ C, int splits, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float s = 0.0f;
    for (int k = 0; k < splits; ++k) s += part[(long)k * n + i];
    C[i] = s;
}

// Rows idx[0..B) (or 0..B) of a [n][w] FP32 array as BF16: [B][ld] and, when
// kept, transposed [w][ldt]; zero between B and Bp.
__global__ void gather_rows(const float* __restrict__ src, const int32_t* __restrict__ idx, uint16_t* __restrict__ dst,
                            uint16_t* __restrict__ dstT, int B, int Bp, int w, long ld, long ldt) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)Bp * w) return;
    const long b = i / w, k = i % w;
    const uint16_t h = b < B ? f2bf(src[(idx ? (long)idx[b] : b) * w + k]) : (uint16_t)0;
    dst[b * ld + k] = h;
    if (dstT) dstT[k * ldt + b] = h;
}

// BF16 copies of the weights of up to MLAYERS layers: W [K][ldn] and in
// fragment order.  One launch: a layer's own is 3 to 5 us of a call that takes
// 25 for a small network.
struct CopyArgs {
    const float* w[MLAYERS];
    uint16_t *wb[MLAYERS], *wt[MLAYERS];
    int K[MLAYERS], N[MLAYERS];
    int first[MLAYERS + 1];                               // first workgroup of each layer
    int layers;
};

__global__ __launch_bounds__(256) void weights_bf16(CopyArgs a) {
    int l = 0;
    while (l + 1 < a.layers && (int)blockIdx.x >= a.first[l + 1]) ++l;
    const long i = (long)((int)blockIdx.x - a.first[l]) * 256 + threadIdx.x;
    const int K = a.K[l], N = a.N[l];
    if (i >= (long)K * N) return;
    const long k = i / N, j = i % N;
    const uint16_t h = f2bf(a.w[l][i]);
    a.wb[l][k * mpad(N) + j] = h;
    a.wt[l][packed(k, j, kpad(K) >> 4)] = h;
}

// Adam on the FP32 master copy (the weight copies are refreshed afterwards).
__global__ void adam(float* __restrict__ w, const float* __restrict__ gr, float* __restrict__ m, float* __restrict__ v,
                     long n, AdamArgs q) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    w[i] = adam_step(q, gr[i], w[i], m[i], v[i]);
}

}  // namespace ctl

using namespace ctl;

struct ctl_mlp {
    int device = 0;
    hipStream_t stream = nullptr;
    std::vector<int> widths;
    int L = 0;                          // layers
    std::vector<long> woff, boff;       // offsets into the flat parameter vector
    long nparam = 0;
    float *w = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;   // flat fp32: W_1, b_1, ..., W_L, b_L
    std::vector<uint16_t*> wb, wt;      // bf16 copies of W_l, [w_{l-1}][w_l] and in fragment order (padded)
    long step = 0;
    // work buffers: activations for up to cap rows, the rest (training) for up to tcap rows
    int cap = 0, tcap = 0;
    std::vector<uint16_t*> act;         // act[l]: [cap][w_l], l = 0..L-1
    std::vector<uint16_t*> actT;        // transposed, [w_l][tcap]
    std::vector<uint16_t*> err, errT;   // err[l]: error of layer l's output, l = 1..L, both layouts
    float* cpart = nullptr;             // [ceil(tcap / CS_ROWS)][max w] column-sum partials
    float* kpart = nullptr;             // split-K partial tiles of the weight gradients
    long kpart_words = 0;
    double* lacc = nullptr;             // loss total, then the wavefronts' own totals
    long nloss = 0;
    int32_t* idx = nullptr;             // [ndata] epoch permutation
    // training data
    float *dX = nullptr, *dY = nullptr;
    long ndata = 0;
    // host calls: inputs and outputs (or targets) of up to hcap rows
    float *hx = nullptr, *hy = nullptr;
    int hcap = 0;
    std::vector<void*> allocs, abuf, tbuf, hbuf;    // for good; with cap; with tcap; with hcap
};

namespace {

int mfail(hipError_t e, const char* what) {
    char b[256];
    std::snprintf(b, sizeof b, "%s: %s", what, hipGetErrorString(e));
    return ctl::fail(e == hipErrorOutOfMemory ? CTL_E_NOMEM : CTL_E_DEVICE, b);
}

#define MHIP(call, what)                             \
    do {                                             \
        hipError_t e_ = (call);                      \
        if (e_ != hipSuccess) return mfail(e_, what); \
    } while (0)

template <typename T>
int malloc_dev(std::vector<void*>& own, T** p, size_t count) {
    void* q = nullptr;
    hipError_t e = hipMalloc(&q, std::max<size_t>(count, 1) * sizeof(T));
    if (e != hipSuccess) return mfail(e, "hipMalloc");
    own.push_back(q);
    *p = (T*)q;
    return 0;
}

// A padded BF16 array, zero (the padding stays so).
int malloc_bf16(ctl_mlp* n, std::vector<void*>& own, uint16_t** p, long rows, long ld) {
    const size_t count = (size_t)mpad(rows) * (size_t)ld;
    if (int rc = malloc_dev(own, p, count)) return rc;
    MHIP(hipMemsetAsync(*p, 0, count * sizeof(uint16_t), n->stream), "memset");
    return 0;
}

void free_all(std::vector<void*>& own) {
    for (void* q : own) (void)hipFree(q);
    own.clear();
}

// Launches g over the tiles of its output.  128 x 128 tiles of a workgroup
// when they still give every CU one, else 32 x 32 tiles of one wavefront
// (a 256 x 1000 layer of a training batch: 256 of them).
template <int EPI>
void gemm(ctl_mlp* n, GemmArgs g, int splits = 1) {
    const long big = (long)((g.M + 127) / 128) * ((g.N + 127) / 128);
    if (splits == 1) g.kchunk = g.K;
    if (splits == 1 && big >= 256) {
        g.tiles_n = (g.N + 127) / 128;
        hipLaunchKernelGGL(gemm_lds<EPI>, dim3((unsigned)big), dim3(256), 0, n->stream, g);
        return;
    }
    g.tiles_n = (g.N + 31) / 32;
    const long tiles = (long)((g.M + 31) / 32) * g.tiles_n;
    hipLaunchKernelGGL(gemm_frag<EPI>, dim3((unsigned)tiles, (unsigned)splits), dim3(64), 0, n->stream, g);
}

// Activation buffers for B rows.
int ensure_cap(ctl_mlp* n, int B) {
    if (B <= n->cap) return 0;
    MHIP(hipStreamSynchronize(n->stream), "sync");
    free_all(n->abuf);
    n->cap = 0;
    n->act.assign(n->L, nullptr);
    for (int l = 0; l < n->L; ++l)
        if (int rc = malloc_bf16(n, n->abuf, &n->act[l], B, mpad(n->widths[l]))) return rc;
    n->cap = B;
    return 0;
}

// Training buffers for B rows.
int ensure_train(ctl_mlp* n, int B) {
    if (int rc = ensure_cap(n, B)) return rc;
    if (B <= n->tcap) return 0;
    MHIP(hipStreamSynchronize(n->stream), "sync");
    free_all(n->tbuf);
    n->tcap = 0;
    n->kpart = nullptr;
    n->kpart_words = 0;
    n->actT.assign(n->L, nullptr);
    n->err.assign(n->L + 1, nullptr);
    n->errT.assign(n->L + 1, nullptr);
    int rc, wmax = 0;
    for (int w : n->widths) wmax = std::max(wmax, w);
    const long ldb = tpad(B);
    for (int l = 0; l < n->L; ++l) {
        const int w = n->widths[l], wn = n->widths[l + 1];
        if ((rc = malloc_bf16(n, n->tbuf, &n->actT[l], w, ldb)) ||
            (rc = malloc_bf16(n, n->tbuf, &n->err[l + 1], B, mpad(wn))) ||
            (rc = malloc_bf16(n, n->tbuf, &n->errT[l + 1], wn, ldb)))
            return rc;
    }
    // at most one wavefront per 32 x 32 tile of the output layer
    n->nloss = ((long)B + 31) / 32 * ((n->widths[n->L] + 31) / 32) + 4 * ((long)((B + 127) / 128) + 32);
    if ((rc = malloc_dev(n->tbuf, &n->lacc, 1 + n->nloss)) ||
        (rc = malloc_dev(n->tbuf, &n->cpart, (size_t)((B + CS_ROWS - 1) / CS_ROWS) * wmax)))
        return rc;
    if (B >= 2048) {                    // large batches: room for 16 splits of the largest weight block
        long wmn = 0;
        for (int l = 0; l < n->L; ++l) wmn = std::max(wmn, (long)n->widths[l] * n->widths[l + 1]);
        if ((rc = malloc_dev(n->tbuf, &n->kpart, (size_t)16 * wmn))) return rc;
        n->kpart_words = 16 * wmn;
    }
    n->tcap = B;
    return 0;
}

// Device copies of a host call's rows.
int ensure_host(ctl_mlp* n, int B) {
    if (B <= n->hcap) return 0;
    MHIP(hipStreamSynchronize(n->stream), "sync");
    free_all(n->hbuf);
    n->hcap = 0;
    int rc;
    if ((rc = malloc_dev(n->hbuf, &n->hx, (size_t)B * n->widths[0])) ||
        (rc = malloc_dev(n->hbuf, &n->hy, (size_t)B * n->widths[n->L])))
        return rc;
    n->hcap = B;
    return 0;
}

// Input rows src (device, FP32) idx[0..B) as BF16 into act[0].
void load_input(ctl_mlp* n, const float* src, const int32_t* idx, int B, bool train) {
    const int w0 = n->widths[0], Bp = (int)mpad(B);
    hipLaunchKernelGGL(gather_rows, dim3((unsigned)(((long)Bp * w0 + 255) / 256)), dim3(256), 0, n->stream, src, idx,
                       n->act[0], train ? n->actT[0] : (uint16_t*)nullptr, B, Bp, w0, mpad(w0), tpad(n->tcap));
}

// Forward pass of B rows already in act[0].  Inference (out): the output layer
// writes FP32 rows to out.  Training (t): it forms the error against rows
// tidx[0..B) (or 0..B) of t and adds the squared errors to *lacc.
void forward(ctl_mlp* n, int B, float* out, const float* t = nullptr, const int32_t* tidx = nullptr) {
    for (int l = 0; l < n->L; ++l) {
        const int K = n->widths[l], N = n->widths[l + 1];
        GemmArgs g{};
        g.A = n->act[l];
        g.lda = mpad(K);
        g.B = n->wt[l];
        g.ldb = 0;
        g.bks = (int)kpad(K) / 16;
        g.M = B; g.N = N; g.K = (int)mpad(K);
        g.bias = n->w + n->boff[l];
        g.ldc = mpad(N);
        g.ldt = tpad(n->tcap);
        if (l + 1 < n->L) {
            g.C = n->act[l + 1];
            g.CT = t ? n->actT[l + 1] : nullptr;
            gemm<EPI_BIAS_RELU>(n, g);
        } else if (t) {
            g.C = n->err[l + 1];
            g.CT = n->errT[l + 1];
            g.t = t;
            g.tidx = tidx;
            g.scale = 1.0f / (float)((long)B * N);
            g.loss = n->lacc + 1;
            gemm<EPI_BIAS_MSE>(n, g);
        } else {
            g.Cf = out;
            gemm<EPI_BIAS_F32>(n, g);
        }
    }
}

// Inference of B rows of x (device, FP32) into out: one fused launch for inner
// widths up to 256 (four wavefronts of 64 columns), else layer by layer.  A wide
// output in few rows goes by layers too: the fused workgroups of 32 rows walk
// its columns one after the other.  us of the call fused / by layers, 64, 2048
// and 8192 rows: 1000 outputs behind 256s 37 / 35, 38 / 42, 44 / 63; 2000
// behind 200 38 / 26, 40 / 38, 50 / 49; 3000 behind 200 47 / 25, 56 / 40, 63 /
// 66; 8000 behind 256s 124 / 32, 125 / 53, 159 / 131.
int infer(ctl_mlp* n, const float* x, int B, float* out) {
    int wmax = 0;
    for (int l = 0; l < n->L; ++l) wmax = std::max(wmax, n->widths[l]);
    const bool tall = n->widths[n->L] <= 1024 || B >= 8192;
    if (wmax <= 256 && n->L <= MLAYERS && tall) {
        FusedArgs f{};
        f.x = x;
        f.y = out;
        f.rows = B;
        f.L = n->L;
        f.ldk = (int)kpad(wmax) + 8;
        for (int l = 0; l <= n->L; ++l) f.w[l] = n->widths[l];
        for (int l = 0; l < n->L; ++l) {
            f.wt[l] = n->wt[l];
            f.bias[l] = n->w + n->boff[l];
        }
        size_t lds = (size_t)32 * f.ldk * sizeof(uint16_t);
        for (int l = 1; l <= n->L; ++l) lds += sizeof(float) * kpad(n->widths[l]);
        if (lds <= 65536) {
            hipLaunchKernelGGL(mlp_fused, dim3((unsigned)((B + 31) / 32)), dim3(256), lds, n->stream, f);
            return 0;
        }
    }
    if (int rc = ensure_cap(n, B)) return rc;
    load_input(n, x, nullptr, B, false);
    forward(n, B, out);
    return 0;
}

// Refreshes the BF16 copies of every layer's weights.
void refresh_bf16(ctl_mlp* n) {
    for (int l0 = 0; l0 < n->L; l0 += MLAYERS) {
        CopyArgs a{};
        a.layers = std::min(MLAYERS, n->L - l0);
        int blocks = 0;
        for (int i = 0; i < a.layers; ++i) {
            const int l = l0 + i;
            a.w[i] = n->w + n->woff[l];
            a.wb[i] = n->wb[l];
            a.wt[i] = n->wt[l];
            a.K[i] = n->widths[l];
            a.N[i] = n->widths[l + 1];
            a.first[i] = blocks;
            blocks += (int)(((long)a.K[i] * a.N[i] + 255) / 256);
        }
        a.first[a.layers] = blocks;
        hipLaunchKernelGGL(weights_bf16, dim3((unsigned)blocks), dim3(256), 0, n->stream, a);
    }
}

// Backward pass from the output error: the gradient into n->g or, with q,
// one Adam step of every parameter.
void backward(ctl_mlp* n, int B, const AdamArgs* q) {
    const long ldt = tpad(n->tcap);
    for (int l = n->L - 1; l > 0; --l) {
        // err[l] = (err[l+1] W_l^T) gated by act[l] > 0
        const int K = n->widths[l], N = n->widths[l + 1];
        GemmArgs g{};
        g.A = n->err[l + 1];
        g.lda = mpad(N);
        g.B = n->wb[l];
        g.ldb = mpad(N);
        g.M = B; g.N = K; g.K = (int)mpad(N);
        g.maskT = n->actT[l];
        g.C = n->err[l];
        g.CT = n->errT[l];
        g.ldc = mpad(K);
        g.ldt = ldt;
        gemm<EPI_MASK>(n, g);
    }
    // dW_l = act[l]^T err[l+1] : (K x B) (B x N)
    bool split = false;
    std::vector<int> splits(n->L, 1);
    std::vector<GemmArgs> gw(n->L);
    for (int l = 0; l < n->L; ++l) {
        const int K = n->widths[l], N = n->widths[l + 1];
        GemmArgs& g = gw[l];
        g.A = n->actT[l];
        g.B = n->errT[l + 1];
        g.lda = g.ldb = ldt;
        g.M = K; g.N = N; g.K = (int)mpad(B);
        g.tiles_n = (N + 31) / 32;
        g.kchunk = g.K;
        // a long k loop over few tiles (a large batch): split k so that about
        // 1024 64 x 64 tiles run, partial products summed in order
        const long tiles = (long)((K + 63) / 64) * ((N + 63) / 64);
        const long big = (long)((K + 127) / 128) * ((N + 127) / 128);
        if (n->kpart && big < 256)
            while (splits[l] < 64 && tiles * splits[l] * 2 <= 1024 && B / (splits[l] * 2) >= 1024 &&
                   (long)splits[l] * 2 * K * N <= n->kpart_words)
                splits[l] *= 2;
        split = split || splits[l] > 1 || big >= 256 || B > 4 * CS_ROWS;
    }
    if (!split) {
        for (int l0 = 0; l0 < n->L; l0 += MLAYERS) {
            StepArgs a{};
            a.layers = std::min(MLAYERS, n->L - l0);
            a.rows = B;
            int blocks = 0;
            for (int i = 0; i < a.layers; ++i) {
                const int l = l0 + i;
                GemmArgs& g = a.g[i];
                g = gw[l];
                float* p = q ? n->w : n->g;
                g.Cf = p + n->woff[l];
                a.bw[i] = p + n->boff[l];
                if (q) {
                    g.adam = *q;
                    g.am = n->m + n->woff[l];
                    g.av = n->v + n->woff[l];
                    a.bm[i] = n->m + n->boff[l];
                    a.bv[i] = n->v + n->boff[l];
                    g.C = n->wb[l];
                    g.CT = n->wt[l];
                    g.ldc = mpad(g.N);
                    g.ldt = kpad(g.M);
                }
                a.first[i] = blocks;
                blocks += (g.M + 31) / 32 * g.tiles_n + (g.N + 63) / 64;
            }
            a.first[a.layers] = blocks;
            if (q) hipLaunchKernelGGL(grad_step<EPI_ADAM>, dim3((unsigned)blocks), dim3(64), 0, n->stream, a);
            else hipLaunchKernelGGL(grad_step<EPI_GRAD>, dim3((unsigned)blocks), dim3(64), 0, n->stream, a);
        }
        return;
    }
    for (int l = 0; l < n->L; ++l) {
        GemmArgs& g = gw[l];
        const long mn = (long)g.M * g.N;
        g.Cf = splits[l] > 1 ? n->kpart : n->g + n->woff[l];
        if (splits[l] > 1) {
            const int chunk = (B + splits[l] - 1) / splits[l];
            g.kchunk = (int)mpad(chunk);
        }
        gemm<EPI_STORE_F32>(n, g, splits[l]);
        if (splits[l] > 1)
            hipLaunchKernelGGL(ksplit_sum, dim3((unsigned)((mn + 255) / 256)), dim3(256), 0, n->stream, n->kpart,
                               n->g + n->woff[l], splits[l], mn);
        const int chunks = (B + CS_ROWS - 1) / CS_ROWS;
        hipLaunchKernelGGL(col_sum_part, dim3((g.N + 63) / 64, chunks), dim3(64), 0, n->stream, n->errT[l + 1], ldt,
                           n->cpart, B, g.N);
        hipLaunchKernelGGL(col_sum, dim3((g.N + 255) / 256), dim3(256), 0, n->stream, n->cpart, n->g + n->boff[l],
                           chunks, g.N);
    }
    if (q) {
        hipLaunchKernelGGL(adam, dim3((unsigned)((n->nparam + 255) / 256)), dim3(256), 0, n->stream, n->w, n->g, n->m,
                           n->v, n->nparam, *q);
        refresh_bf16(n);
    }
}

}  // namespace

extern "C" {

int ctl_mlp_create(const int32_t* widths, int32_t nlayers, int32_t gpu, uint64_t seed, ctl_mlp** out) {
    ctl::clear_error();
    if (!widths || nlayers < 1 || !out) return ctl::fail(CTL_E_ARGS, "bad arguments");
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
        return ctl::fail(CTL_E_DEVICE, "no HIP device available: libctl needs an AMD GPU (gfx950)");
    for (int l = 0; l <= nlayers; ++l)
        if (widths[l] <= 0) return ctl::fail(CTL_E_ARGS, "layer widths must be positive");
    ctl_mlp* n = new ctl_mlp();
    auto bail = [&](int rc) { ctl_mlp_destroy(n); return rc; };
    n->device = gpu;
    n->L = nlayers;
    n->widths.assign(widths, widths + nlayers + 1);
    hipError_t e = hipSetDevice(gpu);
    if (e != hipSuccess) return bail(mfail(e, "hipSetDevice"));
    if ((e = hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking)) != hipSuccess) return bail(mfail(e, "stream"));
    long off = 0;
    for (int l = 0; l < nlayers; ++l) {
        n->woff.push_back(off);
        off += (long)widths[l] * widths[l + 1];
        n->boff.push_back(off);
        off += widths[l + 1];
    }
    n->nparam = off;
    int rc;
    if ((rc = malloc_dev(n->allocs, &n->w, off)) || (rc = malloc_dev(n->allocs, &n->g, off)) ||
        (rc = malloc_dev(n->allocs, &n->m, off)) || (rc = malloc_dev(n->allocs, &n->v, off)))
        return bail(rc);
    n->wb.assign(nlayers, nullptr);
    n->wt.assign(nlayers, nullptr);
    for (int l = 0; l < nlayers; ++l)
        if ((rc = malloc_bf16(n, n->allocs, &n->wb[l], widths[l], mpad(widths[l + 1]))) ||
            (rc = malloc_bf16(n, n->allocs, &n->wt[l], widths[l + 1] + 32, kpad(widths[l]))))
            return bail(rc);
    // He-uniform weights, zero biases (host RNG, seeded)
    std::vector<float> h(off, 0.0f);
    std::mt19937_64 rng(seed);
    for (int l = 0; l < nlayers; ++l) {
        const float a = std::sqrt(6.0f / (float)widths[l]);
        std::uniform_real_distribution<float> U(-a, a);
        for (long i = 0; i < (long)widths[l] * widths[l + 1]; ++i) h[n->woff[l] + i] = U(rng);
    }
    if ((e = hipMemcpy(n->w, h.data(), sizeof(float) * off, hipMemcpyHostToDevice)) != hipSuccess) return bail(mfail(e, "H2D"));
    if ((e = hipMemsetAsync(n->m, 0, sizeof(float) * off, n->stream)) != hipSuccess ||
        (e = hipMemsetAsync(n->v, 0, sizeof(float) * off, n->stream)) != hipSuccess)
        return bail(mfail(e, "memset"));
    refresh_bf16(n);
    if ((e = hipStreamSynchronize(n->stream)) != hipSuccess) return bail(mfail(e, "init"));
    *out = n;
    return 0;
}

int ctl_mlp_num_params(const ctl_mlp* n, int64_t* count) {
    if (!n || !count) return ctl::fail(CTL_E_ARGS, "null argument");
    *count = n->nparam;
    return 0;
}

int ctl_mlp_params(ctl_mlp* n, float* host, size_t count, int32_t set) {
    ctl::clear_error();
    if (!n || !host || count != (size_t)n->nparam) return ctl::fail(CTL_E_ARGS, "count must equal the parameter count");
    MHIP(hipSetDevice(n->device), "hipSetDevice");
    if (set) {
        MHIP(hipMemcpy(n->w, host, sizeof(float) * count, hipMemcpyHostToDevice), "H2D");
        refresh_bf16(n);
        MHIP(hipStreamSynchronize(n->stream), "sync");
    } else {
        MHIP(hipMemcpy(host, n->w, sizeof(float) * count, hipMemcpyDeviceToHost), "D2H");
    }
    return 0;
}

int ctl_mlp_forward(ctl_mlp* n, const float* x, int64_t rows, float* y) {
    ctl::clear_error();
    if (!n || !x || !y || rows <= 0) return ctl::fail(CTL_E_ARGS, "bad arguments");
    MHIP(hipSetDevice(n->device), "hipSetDevice");
    const int chunk = 8192;
    const int w0 = n->widths[0], wL = n->widths[n->L];
    const int cap = (int)std::min<int64_t>(rows, chunk);
    int rc = ensure_host(n, cap);
    if (rc) return rc;
    for (int64_t r0 = 0; r0 < rows; r0 += chunk) {
        const int B = (int)std::min<int64_t>(chunk, rows - r0);
        MHIP(hipMemcpyAsync(n->hx, x + r0 * w0, sizeof(float) * (size_t)B * w0, hipMemcpyHostToDevice, n->stream), "H2D");
        if ((rc = infer(n, n->hx, B, n->hy))) return rc;
        MHIP(hipGetLastError(), "forward launch");
        MHIP(hipMemcpyAsync(y + r0 * wL, n->hy, sizeof(float) * (size_t)B * wL, hipMemcpyDeviceToHost, n->stream), "D2H");
        MHIP(hipStreamSynchronize(n->stream), "forward");
    }
    return 0;
}

int ctl_mlp_forward_device(ctl_mlp* n, const float* x_dev, int64_t rows, float* y_dev, float* ms) {
    ctl::clear_error();
    if (!n || !x_dev || !y_dev || rows <= 0) return ctl::fail(CTL_E_ARGS, "bad arguments");
    MHIP(hipSetDevice(n->device), "hipSetDevice");
    const int chunk = 65536;
    int rc = 0;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (ms) {
        MHIP(hipEventCreate(&e0), "event");
        MHIP(hipEventCreate(&e1), "event");
        MHIP(hipEventRecord(e0, n->stream), "event");
    }
    const int w0 = n->widths[0], wL = n->widths[n->L];
    for (int64_t r0 = 0; r0 < rows; r0 += chunk) {
        const int B = (int)std::min<int64_t>(chunk, rows - r0);
        if ((rc = infer(n, x_dev + r0 * w0, B, y_dev + r0 * wL))) break;   // straight into the caller's rows
    }
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && ms) e = hipEventRecord(e1, n->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(n->stream);
    if (e == hipSuccess && ms) e = hipEventElapsedTime(ms, e0, e1);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (rc) return rc;
    if (e != hipSuccess) return mfail(e, "forward");
    return 0;
}

// One forward + backward on rows (x, t); returns the loss and the FP32
// gradient of the mean squared error with respect to every parameter.
int ctl_mlp_gradient(ctl_mlp* n, const float* x, const float* t, int32_t rows, float* grad, size_t count, float* loss) {
    ctl::clear_error();
    if (!n || !x || !t || rows <= 0 || rows > 65536 || (grad && count != (size_t)n->nparam)) return ctl::fail(CTL_E_ARGS, "bad arguments");
    MHIP(hipSetDevice(n->device), "hipSetDevice");
    int rc;
    if ((rc = ensure_train(n, rows)) || (rc = ensure_host(n, rows))) return rc;
    const size_t nin = (size_t)rows * n->widths[0], nout = (size_t)rows * n->widths[n->L];
    MHIP(hipMemcpyAsync(n->hx, x, sizeof(float) * nin, hipMemcpyHostToDevice, n->stream), "H2D");
    MHIP(hipMemcpyAsync(n->hy, t, sizeof(float) * nout, hipMemcpyHostToDevice, n->stream), "H2D");
    MHIP(hipMemsetAsync(n->lacc, 0, sizeof(double) * (1 + n->nloss), n->stream), "memset");
    load_input(n, n->hx, nullptr, rows, true);
    forward(n, rows, nullptr, n->hy);
    backward(n, rows, nullptr);
    hipLaunchKernelGGL(loss_sum, dim3(1), dim3(256), 0, n->stream, n->lacc + 1, n->lacc, n->nloss);
    MHIP(hipGetLastError(), "gradient launch");
    double sum = 0.0;
    MHIP(hipMemcpyAsync(&sum, n->lacc, sizeof(double), hipMemcpyDeviceToHost, n->stream), "D2H");
    if (grad) MHIP(hipMemcpyAsync(grad, n->g, sizeof(float) * count, hipMemcpyDeviceToHost, n->stream), "D2H");
    MHIP(hipStreamSynchronize(n->stream), "gradient");
    if (loss) *loss = (float)(sum / (double)nout);
    return 0;
}

// Training data (normalised inputs [n][w0], targets [n][wL]) kept on the device.
int ctl_mlp_set_data(ctl_mlp* n, const float* x, const float* t, int64_t rows) {
    ctl::clear_error();
    if (!n || !x || !t || rows <= 0) return ctl::fail(CTL_E_ARGS, "bad arguments");
    MHIP(hipSetDevice(n->device), "hipSetDevice");
    if (n->dX) { (void)hipFree(n->dX); n->dX = nullptr; }
    if (n->dY) { (void)hipFree(n->dY); n->dY = nullptr; }
    MHIP(hipMalloc(&n->dX, sizeof(float) * rows * n->widths[0]), "hipMalloc");
    MHIP(hipMalloc(&n->dY, sizeof(float) * rows * n->widths[n->L]), "hipMalloc");
    MHIP(hipMemcpy(n->dX, x, sizeof(float) * rows * n->widths[0], hipMemcpyHostToDevice), "H2D");
    MHIP(hipMemcpy(n->dY, t, sizeof(float) * rows * n->widths[n->L], hipMemcpyHostToDevice), "H2D");
    if (n->idx) { (void)hipFree(n->idx); n->idx = nullptr; }
    MHIP(hipMalloc(&n->idx, sizeof(int32_t) * rows), "hipMalloc");
    n->ndata = rows;
    return 0;
}

// Mini-batch Adam over the device data: epochs of shuffled batches.
// losses[e] receives the mean training loss of epoch e.
int ctl_mlp_train(ctl_mlp* n, int32_t epochs, int32_t batch, float lr, uint64_t seed, float* losses) {
    ctl::clear_error();
    if (!n || epochs <= 0 || batch <= 0) return ctl::fail(CTL_E_ARGS, "bad arguments");
    if (!n->ndata) return ctl::fail(CTL_E_STATE, "no training data");
    MHIP(hipSetDevice(n->device), "hipSetDevice");
    int rc = ensure_train(n, batch);
    if (rc) return rc;
    std::mt19937_64 rng(seed);
    std::vector<int32_t> perm(n->ndata);
    for (long i = 0; i < n->ndata; ++i) perm[i] = (int32_t)i;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const long total = (long)batch * n->widths[n->L];
    for (int ep = 0; ep < epochs; ++ep) {
        // one upload of the epoch's permutation; the loss stays on the device
        // until the epoch ends, so the batches run without host round trips
        std::shuffle(perm.begin(), perm.end(), rng);
        MHIP(hipMemcpyAsync(n->idx, perm.data(), sizeof(int32_t) * n->ndata, hipMemcpyHostToDevice, n->stream), "H2D");
        MHIP(hipMemsetAsync(n->lacc, 0, sizeof(double) * (1 + n->nloss), n->stream), "memset");
        long nb = 0;
        for (long s0 = 0; s0 + batch <= n->ndata; s0 += batch) {
            load_input(n, n->dX, n->idx + s0, batch, true);
            forward(n, batch, nullptr, n->dY, n->idx + s0);
            n->step += 1;
            const AdamArgs q{lr, b1, b2, eps, 1.0f - std::pow(b1, (float)n->step), 1.0f - std::pow(b2, (float)n->step)};
            backward(n, batch, &q);
            ++nb;
        }
        hipLaunchKernelGGL(loss_sum, dim3(1), dim3(256), 0, n->stream, n->lacc + 1, n->lacc, n->nloss);
        MHIP(hipGetLastError(), "train launch");
        double sum = 0.0;
        MHIP(hipMemcpyAsync(&sum, n->lacc, sizeof(double), hipMemcpyDeviceToHost, n->stream), "D2H");
        MHIP(hipStreamSynchronize(n->stream), "train");
        if (losses) losses[ep] = nb ? (float)(sum / ((double)total * nb)) : NAN;
    }
    return 0;
}

void ctl_mlp_destroy(ctl_mlp* n) {
    if (!n) return;
    (void)hipSetDevice(n->device);
    for (auto* own : {&n->allocs, &n->abuf, &n->tbuf, &n->hbuf}) free_all(*own);
    if (n->dX) (void)hipFree(n->dX);
    if (n->dY) (void)hipFree(n->dY);
    if (n->idx) (void)hipFree(n->idx);
    if (n->stream) (void)hipStreamDestroy(n->stream);
    delete n;
}

}  // extern "C"
