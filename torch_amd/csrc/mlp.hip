// mlp.hip -- BF16 MFMA kernels of the cooling-surrogate MLP (gfx950).
//
// Network: 8 input features -> 4 hidden layers of width 128 (SiLU) -> NOUT = 3
// outputs (d log10 T, d HII fraction, log10 of the estimated relative T
// error).  Every product takes bfloat16 operands and accumulates in FP32 with
// v_mfma_f32_16x16x32_bf16.
//
// Fragment layout.  Layers are computed transposed (D = W . H^T, output
// features along MFMA rows, cells along columns), so that the FP32
// accumulator of one layer, after SiLU and rounding, is directly the B
// operand of the next and a wave carries its cells through every layer in
// registers, forwards and backwards, with no exchange between waves.  Inside a
// 32-wide K step that takes a permutation: of the columns (kslot) in the
// inference fragments, of the rows (row_feature) in the training ones, whose
// products so add their terms in the features' order.  The fragments are kept
// packed in the order the lanes read them: one conflict-free 16-byte LDS read
// (or one contiguous 1 KB L2 read per wave) per fragment.  Row-major weights
// in LDS, whose 256-byte rows put the 16 lanes of a row group on the same
// banks, ran the 2^20-cell inference in 258 us (408 TFLOP/s); the fragments,
// staged by 16-byte copies, run it in 157 us (669 TFLOP/s).
//
// Training of a batch is three launches:
//   mlp_train_kernel    forward, loss and data gradients, 16 cells per wave,
//                       SiLU derivatives in registers; writes the activations
//                       and their gradients in bfloat16, cells contiguous, and
//                       the bias-gradient terms of its cells
//   mlp_wgrad_kernel    weight gradients dZ^T H as split-K products whose
//                       operands are read as fragments straight from those
//                       arrays (cells are the contraction index), no LDS; loss
//                       and output-bias gradients of 256 cells
//   reduce_adam_kernel  fixed-order sums of the partials, Adam, and the new
//                       weights into their fragments
// A batch of 65,536 took 2,700 us per step as one tiled GEMM launch per
// product with scalar operand loads, FP32 pre-activations in memory and a
// serial sum of up to 1,024 bias partials per thread; it takes 156 us (101 in
// the fused kernel, 38 in the weight gradients, 17 in the sums and Adam), the
// same bits: every sum runs in that form's order.  With the hardware
// exponential and reciprocal in the SiLU, and sums in whatever order suits the
// launches, it took 126 us (87, 33, 13 in a trace), activations up to 1e-6 off and weights
// 5e-4 after four steps.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "mlp.hpp"

namespace tg {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
// four floats of a caller's array, which is only float-aligned
typedef f32x4 f32x4_u __attribute__((aligned(4)));
typedef uint16_t bf16_t;

// float -> bfloat16 bits, round to nearest even (NaN -> quiet NaN)
__device__ __forceinline__ bf16_t to_bf16(float x) {
    unsigned int u = __float_as_uint(x);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (bf16_t)0x7fc0;
    u += 0x7fffu + ((u >> 16) & 1u);
    return (bf16_t)(u >> 16);
}
// two floats -> two bfloat16 (the hardware conversion, round to nearest even)
__device__ __forceinline__ unsigned int pack_bf16(float lo, float hi) {
    return __builtin_bit_cast(unsigned int, __builtin_convertvector((f32x2){lo, hi}, bf16x2));
}
__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

// Logistic function of the inference kernel, from the hardware base-2
// exponential and reciprocal.  The product below is rounded before the
// exponential, so the relative error grows with |z|: 1e-7 near 0, 1e-6 at z =
// -20.  The activations that follow from it keep 8 significant bits.
__device__ __forceinline__ float sigmoid_f(float z) {
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * z));
}

// k-permutation of one 32-wide K step (inference): lane group q holds, after a
// layer's 16x16 D tiles 2s and 2s+1, the features 32s + 4q + e (e < 4) and
// 32s + 16 + 4q + (e - 4) (e >= 4) as its 8 B-operand entries.  kslot is its
// inverse: the place 8 q + e of position k.
__device__ __forceinline__ int kslot(int k) { return k < 16 ? 8 * (k >> 2) + (k & 3) : 8 * ((k - 16) >> 2) + 4 + (k & 3); }

// Row permutation of a layer's 16-row tiles (training): row 4q + e of tile
// 2s + h is feature 32s + 8q + 4h + e, which leaves the 8 features 32s + 8q ..
// of the next K step with lane group q, in their order.
__device__ __forceinline__ int row_feature(int t, int q) { return 32 * (t >> 1) + 8 * q + 4 * (t & 1); }  // e = 0
__device__ __forceinline__ int feature_tile(int f) { return 2 * (f >> 5) + ((f >> 2) & 1); }
__device__ __forceinline__ int feature_row(int f) { return 4 * ((f >> 3) & 3) + (f & 3); }

// Place of row `row` of tile t and slot s (0 .. 31) of K step ks in a fragment
// grid with `nks` K steps per tile.
__device__ __forceinline__ int frag_at(int base, int nks, int t, int row, int ks, int s) {
    return (base + t * nks + ks) * MLP_FRAG + ((s >> 3) * 16 + row) * 8 + (s & 7);
}

// Writes weight i of the master layout into its fragments (the padding stays
// as it was set at creation: zero).
__device__ __forceinline__ void pack_weight(int i, float w, bf16_t* __restrict__ packed) {
    const bf16_t v = to_bf16(w);
    bf16_t* fwd = packed + MLP_NFF * MLP_FRAG;
    bf16_t* bwd = fwd + MLP_NFF * MLP_FRAG;
    if (i < MLP_H * MLP_IN) {  // W1: lane group 0 carries the 8 features
        const int o = i / MLP_IN, c = i % MLP_IN;
        packed[frag_at(0, 1, o >> 4, o & 15, 0, c)] = v;
        fwd[frag_at(0, 1, feature_tile(o), feature_row(o), 0, c)] = v;
        return;
    }
    i -= MLP_H * MLP_IN;
    const int l = i / (MLP_H * MLP_H);
    const int c = i % MLP_H, o = l < 3 ? (i / MLP_H) % MLP_H : (i - 3 * MLP_H * MLP_H) / MLP_H;
    if (l < 3) {
        const int base = 8 + l * 32;
        packed[frag_at(base, 4, o >> 4, o & 15, c >> 5, kslot(c & 31))] = v;
        fwd[frag_at(base, 4, feature_tile(o), feature_row(o), c >> 5, c & 31)] = v;
        bwd[frag_at(base, 4, feature_tile(c), feature_row(c), o >> 5, o & 31)] = v;
    } else {
        packed[frag_at(8 + 96, 4, 0, o, c >> 5, kslot(c & 31))] = v;
        fwd[frag_at(8 + 96, 4, 0, o, c >> 5, c & 31)] = v;
        bwd[frag_at(0, 1, feature_tile(c), feature_row(c), 0, o)] = v;
    }
}

__global__ void pack_kernel(const float* __restrict__ W, bf16_t* __restrict__ packed) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < (int)MLP_NW) pack_weight(i, W[i], packed);
}

// ---------------------------------------------------------------------------
// One layer of a wave's cells.  w: the layer's fragments (row tile t, K step
// k at t nks + k), in LDS or global memory; init: the accumulators' start
// (bias, or zero).
// ---------------------------------------------------------------------------
template <int NKS, int NT>
__device__ __forceinline__ void row_tile(const u32x4* w, int t, int lane, const u32x4 (&x)[NKS][NT], f32x4 (&acc)[NT]) {
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
        // uniform base + 32-bit lane offset: no per-fragment vector addresses
        const char* f = reinterpret_cast<const char*>(w + (t * NKS + ks) * 64);
        const bf16x8 av = as_bf16x8(*reinterpret_cast<const u32x4*>(f + (unsigned int)lane * 16u));
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, as_bf16x8(x[ks][nt]), acc[nt], 0, 0, 0);
    }
}

// The features of cell `c` (zero past n) as the layer-1 B operand: lane
// group 0 carries all 8.
__device__ __forceinline__ u32x4 load_features(const float* __restrict__ feat, long long c, long long n, int q) {
    u32x4 x = {0u, 0u, 0u, 0u};
    if (q == 0 && c < n) {
        const f32x4 a = *reinterpret_cast<const f32x4_u*>(feat + c * MLP_IN);
        const f32x4 b = *reinterpret_cast<const f32x4_u*>(feat + c * MLP_IN + 4);
        x = u32x4{pack_bf16(a[0], a[1]), pack_bf16(a[2], a[3]), pack_bf16(b[0], b[1]), pack_bf16(b[2], b[3])};
    }
    return x;
}

struct NetLDS {
    float b[4 * MLP_H + 16]; // biases, the output layer's padded with zeros
    u32x4 w[MLP_NFF * 64];   // forward fragments, 108 KB
};

__device__ __forceinline__ void stage_net(NetLDS& s, const bf16_t* __restrict__ packed, const float* __restrict__ bias,
                                          int tid, int nthreads) {
    const u32x4* src = reinterpret_cast<const u32x4*>(packed);
    for (int i = tid; i < MLP_NFF * 64; i += nthreads) s.w[i] = src[i];
    for (int i = tid; i < 4 * MLP_H + 16; i += nthreads) s.b[i] = i < (int)MLP_NB ? bias[i] : 0.f;
    __syncthreads();
}

// ---------------------------------------------------------------------------
// Inference: features [n][8] fp32 (normalised), outputs [n][NOUT] fp32.
// Bound by the SiLU's two transcendentals per hidden unit beside the MFMA:
// 512 units of about 30 issue cycles each per cell against 196 / 32 MFMAs of
// 16 cycles.  The bias enters as the accumulators' start.
// ---------------------------------------------------------------------------
template <int NKS, int NT>
__device__ __forceinline__ void infer_layer(const u32x4* w, const float* b, const u32x4 (&x)[NKS][NT],
                                            u32x4 (&h)[4][NT], int lane) {
    const int q = lane >> 4;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        f32x4 acc[NT];
        const f32x4 bv = *reinterpret_cast<const f32x4*>(b + t * 16 + 4 * q);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[nt] = bv;
        row_tile<NKS, NT>(w, t, lane, x, acc);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            f32x4 a;
#pragma unroll
            for (int e = 0; e < 4; ++e) a[e] = acc[nt][e] * sigmoid_f(acc[nt][e]);
            h[t >> 1][nt][(t & 1) * 2] = pack_bf16(a[0], a[1]);
            h[t >> 1][nt][(t & 1) * 2 + 1] = pack_bf16(a[2], a[3]);
        }
    }
}

constexpr int INFER_THREADS = 512;
constexpr int INFER_NT = 2;  // 32 cells per wave per iteration

__global__ __launch_bounds__(INFER_THREADS) void mlp_infer_kernel(const bf16_t* __restrict__ packed,
                                                                 const float* __restrict__ bias,
                                                                 const float* __restrict__ feat, long long n,
                                                                 const unsigned long long* __restrict__ n_dev,
                                                                 float* __restrict__ y) {
    __shared__ NetLDS s;
    constexpr int NT = INFER_NT, NW = INFER_THREADS / 64;
    if (n_dev) n = (long long)*n_dev;
    // a block with no cells (the grid is sized for the largest queue) leaves
    // before staging the weights
    if ((long long)blockIdx.x * NW * 16 * NT >= n) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    stage_net(s, packed, bias, tid, INFER_THREADS);
    const int q = lane >> 4, r = lane & 15;
    const long long ntiles = (n + 16 * NT - 1) / (16 * NT);
    for (long long tile = (long long)blockIdx.x * NW + wave; tile < ntiles; tile += (long long)gridDim.x * NW) {
        // keeps the (loop-invariant) LDS weight fragments from being hoisted
        // out of the tile loop into registers
        asm volatile("" ::: "memory");
        const long long c0 = tile * 16 * NT;
        u32x4 x1[1][NT], ha[4][NT], hb[4][NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) x1[0][nt] = load_features(feat, c0 + nt * 16 + r, n, q);
        infer_layer<1, NT>(s.w, s.b, x1, ha, lane);
        infer_layer<4, NT>(s.w + 8 * 64, s.b + MLP_H, ha, hb, lane);
        infer_layer<4, NT>(s.w + 40 * 64, s.b + 2 * MLP_H, hb, ha, lane);
        infer_layer<4, NT>(s.w + 72 * 64, s.b + 3 * MLP_H, ha, hb, lane);
        f32x4 acc[NT];
        const f32x4 bo = *reinterpret_cast<const f32x4*>(s.b + 4 * MLP_H + 4 * q);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[nt] = bo;
        row_tile<4, NT>(s.w + 104 * 64, 0, lane, hb, acc);
        if (q == 0) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const long long c = c0 + nt * 16 + r;
                if (c < n) {
#pragma unroll
                    for (int e = 0; e < MLP_NOUT; ++e) y[c * MLP_NOUT + e] = acc[nt][e];
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Training
// ---------------------------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ float dpp_f(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}

// One value of a tile, in the sums below: lane j of each quad, to all four.
template <int J>
__device__ __forceinline__ float quad_f(float x) { return dpp_f<0x55 * J>(x); }

// Bias-gradient terms of two features over a tile's 16 cells, in a fixed
// order: lanes 0-7 of a row return a's sum, lanes 8-15 b's.  Lanes 0-7 of a
// tile are eight consecutive cells and lanes 8-15 the eight 16 further on
// (tile_cell); a quad adds its four cells and the four 16 further on one
// after another, then the two quads are added.  14 steps for two features,
// without a branch.
__device__ __forceinline__ float tile_sums(float a, float b) {
    const int ai = __float_as_int(a), bi = __float_as_int(b);
    const float x = __int_as_float(__builtin_amdgcn_update_dpp(ai, bi, 0x128, 0xf, 0xc, false));  // cells 0-7 of either
    const float y = __int_as_float(__builtin_amdgcn_update_dpp(bi, ai, 0x128, 0xf, 0x3, false));  // and 8-15
    float s = quad_f<0>(x);
    s += quad_f<1>(x);
    s += quad_f<2>(x);
    s += quad_f<3>(x);
    s += quad_f<0>(y);
    s += quad_f<1>(y);
    s += quad_f<2>(y);
    s += quad_f<3>(y);
    return s + dpp_f<0x141>(s);
}

// The cell, within a block of 32, of lane r of the block's tile `half`.
__device__ __forceinline__ int tile_cell(int half, int r) { return 8 * half + (r & 7) + 16 * (r >> 3); }

// Stores the two bfloat16 pairs (features f .. f + 3 of one cell) of tile t as
// cells-contiguous rows dst[feature][32]: lanes 2j and 2j+1 exchange, so that
// each writes two cells of one feature of each pair.  at: the lane's place,
// row_place(), in units of two cells.
__device__ __forceinline__ unsigned int row_place(int q, int c) { return (unsigned int)((8 * q + (c & 1)) * 16 + (c >> 1)); }
__device__ __forceinline__ void store_rows(bf16_t* __restrict__ dst, int t, unsigned int at, int lane, unsigned int p0,
                                           unsigned int p1) {
    const unsigned int sel = (lane & 1) ? 0x03020706u : 0x05040100u;
    const unsigned int n0 = __builtin_amdgcn_update_dpp(0, p0, 0xB1, 0xf, 0xf, true);
    const unsigned int n1 = __builtin_amdgcn_update_dpp(0, p1, 0xB1, 0xf, 0xf, true);
    unsigned int* d = reinterpret_cast<unsigned int*>(dst) + row_feature(t, 0) * 16;
    d[at] = __builtin_amdgcn_perm(n0, p0, sel);
    d[at + 32] = __builtin_amdgcn_perm(n1, p1, sel);  // two features on: 64 bf16
}

constexpr int TRAIN_THREADS = 512, TRAIN_WAVES = TRAIN_THREADS / 64;

// Data gradient through SiLU of one layer: dz = g ds, its sums over the
// tile's cells into sums[128], bfloat16 rows for the weight gradients, and the
// next B operand.
template <int NKS>
__device__ __forceinline__ void train_backward(const u32x4* __restrict__ w, const u32x4 (&g)[NKS][1],
                                               const float (&ds)[32], u32x4 (&out)[4][1], bf16_t* __restrict__ rows,
                                               float* __restrict__ sums, unsigned int at, int lane) {
    const int q = lane >> 4, r = lane & 15;
    float keep[2] = {0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        float d[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int t = 2 * s + h;
            f32x4 acc[1] = {f32x4{0.f, 0.f, 0.f, 0.f}};
            row_tile<NKS, 1>(w, t, lane, g, acc);
#pragma unroll
            for (int e = 0; e < 4; ++e) d[h][e] = acc[0][e] * ds[t * 4 + e];
            const unsigned int p0 = pack_bf16(d[h][0], d[h][1]), p1 = pack_bf16(d[h][2], d[h][3]);
            out[s][0][2 * h] = p0;
            out[s][0][2 * h + 1] = p1;
            store_rows(rows, t, at, lane, p0, p1);
        }
        // lane r keeps the sums of tile 2s + r / 8, s = 2 i + (r / 4) % 2,
        // element r % 4 in keep[i]
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float v = tile_sums(d[0][e], d[1][e]);
            keep[s >> 1] = (r & 7) == (s & 1) * 4 + e ? v : keep[s >> 1];
        }
    }
    const int f = 32 * ((r >> 2) & 1) + 8 * q + 4 * (r >> 3) + (r & 3);
    sums[f] = keep[0];
    sums[64 + f] = keep[1];
}

// Forward layer keeping ds = silu'(z) in registers (FP32) and writing the
// activations' rows.  SiLU and its derivative from expf and exact divisions:
// the hardware exponential and reciprocal of the inference kernel are up to
// 1e-6 off at z = -20, and the gradients see it.
template <int NKS>
__device__ __forceinline__ void train_forward(const u32x4* w, const float* b, const u32x4 (&x)[NKS][1], float (&ds)[32],
                                              u32x4 (&h)[4][1], bf16_t* __restrict__ rows, unsigned int at,
                                              int lane) {
    const int q = lane >> 4;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        f32x4 acc[1] = {f32x4{0.f, 0.f, 0.f, 0.f}};
        row_tile<NKS, 1>(w, t, lane, x, acc);
        const f32x4 bv = *reinterpret_cast<const f32x4*>(b + row_feature(t, 0) + 8 * q);
        float a[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float z = acc[0][e] + bv[e], u = 1.0f + expf(-z), s = 1.0f / u;
            ds[t * 4 + e] = s * (1.0f + z * (1.0f - s));
            a[e] = z / u;
            // computed here: left until the backward pass, z and u would both
            // be held (and spilled)
            asm volatile("" : "+v"(ds[t * 4 + e]));
        }
        const unsigned int p0 = pack_bf16(a[0], a[1]), p1 = pack_bf16(a[2], a[3]);
        h[t >> 1][0][(t & 1) * 2] = p0;
        h[t >> 1][0][(t & 1) * 2 + 1] = p1;
        store_rows(rows, t, at, lane, p0, p1);
    }
}

// Loss 0.5/B sum m_o (y - t)^2; dy = m (y - t) / B.  When err_head >= 0 the
// target of output err_head is log10(|y0 - t0| * ln10 + 1e-5) of the current
// prediction (no gradient through it).  Eight waves share the forward
// fragments in LDS; the backward ones, read once per 16 cells, come from L2
// (both sets do not fit in 160 KB).  Bound by the SiLU's exponential and two
// divisions per unit and the latency of those reads, 101 us for 65,536 cells; at
// most one workgroup per CU so that the 108 KB are staged once.
// 128 registers hold the SiLU derivatives of the four layers, which leaves
// two waves per SIMD.
__global__ __launch_bounds__(TRAIN_THREADS) void mlp_train_kernel(const bf16_t* __restrict__ packed,
                                                                 const float* __restrict__ bias,
                                                                 const float* __restrict__ feat,
                                                                 const float* __restrict__ target, int B, float m0,
                                                                 float m1, float m2, int err_head, TrainBuffers tb) {
    __shared__ NetLDS net;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: scalar addresses
    const int q = lane >> 4, r = lane & 15;
    const bf16_t* fwd = packed + MLP_NFF * MLP_FRAG;
    stage_net(net, fwd, bias, tid, TRAIN_THREADS);
    const int ntiles = 2 * ((B + 31) / 32);  // whole blocks of 32 cells: padding cells get zero gradients
    for (int tile = blockIdx.x * TRAIN_WAVES + wave; tile < ntiles; tile += gridDim.x * TRAIN_WAVES) {
        // as in the inference kernel; the backward fragments' base is made
        // opaque here too, or their addresses are hoisted and spill
        const u32x4* wb = reinterpret_cast<const u32x4*>(fwd + MLP_NFF * MLP_FRAG);
        asm volatile("" : "+s"(wb) : : "memory");
        const long long blk = tile >> 1;
        const int cb = tile_cell(tile & 1, r);
        const long long c = blk * 32 + cb;
        const unsigned int at = row_place(q, cb);
        const auto rows = [&](bf16_t* base) { return base + blk * (MLP_H * 32); };
        float* sums = tb.bsum + (long long)tile * (4 * MLP_H);
        u32x4 x1[1][1], ha[4][1], hb[4][1];
        x1[0][0] = load_features(feat, c, B, q);
        if (q == 0) {
            bf16_t* d = tb.h[0] + blk * (MLP_IN * 32) + cb;
#pragma unroll
            for (int i = 0; i < MLP_IN; ++i) d[i * 32] = (bf16_t)(x1[0][0][i >> 1] >> ((i & 1) * 16));
        }
        float z1[32], z2[32], z3[32], z4[32];
        train_forward<1>(net.w, net.b, x1, z1, ha, rows(tb.h[1]), at, lane);
        train_forward<4>(net.w + 8 * 64, net.b + MLP_H, ha, z2, hb, rows(tb.h[2]), at, lane);
        train_forward<4>(net.w + 40 * 64, net.b + 2 * MLP_H, hb, z3, ha, rows(tb.h[3]), at, lane);
        train_forward<4>(net.w + 72 * 64, net.b + 3 * MLP_H, ha, z4, hb, rows(tb.h[4]), at, lane);
        f32x4 y[1] = {f32x4{0.f, 0.f, 0.f, 0.f}};
        row_tile<4, 1>(net.w + 104 * 64, 0, lane, hb, y);
        y[0] += *reinterpret_cast<const f32x4*>(net.b + 4 * MLP_H + 4 * q);
        // lane group 0 holds the outputs of cell c
        f32x4 dy = {0.f, 0.f, 0.f, 0.f};  // and the cell's loss
        if (q == 0 && c < B) {
            const float ms[3] = {m0, m1, m2};
            const float t0 = target[c * MLP_NOUT];
#pragma unroll
            for (int o = 0; o < MLP_NOUT; ++o) {
                float t = target[c * MLP_NOUT + o];
                if (o == err_head) t = log10f(fabsf(y[0][0] - t0) * 2.302585093f + 1e-5f);
                const float d = y[0][o] - t;
                dy[3] += 0.5f * ms[o] * d * d;
                dy[o] = ms[o] * d / (float)B;
            }
        }
        u32x4 g[1][1] = {{u32x4{pack_bf16(dy[0], dy[1]), pack_bf16(dy[2], 0.f), 0u, 0u}}};
        if (q == 0) {
            tb.cell[c] = dy;
            bf16_t* d = tb.dz[5] + blk * (4 * 32) + cb;
#pragma unroll
            for (int o = 0; o < MLP_NOUT; ++o) d[o * 32] = (bf16_t)(g[0][0][o >> 1] >> ((o & 1) * 16));
        }
        train_backward<1>(wb, g, z4, ha, rows(tb.dz[4]), sums + 3 * MLP_H, at, lane);
        train_backward<4>(wb + 72 * 64, ha, z3, hb, rows(tb.dz[3]), sums + 2 * MLP_H, at, lane);
        train_backward<4>(wb + 40 * 64, hb, z2, ha, rows(tb.dz[2]), sums + MLP_H, at, lane);
        train_backward<4>(wb + 8 * 64, ha, z1, hb, rows(tb.dz[1]), sums, at, lane);
    }
}

// Fragment of 16 feature rows x 32 cells of block `blk`: lane (q, r) takes
// the 8 cells 8q.. of row m + r, zero for rows past `valid` of the `rows`
// stored.
__device__ __forceinline__ bf16x8 load_rows(const bf16_t* __restrict__ a, long long blk, int rows, int valid, int m, int q,
                                            int r) {
    u32x4 v = {0u, 0u, 0u, 0u};
    if (valid >= MLP_H || m + r < valid) v = *reinterpret_cast<const u32x4*>(a + (blk * rows + m + r) * 32 + q * 8);
    return as_bf16x8(v);
}

// C tile (rows m.., columns n..) of a gradient [.][ldn] into this chunk's partial.
__device__ __forceinline__ void store_tile(float* __restrict__ p, int ldn, int rows, int m, int n, int q, int r,
                                           const f32x4& c) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (m + 4 * q + e < rows && n + r < ldn) p[(m + 4 * q + e) * ldn + n + r] = c[e];
}

// Loss and output-bias gradient of 256 cells: the loss as a binary tree, each
// output's gradient one cell after another.
__device__ __forceinline__ void output_sums(const TrainBuffers& tb, int blk, int B) {
    __shared__ f32x4 v[256];
    __shared__ float tree[256];
    const int tid = threadIdx.x;
    const long long c = (long long)blk * 256 + tid;
    const f32x4 x = c < B ? tb.cell[c] : f32x4{0.f, 0.f, 0.f, 0.f};
    v[tid] = x;
    tree[tid] = x[3];
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (tid < s) tree[tid] += tree[tid + s];
        __syncthreads();
    }
    if (tid == 0) tb.loss_part[blk] = tree[0];
    if (tid < MLP_NOUT) {
        const float* col = reinterpret_cast<const float*>(v) + tid;
        float s = 0.f;
#pragma unroll 16
        for (int i = 0; i < 256; ++i) s += col[4 * i];  // zeros past the last cell
        tb.opart[(long long)blk * MLP_NOUT + tid] = s;
    }
}

// Weight gradients of `nblk` blocks of 32 cells: workgroup (chunk, job) of
// the first nz * WGRAD_JOBS, jobs 0 .. 11 a 64 x 64 quadrant of a 128 x 128
// layer (32 x 32 per wave), jobs 12 and 13 half of the first and the output
// layer; the workgroups past them sum the outputs of 256 cells each.  Bound
// by the latency of the fragment reads, eight blocks in flight per wave: 38 us for
// 65,536 cells (33 as 128 chunks of 64 x 64 tiles per wave, another order of
// sums).
// At most 32 chunks, whose sums are then added in order: a gradient is the
// same however the batch is spread over the chip.
constexpr int WGRAD_JOBS = 14, WGRAD_AHEAD = 8;
__global__ __launch_bounds__(256) void mlp_wgrad_kernel(int B, int blocks, int nblk, int nz, TrainBuffers tb) {
    if ((int)blockIdx.x >= nz * WGRAD_JOBS) {
        output_sums(tb, (int)blockIdx.x - nz * WGRAD_JOBS, B);
        return;
    }
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = lane >> 4, r = lane & 15, job = blockIdx.x % WGRAD_JOBS, chunk = blockIdx.x / WGRAD_JOBS;
    const long long b0 = (long long)chunk * nblk, b1 = min((long long)blocks, b0 + nblk);
    float* part = tb.wpart + (long long)chunk * MLP_NW;
    if (job < 12) {
        const int l = job >> 2;
        const bf16_t* dz = tb.dz[l + 2];
        const bf16_t* h = tb.h[l + 1];
        const int m0 = ((job >> 1) & 1) * 64 + (wave >> 1) * 32, n0 = (job & 1) * 64 + (wave & 1) * 32;
        f32x4 acc[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        const auto step = [&](auto nb, long long blk) {  // nb blocks, their loads first
            constexpr int N = decltype(nb)::value;
            bf16x8 a[N][2], b[N][2];
#pragma unroll
            for (int k = 0; k < N; ++k)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    a[k][i] = load_rows(dz, blk + k, MLP_H, MLP_H, m0 + i * 16, q, r);
                    b[k][i] = load_rows(h, blk + k, MLP_H, MLP_H, n0 + i * 16, q, r);
                }
#pragma unroll
            for (int k = 0; k < N; ++k)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[k][i], b[k][j], acc[i][j], 0, 0, 0);
        };
        long long blk = b0;
        for (; blk + WGRAD_AHEAD <= b1; blk += WGRAD_AHEAD) step(std::integral_constant<int, WGRAD_AHEAD>{}, blk);
        for (; blk < b1; ++blk) step(std::integral_constant<int, 1>{}, blk);
        float* p = part + MLP_H * MLP_IN + l * MLP_H * MLP_H;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) store_tile(p, MLP_H, MLP_H, m0 + i * 16, n0 + j * 16, q, r, acc[i][j]);
        return;
    }
    const int f = ((job - 12) * 4 + wave) * 16;
    f32x4 c1 = {0.f, 0.f, 0.f, 0.f}, c5 = c1;
    const auto step = [&](auto nb, long long blk) {
        constexpr int N = decltype(nb)::value;
        bf16x8 a1[N], b1[N], a5[N], b5[N];
#pragma unroll
        for (int k = 0; k < N; ++k) {
            a1[k] = load_rows(tb.dz[1], blk + k, MLP_H, MLP_H, f, q, r);
            b1[k] = load_rows(tb.h[0], blk + k, MLP_IN, MLP_IN, 0, q, r);
            a5[k] = load_rows(tb.dz[5], blk + k, 4, MLP_NOUT, 0, q, r);
            b5[k] = load_rows(tb.h[4], blk + k, MLP_H, MLP_H, f, q, r);
        }
#pragma unroll
        for (int k = 0; k < N; ++k) {
            c1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[k], b1[k], c1, 0, 0, 0);
            c5 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a5[k], b5[k], c5, 0, 0, 0);
        }
    };
    long long blk = b0;
    for (; blk + WGRAD_AHEAD <= b1; blk += WGRAD_AHEAD) step(std::integral_constant<int, WGRAD_AHEAD>{}, blk);
    for (; blk < b1; ++blk) step(std::integral_constant<int, 1>{}, blk);
    store_tile(part, MLP_IN, MLP_H, f, 0, q, r, c1);
    store_tile(part + MLP_H * MLP_IN + 3 * MLP_H * MLP_H, MLP_H, MLP_NOUT, 0, f, q, r, c5);
}

// Adam on one fp32 master parameter; returns its new value.
__device__ __forceinline__ float adam_step(const AdamArgs& a, float p, float g, float* m, float* v, float wd) {
    const float gi = g + wd * p;
    const float mi = a.b1 * *m + (1.f - a.b1) * gi;
    const float vi = a.b2 * *v + (1.f - a.b2) * gi * gi;
    *m = mi;
    *v = vi;
    return p - a.lr * (mi / a.bc1) / (sqrtf(vi / a.bc2) + a.eps);
}

constexpr int REDUCE_WBLOCKS = (int)((MLP_NW + 255) / 256);
constexpr int REDUCE_BIAS = 16;                               // hidden biases per workgroup
constexpr int REDUCE_BBLOCKS = 4 * MLP_H / REDUCE_BIAS + 1;   // the last: the output biases
constexpr int REDUCE_CHUNK = 512;

// Gradients from the partials, each sum from the first to the last: a thread
// per weight; 16 hidden biases per workgroup, whose terms of 64 cells (four
// tiles, added in pairs) all its threads load into LDS for one thread per bias to
// add up; the output biases likewise from their sums of 256 cells.  With
// a.update also Adam and the new weights' fragments.
__global__ __launch_bounds__(256) void reduce_adam_kernel(TrainBuffers tb, int B, int nz, float* __restrict__ gW,
                                                          float* __restrict__ gb, AdamArgs a) {
    __shared__ f32x4 term[REDUCE_CHUNK][REDUCE_BIAS / 4];
    const int tid = threadIdx.x;
    if (blockIdx.x < REDUCE_WBLOCKS) {
        const int i = blockIdx.x * 256 + tid;
        if (i >= (int)MLP_NW) return;
        float g = 0.f;
#pragma unroll 8
        for (int z = 0; z < nz; ++z) g += tb.wpart[(long long)z * MLP_NW + i];
        gW[i] = g;
        if (a.update) {
            const float p = adam_step(a, a.W[i], g, a.mW + i, a.vW + i, a.wd);
            a.W[i] = p;
            pack_weight(i, p, a.packed);
        }
        return;
    }
    const int i0 = (blockIdx.x - REDUCE_WBLOCKS) * REDUCE_BIAS;
    const bool out = i0 == 4 * MLP_H;
    const int nbias = out ? MLP_NOUT : REDUCE_BIAS;
    const int tiles = 2 * ((B + 31) / 32);
    const long long n = out ? ((long long)B + 255) / 256 : ((long long)B + 63) / 64;
    const float* col = reinterpret_cast<const float*>(term) + tid;
    float g = 0.f;
    for (long long t0 = 0; t0 < n; t0 += REDUCE_CHUNK) {
        const int m = (int)min((long long)REDUCE_CHUNK, n - t0);
        __syncthreads();
        if (out) {
            for (int j = tid; j < m; j += 256) {
                const float* p = tb.opart + (t0 + j) * MLP_NOUT;
                term[j][0] = f32x4{p[0], p[1], p[2], 0.f};
            }
        } else {
            const int b4 = tid % (REDUCE_BIAS / 4);
#pragma unroll 4
            for (int j = tid / (REDUCE_BIAS / 4); j < m; j += 256 / (REDUCE_BIAS / 4)) {
                const long long t = 4 * (t0 + j);
                const f32x4* p = reinterpret_cast<const f32x4*>(tb.bsum + t * (4 * MLP_H) + i0) + b4;
                f32x4 lo = p[0] + p[MLP_H], hi = {0.f, 0.f, 0.f, 0.f};  // p[MLP_H]: the next tile
                if (t + 2 < tiles) hi = p[2 * MLP_H] + p[3 * MLP_H];
                term[j][b4] = lo + hi;
            }
        }
        __syncthreads();
        if (tid < nbias) {
#pragma unroll 16
            for (int j = 0; j < m; ++j) g += col[j * REDUCE_BIAS];
        }
    }
    if (tid < nbias) {
        const int i = i0 + tid;
        gb[i] = g;
        if (a.update) a.b[i] = adam_step(a, a.b[i], g, a.mb + i, a.vb + i, 0.f);
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
hipError_t launch_mlp_pack(const float* W, uint16_t* packed, hipStream_t stream) {
    hipLaunchKernelGGL(pack_kernel, dim3((unsigned)((MLP_NW + 255) / 256)), dim3(256), 0, stream, W, packed);
    return hipGetLastError();
}

hipError_t launch_mlp_train_fused(const uint16_t* packed, const float* bias, const float* feat, const float* target,
                                  int B, float m0, float m1, float m2, int err_head, const TrainBuffers& t,
                                  hipStream_t stream) {
    const int tiles = 2 * ((B + 31) / 32);
    int nb = (tiles + TRAIN_WAVES - 1) / TRAIN_WAVES;
    if (nb > MLP_TRAIN_MAX_WG) nb = MLP_TRAIN_MAX_WG;
    hipLaunchKernelGGL(mlp_train_kernel, dim3((unsigned)nb), dim3(TRAIN_THREADS), 0, stream, packed, bias, feat,
                       target, B, m0, m1, m2, err_head, t);
    return hipGetLastError();
}

hipError_t launch_mlp_weight_grad(int B, const TrainBuffers& t, int* nz, hipStream_t stream) {
    const int blocks = (B + 31) / 32;
    const int nblk = (blocks + MLP_TRAIN_MAX_NZ - 1) / MLP_TRAIN_MAX_NZ;
    *nz = (blocks + nblk - 1) / nblk;
    hipLaunchKernelGGL(mlp_wgrad_kernel, dim3((unsigned)(*nz * WGRAD_JOBS + (B + 255) / 256)), dim3(256), 0, stream, B,
                       blocks, nblk, *nz, t);
    return hipGetLastError();
}

hipError_t launch_mlp_reduce_adam(int B, const TrainBuffers& t, int nz, float* gW, float* gb, const AdamArgs& a,
                                  hipStream_t stream) {
    hipLaunchKernelGGL(reduce_adam_kernel, dim3(REDUCE_WBLOCKS + REDUCE_BBLOCKS), dim3(256), 0, stream, t, B, nz, gW, gb,
                       a);
    return hipGetLastError();
}

static unsigned infer_blocks(long long n, int nblocks) {
    const long long per = 16 * INFER_NT * (INFER_THREADS / 64);
    const long long nb = (n + per - 1) / per;
    return (unsigned)(nb > nblocks ? nblocks : nb);
}

hipError_t launch_mlp_infer(const uint16_t* packed, const float* bias, const float* feat, long long n, float* y,
                            int nblocks, hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(mlp_infer_kernel, dim3(infer_blocks(n, nblocks)), dim3(INFER_THREADS), 0, stream, packed, bias,
                       feat, n, (const unsigned long long*)nullptr, y);
    return hipGetLastError();
}

hipError_t launch_mlp_infer_dev(const uint16_t* packed, const float* bias, const float* feat,
                                const unsigned long long* n_dev, long long n_max, float* y, int nblocks,
                                hipStream_t stream) {
    if (n_max <= 0) return hipSuccess;
    hipLaunchKernelGGL(mlp_infer_kernel, dim3(infer_blocks(n_max, nblocks)), dim3(INFER_THREADS), 0, stream, packed,
                       bias, feat, n_max, n_dev, y);
    return hipGetLastError();
}

}  // namespace tg
