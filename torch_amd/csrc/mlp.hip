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
// registers, forwards and backwards, with no exchange between waves.  The
// k-order this implies inside each 32-wide K step (kperm) is built into the
// weight fragments, which are kept packed in the order the lanes read them:
// one conflict-free 16-byte LDS read (or one contiguous 1 KB L2 read per wave)
// per fragment.  Row-major weights in LDS, whose 256-byte rows put the 16
// lanes of a row group on the same banks, ran the 2^20-cell inference in
// 258 us (408 TFLOP/s); the fragments, staged by 16-byte copies, run it in 157
// us (669 TFLOP/s).
//
// Training of a batch is three launches:
//   mlp_train_kernel    forward, loss and data gradients, 16 cells per wave,
//                       SiLU derivatives in registers; writes the activations
//                       and their gradients in bfloat16, cells contiguous
//   mlp_wgrad_kernel    weight gradients dZ^T H as split-K products whose
//                       operands are read as fragments straight from those
//                       arrays (cells are the contraction index), no LDS
//   reduce_adam_kernel  fixed-order sums of the partials, Adam, and the new
//                       weights into their fragments
// A batch of 65,536 took 2,750 us per step as one tiled GEMM launch per
// product with scalar operand loads, FP32 pre-activations in memory and a
// serial sum of up to 1,024 bias partials per thread; it takes 161 us (87 in
// the fused kernel, 33 in the weight gradients, 13 in the sums and Adam).  All
// sums run in a fixed order: training is deterministic.
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

// Logistic function from the hardware base-2 exponential and reciprocal
// (about 1 ulp each): the activations that follow from it keep 8 significant
// bits, and the gradients are summed from bfloat16 operands.
__device__ __forceinline__ float sigmoid_f(float z) {
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * z));
}

// k-permutation of one 32-wide K step: lane group q holds, after a layer's
// 16x16 D tiles 2s and 2s+1, the features 32s + 4q + e (e < 4) and
// 32s + 16 + 4q + (e - 4) (e >= 4) as its 8 B-operand entries.  kslot is its
// inverse: the place 8 q + e of position k.
__device__ __forceinline__ int kslot(int k) { return k < 16 ? 8 * (k >> 2) + (k & 3) : 8 * ((k - 16) >> 2) + 4 + (k & 3); }

// Place of element (row m, column k) of a fragment grid with `nks` K steps
// per row tile, permuted columns.
__device__ __forceinline__ int frag_at(int base, int nks, int m, int k) {
    const int s = kslot(k & 31);
    return (base + (m >> 4) * nks + (k >> 5)) * MLP_FRAG + ((s >> 3) * 16 + (m & 15)) * 8 + (s & 7);
}

// Writes weight i of the master layout into its forward and backward
// fragments (the padding stays as it was set at creation: zero).
__device__ __forceinline__ void pack_weight(int i, float w, bf16_t* __restrict__ packed) {
    const bf16_t v = to_bf16(w);
    bf16_t* bwd = packed + MLP_NFF * MLP_FRAG;
    if (i < MLP_H * MLP_IN) {  // W1: lane group 0 carries the 8 features, unpermuted
        const int o = i / MLP_IN, c = i % MLP_IN;
        packed[(o >> 4) * MLP_FRAG + (o & 15) * 8 + c] = v;
        return;
    }
    i -= MLP_H * MLP_IN;
    const int l = i / (MLP_H * MLP_H);
    if (l < 3) {
        const int o = (i / MLP_H) % MLP_H, c = i % MLP_H;
        packed[frag_at(8 + l * 32, 4, o, c)] = v;
        bwd[frag_at(8 + l * 32, 4, c, o)] = v;
    } else {
        const int o = (i - 3 * MLP_H * MLP_H) / MLP_H, c = i % MLP_H;
        packed[frag_at(8 + 96, 4, o, c)] = v;
        bwd[frag_at(0, 1, c, o)] = v;
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
    u32x4 w[MLP_NFF * 64];   // forward fragments, 108 KB
    float b[4 * MLP_H + 16]; // biases, the output layer's padded with zeros
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

// Sums of 16 values over the 16 lanes of a row: lane r returns the sum of
// v[r].  Each step halves the values a lane carries: it keeps those of its
// own side of a lane bit and adds its partner's, through DPP (row mirror,
// half mirror, quad swaps).  15 steps and no branch; a rotation sum and a
// guarded LDS add per value made 137 branches per 16 cells, which kept the
// scheduler from overlapping the fragment loads.
__device__ __forceinline__ float row_sums(float (&v)[16], int r) {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = ((r & 8) ? v[i + 8] : v[i]) + dpp_f<0x140>((r & 8) ? v[i] : v[i + 8]);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = ((r & 4) ? v[i + 4] : v[i]) + dpp_f<0x141>((r & 4) ? v[i] : v[i + 4]);
#pragma unroll
    for (int i = 0; i < 2; ++i) v[i] = ((r & 2) ? v[i + 2] : v[i]) + dpp_f<0x4E>((r & 2) ? v[i] : v[i + 2]);
    return ((r & 1) ? v[1] : v[0]) + dpp_f<0xB1>((r & 1) ? v[0] : v[1]);
}

// Stores the two bfloat16 pairs (features f, f+1 and f+2, f+3 of the lane's
// cell r) of a 16-cell tile as cells-contiguous rows dst[feature][32]: lanes
// 2j and 2j+1 exchange, so that each writes two cells of one feature of each
// pair (4-byte stores, 32 contiguous bytes per feature).
__device__ __forceinline__ void store_rows(bf16_t* __restrict__ dst, int f, int r, unsigned int p0, unsigned int p1) {
    const unsigned int sel = (r & 1) ? 0x03020706u : 0x05040100u;
    const unsigned int n0 = __builtin_amdgcn_update_dpp(0, p0, 0xB1, 0xf, 0xf, true);
    const unsigned int n1 = __builtin_amdgcn_update_dpp(0, p1, 0xB1, 0xf, 0xf, true);
    unsigned int* d = reinterpret_cast<unsigned int*>(dst);
    const unsigned int o = (unsigned int)((f + (r & 1)) * 16 + (r >> 1));
    d[o] = __builtin_amdgcn_perm(n0, p0, sel);
    d[o + 32] = __builtin_amdgcn_perm(n1, p1, sel);  // two features on: 64 bf16
}

constexpr int TRAIN_THREADS = 512, TRAIN_WAVES = TRAIN_THREADS / 64;

struct TrainLDS {
    NetLDS net;
    float gb[TRAIN_WAVES][4 * MLP_H + 4];  // bias gradients of each wave's cells
    float loss[TRAIN_WAVES];
};

// Data gradient through SiLU of one layer: dz = g ds, its sums over the
// cells into gb (lane (q, r) keeps those of the features 64 i + 16 (r / 4) +
// 4 q + r % 4), bfloat16 rows for the weight gradients, and the next B
// operand.
template <int NKS>
__device__ __forceinline__ void train_backward(const u32x4* __restrict__ w, const u32x4 (&g)[NKS][1],
                                               const float (&ds)[32], u32x4 (&out)[4][1], bf16_t* __restrict__ rows,
                                               float (&gb)[2], int lane) {
    const int q = lane >> 4, r = lane & 15;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        float d[16];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int t = 4 * i + j;
            f32x4 acc[1] = {f32x4{0.f, 0.f, 0.f, 0.f}};
            row_tile<NKS, 1>(w, t, lane, g, acc);
#pragma unroll
            for (int e = 0; e < 4; ++e) d[4 * j + e] = acc[0][e] * ds[t * 4 + e];
            const unsigned int p0 = pack_bf16(d[4 * j], d[4 * j + 1]), p1 = pack_bf16(d[4 * j + 2], d[4 * j + 3]);
            out[t >> 1][0][(t & 1) * 2] = p0;
            out[t >> 1][0][(t & 1) * 2 + 1] = p1;
            store_rows(rows, t * 16 + 4 * q, r, p0, p1);
        }
        gb[i] += row_sums(d, r);
    }
}

// Forward layer keeping ds = silu'(z) in registers (FP32) and writing the
// activations' rows.
template <int NKS>
__device__ __forceinline__ void train_forward(const u32x4* w, const float* b, const u32x4 (&x)[NKS][1], float (&ds)[32],
                                              u32x4 (&h)[4][1], bf16_t* __restrict__ rows, int lane) {
    const int q = lane >> 4, r = lane & 15;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        f32x4 acc[1] = {*reinterpret_cast<const f32x4*>(b + t * 16 + 4 * q)};
        row_tile<NKS, 1>(w, t, lane, x, acc);
        float a[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float z = acc[0][e], s = sigmoid_f(z);
            ds[t * 4 + e] = s * (1.0f + z * (1.0f - s));
            a[e] = z * s;
        }
        const unsigned int p0 = pack_bf16(a[0], a[1]), p1 = pack_bf16(a[2], a[3]);
        h[t >> 1][0][(t & 1) * 2] = p0;
        h[t >> 1][0][(t & 1) * 2 + 1] = p1;
        store_rows(rows, t * 16 + 4 * q, r, p0, p1);
    }
}

// Loss 0.5/B sum m_o (y - t)^2; dy = m (y - t) / B.  When err_head >= 0 the
// target of output err_head is log10(|y0 - t0| * ln10 + 1e-5) of the current
// prediction (no gradient through it).  Eight waves share the forward
// fragments in LDS; the backward ones, read once per 16 cells, come from L2
// (both sets do not fit in 160 KB).  Bound by the latency of those reads and
// the SiLU: 87 us for 65,536 cells, at most one workgroup per CU so that the
// 108 KB are staged once.
// 128 registers hold the SiLU derivatives of the four layers, which leaves
// two waves per SIMD.
__global__ __launch_bounds__(TRAIN_THREADS) void mlp_train_kernel(const bf16_t* __restrict__ packed,
                                                                 const float* __restrict__ bias,
                                                                 const float* __restrict__ feat,
                                                                 const float* __restrict__ target, int B, float m0,
                                                                 float m1, float m2, int err_head, TrainBuffers tb) {
    __shared__ TrainLDS s;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: scalar addresses
    const int q = lane >> 4, r = lane & 15;
    stage_net(s.net, packed, bias, tid, TRAIN_THREADS);
    const int ntiles = 2 * ((B + 31) / 32);  // whole blocks of 32 cells: padding cells get zero gradients
    float gb[4][2] = {}, gbo[3] = {0.f, 0.f, 0.f};
    float loss = 0.f;
    for (int tile = blockIdx.x * TRAIN_WAVES + wave; tile < ntiles; tile += gridDim.x * TRAIN_WAVES) {
        // as in the inference kernel; the backward fragments' base is made
        // opaque here too, or their addresses are hoisted and spill
        const u32x4* wb = reinterpret_cast<const u32x4*>(packed + MLP_NFF * MLP_FRAG);
        asm volatile("" : "+s"(wb) : : "memory");
        const int c = tile * 16 + r;
        const long long blk = tile >> 1;
        const int half = (tile & 1) * 16;
        const auto rows = [&](bf16_t* base) { return base + blk * (MLP_H * 32) + half; };
        u32x4 x1[1][1], ha[4][1], hb[4][1];
        x1[0][0] = load_features(feat, c, B, q);
        if (q == 0) {
            bf16_t* d = tb.h[0] + blk * (MLP_IN * 32) + half + r;
#pragma unroll
            for (int i = 0; i < MLP_IN; ++i) d[i * 32] = (bf16_t)(x1[0][0][i >> 1] >> ((i & 1) * 16));
        }
        float z1[32], z2[32], z3[32], z4[32];
        train_forward<1>(s.net.w, s.net.b, x1, z1, ha, rows(tb.h[1]), lane);
        train_forward<4>(s.net.w + 8 * 64, s.net.b + MLP_H, ha, z2, hb, rows(tb.h[2]), lane);
        train_forward<4>(s.net.w + 40 * 64, s.net.b + 2 * MLP_H, hb, z3, ha, rows(tb.h[3]), lane);
        train_forward<4>(s.net.w + 72 * 64, s.net.b + 3 * MLP_H, ha, z4, hb, rows(tb.h[4]), lane);
        f32x4 y[1] = {*reinterpret_cast<const f32x4*>(s.net.b + 4 * MLP_H + 4 * q)};
        row_tile<4, 1>(s.net.w + 104 * 64, 0, lane, hb, y);
        // lane group 0 holds the outputs of cell c
        float dy[3] = {0.f, 0.f, 0.f};
        if (q == 0 && c < B) {
            const float ms[3] = {m0, m1, m2};
            const float t0 = target[(long long)c * MLP_NOUT];
#pragma unroll
            for (int o = 0; o < MLP_NOUT; ++o) {
                float t = target[(long long)c * MLP_NOUT + o];
                if (o == err_head) t = log10f(fabsf(y[0][0] - t0) * 2.302585093f + 1e-5f);
                const float d = y[0][o] - t;
                loss += 0.5f * ms[o] * d * d;
                dy[o] = ms[o] * d / (float)B;
            }
        }
        u32x4 g[1][1] = {{u32x4{pack_bf16(dy[0], dy[1]), pack_bf16(dy[2], 0.f), 0u, 0u}}};
        if (q == 0) {
            bf16_t* d = tb.dz[5] + blk * (4 * 32) + half + r;
#pragma unroll
            for (int o = 0; o < MLP_NOUT; ++o) d[o * 32] = (bf16_t)(g[0][0][o >> 1] >> ((o & 1) * 16));
        }
#pragma unroll
        for (int o = 0; o < MLP_NOUT; ++o) gbo[o] += dy[o];
        train_backward<1>(wb, g, z4, ha, rows(tb.dz[4]), gb[3], lane);
        train_backward<4>(wb + 72 * 64, ha, z3, hb, rows(tb.dz[3]), gb[2], lane);
        train_backward<4>(wb + 40 * 64, hb, z2, ha, rows(tb.dz[2]), gb[1], lane);
        train_backward<4>(wb + 8 * 64, ha, z1, hb, rows(tb.dz[1]), gb[0], lane);
    }
#pragma unroll
    for (int l = 0; l < 4; ++l)
#pragma unroll
        for (int i = 0; i < 2; ++i) s.gb[wave][l * MLP_H + 64 * i + 16 * (r >> 2) + 4 * q + (r & 3)] = gb[l][i];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        loss += __shfl_xor(loss, off, 64);
#pragma unroll
        for (int o = 0; o < MLP_NOUT; ++o) gbo[o] += __shfl_xor(gbo[o], off, 64);
    }
    if (lane == 0) {
        s.loss[wave] = loss;
#pragma unroll
        for (int o = 0; o < MLP_NOUT; ++o) s.gb[wave][4 * MLP_H + o] = gbo[o];
    }
    __syncthreads();
    for (int i = tid; i < (int)MLP_NB; i += TRAIN_THREADS) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < TRAIN_WAVES; ++w) v += s.gb[w][i];
        tb.bpart[(long long)blockIdx.x * MLP_NB + i] = v;
    }
    if (tid == 0) {
        float v = 0.f;
        for (int w = 0; w < TRAIN_WAVES; ++w) v += s.loss[w];
        tb.loss_part[blockIdx.x] = v;
    }
}

// Fragment of 16 feature rows x 32 cells of block `blk`: lane (q, r) takes
// the 8 cells 8q.. of row m + r, zero for rows past `rows`.
__device__ __forceinline__ bf16x8 load_rows(const bf16_t* __restrict__ a, long long blk, int rows, int m, int q, int r) {
    u32x4 v = {0u, 0u, 0u, 0u};
    if (m + r < rows) v = *reinterpret_cast<const u32x4*>(a + (blk * rows + m + r) * 32 + q * 8);
    return as_bf16x8(v);
}

// C tile (rows m.., columns n..) of a gradient [.][ldn] into this chunk's partial.
__device__ __forceinline__ void store_tile(float* __restrict__ p, int ldn, int rows, int m, int n, int q, int r,
                                           const f32x4& c) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (m + 4 * q + e < rows && n + r < ldn) p[(m + 4 * q + e) * ldn + n + r] = c[e];
}

// Weight gradients of chunk blockIdx.x (`nblk` blocks of 32 cells): job 0..2
// the 128 x 128 layers (a 64 x 64 quadrant per wave), job 3 the first and the
// output layer.  Bound by the latency of the fragment reads: two blocks in
// flight and up to 128 chunks took 65,536 cells from 66 to 33 us, and the
// longer sum of partials in reduce_adam_kernel from 10 to 13.
__global__ __launch_bounds__(256) void mlp_wgrad_kernel(int blocks, int nblk, TrainBuffers tb) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = lane >> 4, r = lane & 15, job = blockIdx.y;
    const long long b0 = (long long)blockIdx.x * nblk, b1 = min((long long)blocks, b0 + nblk);
    float* part = tb.wpart + (long long)blockIdx.x * MLP_NW;
    if (job < 3) {
        const bf16_t* dz = tb.dz[job + 2];
        const bf16_t* h = tb.h[job + 1];
        const int m0 = (wave >> 1) * 64, n0 = (wave & 1) * 64;
        f32x4 acc[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
        for (long long blk = b0; blk < b1; ++blk) {
            bf16x8 a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                a[i] = load_rows(dz, blk, MLP_H, m0 + i * 16, q, r);
                b[i] = load_rows(h, blk, MLP_H, n0 + i * 16, q, r);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        float* p = part + MLP_H * MLP_IN + job * MLP_H * MLP_H;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) store_tile(p, MLP_H, MLP_H, m0 + i * 16, n0 + j * 16, q, r, acc[i][j]);
        return;
    }
    f32x4 c1[2], c5[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) c1[i] = c5[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (long long blk = b0; blk < b1; ++blk) {
        const bf16x8 x = load_rows(tb.h[0], blk, MLP_IN, 0, q, r);
        bf16x8 dy;
        {
            u32x4 v = {0u, 0u, 0u, 0u};
            if (r < MLP_NOUT) v = *reinterpret_cast<const u32x4*>(tb.dz[5] + (blk * 4 + r) * 32 + q * 8);
            dy = as_bf16x8(v);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int f = (wave * 2 + i) * 16;
            c1[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(load_rows(tb.dz[1], blk, MLP_H, f, q, r), x, c1[i], 0, 0, 0);
            c5[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(dy, load_rows(tb.h[4], blk, MLP_H, f, q, r), c5[i], 0, 0, 0);
        }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int f = (wave * 2 + i) * 16;
        store_tile(part, MLP_IN, MLP_H, f, 0, q, r, c1[i]);
        store_tile(part + MLP_H * MLP_IN + 3 * MLP_H * MLP_H, MLP_H, MLP_NOUT, 0, f, q, r, c5[i]);
    }
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

// Gradients from the partials: a thread per weight (chunks in ascending
// order), then a wave per bias (64 interleaved sums, added by a shuffle
// tree); with a.update also Adam and the new weights' fragments.
__global__ __launch_bounds__(256) void reduce_adam_kernel(TrainBuffers tb, int nz, int nwg, float* __restrict__ gW,
                                                          float* __restrict__ gb, AdamArgs a) {
    if (blockIdx.x < REDUCE_WBLOCKS) {
        const int i = blockIdx.x * 256 + threadIdx.x;
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
    const int i = (blockIdx.x - REDUCE_WBLOCKS) * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= (int)MLP_NB) return;
    float g = 0.f;
    for (int k = lane; k < nwg; k += 64) g += tb.bpart[(long long)k * MLP_NB + i];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) g += __shfl_xor(g, off, 64);
    if (lane == 0) {
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
                                  int B, float m0, float m1, float m2, int err_head, const TrainBuffers& t, int* nwg,
                                  hipStream_t stream) {
    const int tiles = 2 * ((B + 31) / 32);
    int nb = (tiles + TRAIN_WAVES - 1) / TRAIN_WAVES;
    if (nb > MLP_TRAIN_MAX_WG) nb = MLP_TRAIN_MAX_WG;
    *nwg = nb;
    hipLaunchKernelGGL(mlp_train_kernel, dim3((unsigned)nb), dim3(TRAIN_THREADS), 0, stream, packed, bias, feat,
                       target, B, m0, m1, m2, err_head, t);
    return hipGetLastError();
}

hipError_t launch_mlp_weight_grad(int B, const TrainBuffers& t, int* nz, hipStream_t stream) {
    const int blocks = (B + 31) / 32;
    const int nblk = (blocks + MLP_TRAIN_MAX_NZ - 1) / MLP_TRAIN_MAX_NZ;
    *nz = (blocks + nblk - 1) / nblk;
    hipLaunchKernelGGL(mlp_wgrad_kernel, dim3((unsigned)*nz, 4), dim3(256), 0, stream, blocks, nblk, t);
    return hipGetLastError();
}

hipError_t launch_mlp_reduce_adam(const TrainBuffers& t, int nz, int nwg, float* gW, float* gb, const AdamArgs& a,
                                  hipStream_t stream) {
    hipLaunchKernelGGL(reduce_adam_kernel, dim3(REDUCE_WBLOCKS + (unsigned)((MLP_NB + 3) / 4)), dim3(256), 0, stream, t,
                       nz, nwg, gW, gb, a);
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
