// mlp.hpp -- launch interface of the surrogate MLP kernels (mlp.hip).
// bfloat16 values are stored as their 16-bit patterns (uint16_t).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace tg {

constexpr int MLP_IN = 8;     // input features (6 used, 2 zero)
constexpr int MLP_H = 128;    // hidden width
constexpr int MLP_NOUT = 3;   // d log10 T, d HII fraction, log10 estimated relative error
// fp32 master weights: W1[128][8] | W2 | W3 | W4 [128][128] | W5[NOUT][128]
constexpr long long MLP_NW = (long long)MLP_H * MLP_IN + 3LL * MLP_H * MLP_H + (long long)MLP_NOUT * MLP_H;
// fp32 bias blob: b1 | b2 | b3 | b4 [128] | b5[NOUT]
constexpr long long MLP_NB = 4LL * MLP_H + MLP_NOUT;

// The kernels read the weights as bfloat16 MFMA A fragments (16 x 32, 64
// lanes x 8 values, 1 KB each), so that a fragment is one contiguous 16-byte
// load per lane from LDS or L2 (mlp.hip, fragment layout):
//   inference, then training forward
//     W1: 8 | W2, W3, W4: 8 row tiles x 4 K steps each | W5: 4 K steps
//   training backward
//     W5^T: 8 | W2^T, W3^T, W4^T: 8 x 4 each
constexpr int MLP_FRAG = 512;
constexpr int MLP_NFF = 8 + 3 * 32 + 4, MLP_NFB = 8 + 3 * 32;
constexpr int MLP_PACKED = (2 * MLP_NFF + MLP_NFB) * MLP_FRAG;  // bf16 values

typedef __attribute__((ext_vector_type(4))) float mlp_f32x4;

// One training batch: activations and their gradients for the weight
// gradients, bfloat16, cells in blocks of 32: [block][feature][32 cells].
struct TrainBuffers {
    uint16_t* h[5];    // H0 [.][8][32], H1..H4 [.][128][32]
    uint16_t* dz[6];   // dZ1..dZ4 [.][128][32], dZ5 = dy [.][4][32] (indices 1..5)
    mlp_f32x4* cell;   // FP32 output gradients and loss of each cell
    float* bsum;       // hidden bias-gradient terms [16-cell tile][4][128]
    float* wpart;      // weight-gradient partials [nz][MLP_NW]
    float* opart;      // output-bias partials [256 cells][NOUT]
    float* loss_part;  // [256 cells]
};
constexpr int MLP_TRAIN_MAX_WG = 256, MLP_TRAIN_MAX_NZ = 32;

// Adam state of the weights and biases; update 0: gradients only.
struct AdamArgs {
    float *W, *mW, *vW, *b, *mb, *vb;
    uint16_t* packed;
    float lr, b1, b2, eps, bc1, bc2, wd;
    int update;
};

// fp32 master weights -> the fragments
hipError_t launch_mlp_pack(const float* W, uint16_t* packed, hipStream_t stream);
// forward, loss and the data gradients of B cells
hipError_t launch_mlp_train_fused(const uint16_t* packed, const float* bias, const float* feat, const float* target,
                                  int B, float m0, float m1, float m2, int err_head, const TrainBuffers& t,
                                  hipStream_t stream);
// weight-gradient, output-bias and loss partials, then the gradients
// (fixed-order sums) and Adam
hipError_t launch_mlp_weight_grad(int B, const TrainBuffers& t, int* nz, hipStream_t stream);
hipError_t launch_mlp_reduce_adam(int B, const TrainBuffers& t, int nz, float* gW, float* gb, const AdamArgs& a,
                                  hipStream_t stream);
hipError_t launch_mlp_infer(const uint16_t* packed, const float* bias, const float* feat, long long n, float* y,
                            int nblocks, hipStream_t stream);
// as launch_mlp_infer with the cell count read from device memory (<= n_max)
hipError_t launch_mlp_infer_dev(const uint16_t* packed, const float* bias, const float* feat,
                                const unsigned long long* n_dev, long long n_max, float* y, int nblocks,
                                hipStream_t stream);

}  // namespace tg
