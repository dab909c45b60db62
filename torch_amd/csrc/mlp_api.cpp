// mlp_api.cpp -- C ABI of the surrogate MLP: parameters, fused inference,
// and training (forward, loss, backward and Adam) over the kernels of
// mlp.hip.  Gradients are partial sums added in a fixed order, so training is
// deterministic.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <vector>

#include "../../include/torchgpu.h"
#include "mlp.hpp"

using tg::MLP_H;
using tg::MLP_IN;
using tg::MLP_NB;
using tg::MLP_NW;

struct torchgpu_mlp {
    hipStream_t stream = nullptr;
    int max_batch = 0;
    int nsm = 256;
    long long step = 0;
    float* W = nullptr;   // fp32 master weights [MLP_NW]
    float* b = nullptr;   // fp32 biases [MLP_NB]
    uint16_t* packed = nullptr;  // the weights as bf16 MFMA fragments [MLP_PACKED]
    float *gW = nullptr, *gb = nullptr;
    float *mW = nullptr, *vW = nullptr, *mb = nullptr, *vb = nullptr;
    tg::TrainBuffers t = {};     // batch workspace for up to max_batch cells
};

namespace {

#define HIP_CHECK(call)                                      \
    do {                                                     \
        hipError_t e_ = (call);                              \
        if (e_ != hipSuccess) {                              \
            std::fprintf(stderr, "torchgpu mlp: %s: %s\n", #call, hipGetErrorString(e_)); \
            return TORCHGPU_ERR_HIP;                         \
        }                                                    \
    } while (0)

// Gradients of a batch (and, with adam.update, the Adam step).
int loss_grad(torchgpu_mlp* m, const float* feat, const float* target, int B, const float* w3, int err_head,
              float* loss, const tg::AdamArgs& adam) {
    if (B <= 0 || B > m->max_batch) return TORCHGPU_ERR_INVALID_ARG;
    const float w0 = w3 ? w3[0] : 1.f, w1 = w3 ? w3[1] : 1.f, w2 = w3 ? w3[2] : 1.f;
    int nz = 0;
    HIP_CHECK(tg::launch_mlp_train_fused(m->packed, m->b, feat, target, B, w0, w1, w2, err_head ? 2 : -1, m->t,
                                         m->stream));
    HIP_CHECK(tg::launch_mlp_weight_grad(B, m->t, &nz, m->stream));
    HIP_CHECK(tg::launch_mlp_reduce_adam(B, m->t, nz, m->gW, m->gb, adam, m->stream));
    if (loss) {
        std::vector<float> lp((B + 255LL) / 256);
        HIP_CHECK(hipMemcpyAsync(lp.data(), m->t.loss_part, lp.size() * sizeof(float), hipMemcpyDeviceToHost, m->stream));
        HIP_CHECK(hipStreamSynchronize(m->stream));
        double s = 0;
        for (float v : lp) s += v;
        *loss = (float)(s / B);
    }
    return TORCHGPU_OK;
}

}  // namespace

extern "C" {

int torchgpu_mlp_create(int max_batch, void* stream, torchgpu_mlp** out) {
    if (!out || max_batch <= 0) return TORCHGPU_ERR_INVALID_ARG;
    *out = nullptr;
    torchgpu_mlp* m = new torchgpu_mlp();
    m->max_batch = max_batch;
    m->stream = (hipStream_t)stream;  // NULL: the null (default) stream
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
        m->nsm = prop.multiProcessorCount;
    const long long blocks = ((long long)max_batch + 31) / 32;
    bool ok = true;
    auto alloc = [&](void** p, size_t bytes) { ok = ok && hipMalloc(p, bytes) == hipSuccess; };
    alloc((void**)&m->W, MLP_NW * 4);
    alloc((void**)&m->b, MLP_NB * 4);
    alloc((void**)&m->packed, tg::MLP_PACKED * 2);
    alloc((void**)&m->gW, MLP_NW * 4);
    alloc((void**)&m->gb, MLP_NB * 4);
    alloc((void**)&m->mW, MLP_NW * 4);
    alloc((void**)&m->vW, MLP_NW * 4);
    alloc((void**)&m->mb, MLP_NB * 4);
    alloc((void**)&m->vb, MLP_NB * 4);
    alloc((void**)&m->t.h[0], blocks * 32 * MLP_IN * 2);
    for (int L = 1; L <= 4; ++L) {
        alloc((void**)&m->t.h[L], blocks * 32 * MLP_H * 2);
        alloc((void**)&m->t.dz[L], blocks * 32 * MLP_H * 2);
    }
    alloc((void**)&m->t.dz[5], blocks * 32 * 4 * 2);
    const long long nz = blocks < tg::MLP_TRAIN_MAX_NZ ? blocks : tg::MLP_TRAIN_MAX_NZ;
    alloc((void**)&m->t.cell, blocks * 32 * sizeof(tg::mlp_f32x4));
    alloc((void**)&m->t.bsum, blocks * 2 * 4 * MLP_H * 4);
    alloc((void**)&m->t.wpart, nz * MLP_NW * 4);
    alloc((void**)&m->t.opart, (max_batch + 255LL) / 256 * tg::MLP_NOUT * 4);
    alloc((void**)&m->t.loss_part, (max_batch + 255LL) / 256 * 4);
    if (!ok) {
        torchgpu_mlp_destroy(m);
        return TORCHGPU_ERR_HIP;
    }
    std::vector<float> zw(MLP_NW, 0.f), zb(MLP_NB, 0.f);
    for (float* p : {m->mW, m->vW}) (void)hipMemcpy(p, zw.data(), MLP_NW * 4, hipMemcpyHostToDevice);
    for (float* p : {m->mb, m->vb}) (void)hipMemcpy(p, zb.data(), MLP_NB * 4, hipMemcpyHostToDevice);
    // the fragments' padding stays zero
    std::vector<uint16_t> zp(tg::MLP_PACKED, 0);
    (void)hipMemcpy(m->packed, zp.data(), tg::MLP_PACKED * 2, hipMemcpyHostToDevice);
    *out = m;
    return TORCHGPU_OK;
}

void torchgpu_mlp_destroy(torchgpu_mlp* m) {
    if (!m) return;
    (void)hipStreamSynchronize(m->stream);
    std::vector<void*> ptrs = {m->W, m->b, m->packed, m->gW, m->gb, m->mW, m->vW, m->mb, m->vb, m->t.cell,
                               m->t.bsum, m->t.wpart, m->t.opart, m->t.loss_part};
    for (int L = 0; L <= 4; ++L) ptrs.push_back(m->t.h[L]);
    for (int L = 1; L <= 5; ++L) ptrs.push_back(m->t.dz[L]);
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    delete m;
}

int torchgpu_mlp_set_params(torchgpu_mlp* m, const float* W, const float* b) {
    if (!m || !W || !b) return TORCHGPU_ERR_INVALID_ARG;
    HIP_CHECK(hipMemcpyAsync(m->W, W, MLP_NW * 4, hipMemcpyHostToDevice, m->stream));
    HIP_CHECK(hipMemcpyAsync(m->b, b, MLP_NB * 4, hipMemcpyHostToDevice, m->stream));
    HIP_CHECK(tg::launch_mlp_pack(m->W, m->packed, m->stream));
    HIP_CHECK(hipStreamSynchronize(m->stream));
    m->step = 0;
    return TORCHGPU_OK;
}

int torchgpu_mlp_get_params(torchgpu_mlp* m, float* W, float* b) {
    if (!m) return TORCHGPU_ERR_INVALID_ARG;
    if (W) HIP_CHECK(hipMemcpyAsync(W, m->W, MLP_NW * 4, hipMemcpyDeviceToHost, m->stream));
    if (b) HIP_CHECK(hipMemcpyAsync(b, m->b, MLP_NB * 4, hipMemcpyDeviceToHost, m->stream));
    HIP_CHECK(hipStreamSynchronize(m->stream));
    return TORCHGPU_OK;
}

int torchgpu_mlp_device_weights(torchgpu_mlp* m, const uint16_t** packed, const float** b) {
    if (!m || !packed || !b) return TORCHGPU_ERR_INVALID_ARG;
    *packed = m->packed;
    *b = m->b;
    return TORCHGPU_OK;
}

int torchgpu_mlp_forward(torchgpu_mlp* m, const float* feat, int64_t B, float* y) {
    if (!m || B < 0 || (B > 0 && (!feat || !y))) return TORCHGPU_ERR_INVALID_ARG;
    HIP_CHECK(tg::launch_mlp_infer(m->packed, m->b, feat, B, y, m->nsm, m->stream));
    return TORCHGPU_OK;
}

int torchgpu_mlp_loss_grad(torchgpu_mlp* m, const float* feat, const float* target, int B, const float* w3,
                           int err_head, float* loss, float* gW, float* gb) {
    if (!m || !feat || !target) return TORCHGPU_ERR_INVALID_ARG;
    int rc = loss_grad(m, feat, target, B, w3, err_head, loss, tg::AdamArgs{});
    if (rc) return rc;
    if (gW) HIP_CHECK(hipMemcpyAsync(gW, m->gW, MLP_NW * 4, hipMemcpyDeviceToHost, m->stream));
    if (gb) HIP_CHECK(hipMemcpyAsync(gb, m->gb, MLP_NB * 4, hipMemcpyDeviceToHost, m->stream));
    HIP_CHECK(hipStreamSynchronize(m->stream));
    return TORCHGPU_OK;
}

int torchgpu_mlp_train_step(torchgpu_mlp* m, const float* feat, const float* target, int B, const float* w3,
                            int err_head, float lr, float weight_decay, float* loss) {
    if (!m || !feat || !target) return TORCHGPU_ERR_INVALID_ARG;
    if (B <= 0 || B > m->max_batch) return TORCHGPU_ERR_INVALID_ARG;
    const double step = (double)(m->step + 1);
    tg::AdamArgs a{};
    a.W = m->W; a.mW = m->mW; a.vW = m->vW;
    a.b = m->b; a.mb = m->mb; a.vb = m->vb;
    a.packed = m->packed;
    a.lr = lr; a.b1 = 0.9f; a.b2 = 0.999f; a.eps = 1e-8f; a.wd = weight_decay;
    a.bc1 = 1.f - (float)std::pow((double)a.b1, step);
    a.bc2 = 1.f - (float)std::pow((double)a.b2, step);
    a.update = 1;
    const int rc = loss_grad(m, feat, target, B, w3, err_head, loss, a);
    if (rc == TORCHGPU_OK) m->step += 1;
    return rc;
}

}  // extern "C"
