// mlp_host.h -- host-side state of an ecm_mlp handle, shared by the MLP
// runtime (mlp_api.cpp) and the step (sim_api.cpp), plus the kernel
// launchers of mlp_kernels.hip.
#pragma once

#include "../../include/ecm_mlp.h"
#include "host_util.h"
#include "mlp.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

namespace ecm {
namespace mlp {

// in: 0 [n][8] chunks of 8 BF16 per agent, 1 the same tiled (chunk c of agent
// i at ((i / 32) * 8 + c) * 32 + i % 32), 2 [n][64] FP32.
hipError_t launch_mlp_infer(const void* feat, int in, const uint32_t* n_dev, int n_host, const void* frags,
                            const float* bias, float theta, uint32_t* mask, float2* vel, float* raw, int n_cu,
                            hipStream_t st);

// One batch: forward, backward, gradient and (grad null) one Adam step.
struct TrainBatch {
    const int32_t* perm;         // rows of x, label and v, or null: in order
    const void* x;
    const uint32_t* label;
    const float2* v;
    int n;
    float pos_w, vel_w;
    void* frags;                 // [kNTrainFrags][64] packed weights, in and (Adam) out
    const float* params;
    void *h[3], *dz[3], *dy;     // [n][128], [n][128], [n][16] BF16
    float* bias_part;            // [max_blocks][kNBiasParams + 1]
    int max_blocks;
    float* part;                 // [train_chunks(n)][kDwFloats]
    float *w, *m, *v2;
    float lr, b1, b2, eps, bc1, bc2;
    float* grad;
    bool first;                  // the loss of this batch starts the sum
    float* loss;                 // += the batch's mean loss
};
// Batch chunks of the weight gradients: at least 128 rows each, few enough
// that summing their 172 KB of partial sums stays cheap.
inline int train_chunks(int n) { return n <= 128 ? 1 : (n >= 96 * 128 ? 96 : (n + 127) / 128); }
hipError_t launch_train_pack(const float* params, void* frags, hipStream_t st);
hipError_t launch_train_batch(const TrainBatch& t, hipStream_t st);
hipError_t launch_fill_f32(float* p, float v, long n, hipStream_t st);
hipError_t launch_copy_f32(float* to, const float* from, long n, hipStream_t st);
hipError_t launch_pack(const float* P, void* frags, float* bias, hipStream_t st);

}  // namespace mlp
}  // namespace ecm

// 16 bytes = 8 BF16 values
struct bf16x8_t { uint32_t w[4]; };

struct ecm_mlp {
    int dev = 0;
    hipStream_t stream = nullptr;
    int n_cu = 256;
    // parameters: FP32 master (grads: the gradient, then the loss), packed inference fragments and biases, and
    // the fragments of a training run (which leaves the others alone)
    ecm::DBuf<float> params, grads, adam_m, adam_v;
    ecm::DBuf<bf16x8_t> frags, tfrags;
    bool tpacked = false;            // tfrags hold the current parameters
    ecm::DBuf<float> pbias;
    int64_t adam_t = 0;
    // dataset
    ecm::DBuf<bf16x8_t> ds_x;      // [cap][8]
    ecm::DBuf<uint32_t> ds_label;  // [cap]
    ecm::DBuf<float2> ds_v;        // [cap]
    ecm::DBuf<uint32_t> ds_count;  // [1] device append counter
    int64_t ds_cap = 0;
    // page-locked staging of host batches and results, 4 MiB from the first
    // call on that goes through it (stage_page_locked)
    unsigned char* stage = nullptr;
    bool host_called = false;
    // staged host batch, for batch size in_batch
    int in_batch = 0;
    ecm::DBuf<bf16x8_t> xb;
    ecm::DBuf<uint32_t> lb;
    ecm::DBuf<float2> vb;
    ecm::DBuf<float> y;
    // training workspace for batch size ws_batch
    int ws_batch = 0;
    ecm::DBuf<int32_t> perm;
    ecm::DBuf<bf16x8_t> h1, h2, h3, dz1, dz2, dz3, dy;
    ecm::DBuf<float> part, bias_part;
};

// Packs the current parameters into the inference layout (stream-ordered).
int ecm_mlp_pack(ecm_mlp* m);
