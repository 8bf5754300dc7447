// mlp_kernels.hip -- gfx950 kernels of the learned ORCA proposal network:
// inference (persistent, weights resident in LDS, one 32-agent MFMA tile
// per wavefront iteration) and training (forward and backward of a tile in
// registers, the weight gradients, and the Adam step).
#include "mlp_host.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

namespace ecm {
namespace mlp {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16 mfma(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// SiLU with the hardware exp2 / reciprocal (both ~1 ulp); the training
// kernels use the same expression.
constexpr float kLog2e = 1.4426950408889634f;
__device__ __forceinline__ float sigmoid_f(float z) { return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-z * kLog2e)); }
__device__ __forceinline__ float silu_f(float z) { return z * sigmoid_f(z); }

// accumulator <- bias of rows 8 j + 4 g + r (register 4 j + r)
__device__ __forceinline__ void bias_init(f32x16& acc, const float* b, int g) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float4 v = *reinterpret_cast<const float4*>(b + 8 * j + 4 * g);
        acc[4 * j + 0] = v.x;
        acc[4 * j + 1] = v.y;
        acc[4 * j + 2] = v.z;
        acc[4 * j + 3] = v.w;
    }
}

// SiLU of one m-tile, packed as B-operand chunks 2 mi and 2 mi + 1 of the
// next layer
__device__ __forceinline__ void act_pack(const f32x16& acc, bf16x8& lo, bf16x8& hi) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        lo[e] = (__bf16)silu_f(acc[e]);
        hi[e] = (__bf16)silu_f(acc[8 + e]);
    }
}

// One 128-wide hidden layer for a 32-agent tile: m-tiles one after the
// other (one live accumulator), inputs `in`, outputs `out`.
template <int NKC>
__device__ __forceinline__ void hidden_layer(const bf16x8* sw, int frag0, const float* sb, int g, int lane,
                                             const bf16x8 (&in)[NKC], bf16x8 (&out)[8]) {
#pragma unroll
    for (int mi = 0; mi < 4; ++mi) {
        f32x16 acc;
        bias_init(acc, sb + 32 * mi, g);
#pragma unroll
        for (int kc = 0; kc < NKC; ++kc) acc = mfma(sw[(frag0 + mi * NKC + kc) * 64 + lane], in[kc], acc);
        act_pack(acc, out[2 * mi], out[2 * mi + 1]);
    }
}

// Input formats: BF16 chunks per agent ([n][8] chunks of 8), the same tiled
// (chunk c of agent i at ((i / 32) * 8 + c) * 32 + i % 32), or FP32 rows that
// start on a 16-byte boundary or anywhere.
enum InferIn { kRows = 0, kTiled = 1, kF32 = 2, kF32Any = 3 };
struct InferArgs {
    const void* feat;         // 64 features per agent
    const uint32_t* n_dev;    // agent count on the device, or null
    int n_host;               // agent count when n_dev is null
    const bf16x8* frags;      // [kNFrags][64] packed A fragments
    const float* bias;        // [kNBias]
    float theta;              // slot predicted active when its logit > theta
    uint32_t* mask;           // [n] predicted active slots
    float2* vel;              // [n] velocity head (m/s), or null
    float* raw;               // [n][16] raw outputs, or null
};

// 8 FP32 features as a BF16 operand chunk, rounded to nearest even.
template <bool ALIGNED>
__device__ __forceinline__ bf16x8 load_f32(const float* p) {
    if (!ALIGNED) {
        bf16x8 v;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (__bf16)p[e];
        return v;
    }
    const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
    bf16x8 v;
    v[0] = (__bf16)a.x; v[1] = (__bf16)a.y; v[2] = (__bf16)a.z; v[3] = (__bf16)a.w;
    v[4] = (__bf16)b.x; v[5] = (__bf16)b.y; v[6] = (__bf16)b.z; v[7] = (__bf16)b.w;
    return v;
}

// 1024 threads = 16 wavefronts per workgroup, one workgroup per CU: the 88
// KiB of fragments are loaded into LDS once and every wavefront loops over
// 32-agent tiles, dealt to the workgroups first: 32,768 samples give every
// CU four tiles, one per SIMD (as 16 tiles to each of 64 CUs they took 18.5
// us).  All 64 lanes execute every MFMA (tile bounds only gate loads and
// stores).
template <int IN>
__global__ __launch_bounds__(1024) void k_mlp_infer(InferArgs a) {
    __shared__ bf16x8 sw[kNFrags * 64];
    __shared__ float sb[kNBias];
    for (int i = threadIdx.x; i < kNFrags * 64; i += blockDim.x) sw[i] = a.frags[i];
    for (int i = threadIdx.x; i < kNBias; i += blockDim.x) sb[i] = a.bias[i];
    __syncthreads();
    const int n = a.n_dev ? (int)*a.n_dev : a.n_host;
    const int lane = threadIdx.x & 63, g = lane >> 5, col = lane & 31;
    const int waves = blockDim.x >> 6;
    const int ntiles = (n + 31) >> 5;
    bf16x8 zero;
#pragma unroll
    for (int e = 0; e < 8; ++e) zero[e] = (__bf16)0.0f;
    for (int tile = (threadIdx.x >> 6) * gridDim.x + blockIdx.x; tile < ntiles; tile += gridDim.x * waves) {
        // the weights are re-read from LDS every tile: without this barrier
        // the compiler hoists all 88 fragments out of the loop and spills
        __asm__ volatile("" ::: "memory");
        const int agent = tile * 32 + col;
        const bool ok = agent < n;
        // layer 1: 64 inputs straight from HBM as B operands
        bf16x8 x[4], h[8], h2[8];
#pragma unroll
        for (int kc = 0; kc < 4; ++kc) {
            const int c = 2 * kc + g;
            if (IN >= kF32) {
                x[kc] = ok ? load_f32<IN == kF32>((const float*)a.feat + (size_t)agent * kInPad + 8 * c) : zero;
            } else {
                const size_t at = IN == kTiled ? ((size_t)tile * 8 + c) * 32 + col : (size_t)agent * 8 + c;
                x[kc] = ok ? ((const bf16x8*)a.feat)[at] : zero;
            }
        }
        hidden_layer<4>(sw, kFragL1, sb + kBiasL1, g, lane, x, h);
        hidden_layer<8>(sw, kFragL2, sb + kBiasL2, g, lane, h, h2);
        hidden_layer<8>(sw, kFragL3, sb + kBiasL3, g, lane, h2, h);
        // layer 4: 16 outputs in rows 0..15 of one padded tile
        f32x16 o;
        bias_init(o, sb + kBiasL4, g);
#pragma unroll
        for (int kc = 0; kc < 8; ++kc) o = mfma(sw[(kFragL4 + kc) * 64 + lane], h[kc], o);
        // lane pair (L, L + 32) holds rows {0-3, 8-11} and {4-7, 12-15}
        uint32_t m = 0;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 8 * j + 4 * g + r;
                if (row < kSlots && o[4 * j + r] > a.theta) m |= 1u << row;
            }
        m |= __shfl_xor(m, 32);
        if (ok) {
            if (g == 0) a.mask[agent] = m;
            else if (a.vel) a.vel[agent] = make_float2(o[6] * (1.0f / kVelScale), o[7] * (1.0f / kVelScale));
            if (a.raw) {
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) a.raw[(size_t)agent * 16 + 8 * j + 4 * g + r] = o[4 * j + r];
            }
        }
    }
}

// ------------------------------------------------------------- training

// One batch is three launches: k_train_tile runs 32-sample tiles through the
// network and back and stores the operands of the weight gradients,
// k_train_dw multiplies those out over batch chunks, k_train_step sums the
// chunks, steps Adam and repacks the weights.  (As a GEMM, an elementwise and
// a column-sum launch per layer and direction a batch of 72,000 took 1.5 ms,
// most of it in uncoalesced 2-byte loads.)  Every product takes its K axis
// in order, so activations and dz have the bits of those GEMMs.
struct TrainArgs {
    const int32_t* perm;      // sample of each batch row, or null: the rows in order
    const bf16x8* x;          // [..][8] features
    const uint32_t* label;
    const float2* v;
    int n;                    // batch rows
    float pos_w, vel_w;
    const bf16x8* frags;      // [kNTrainFrags][64]
    const float* params;      // biases
    // per batch row: [n][16] chunks of h1, h2, h3, dz1, dz2, dz3 and [n][2] of dy
    bf16x8 *h1, *h2, *h3, *dz1, *dz2, *dz3, *dy;
    float* bias_part;         // [blocks][kNBiasParams + 1] bias gradients, loss
};

// Sum of each register over the lanes' 32 samples (the columns), stored to
// the 32 rows at sums.
__device__ __forceinline__ void sum_rows(const f32x16& acc, int lane, float* sums) {
    const int r = lane & 15;
    float mine = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        float v = acc[e];
#pragma unroll
        for (int m = 1; m < 32; m <<= 1) v += __shfl_xor(v, m);
        mine = r == e ? v : mine;
    }
    if ((lane & 16) == 0) sums[8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)] = mine;
}

__device__ __forceinline__ f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int e = 0; e < 16; ++e) z[e] = 0.0f;
    return z;
}

// A 32-row accumulator tile as two B-operand chunks of 16 consecutive K each.
// Lane (column, g) holds rows 8 j + 4 g + r; a chunk wants 8 g + e.  The two
// halves of the wavefront exchange what the other's chunk half is made of.
__device__ __forceinline__ void pack_tile(const f32x16& v, bf16x8 (&out)[2]) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        bf16x8 c;
#pragma unroll
        for (int e = 0; e < 8; ++e) c[e] = (__bf16)v[8 * h + e];
        u32x4 d = __builtin_bit_cast(u32x4, c);
        const auto p = __builtin_amdgcn_permlane32_swap(d[0], d[2], false, false);
        const auto q = __builtin_amdgcn_permlane32_swap(d[1], d[3], false, false);
        d[0] = p[0]; d[2] = p[1];
        d[1] = q[0]; d[3] = q[1];
        out[h] = __builtin_bit_cast(bf16x8, d);
    }
}

// Forward, loss and backward of 32-sample tiles, one at a time per workgroup:
// wavefront w computes units [32 w, 32 w + 32) of every layer in both
// directions, with its share of the weights (45 fragments, 180 registers) and
// silu'(z) of its units in registers, and hands its two operand chunks to the
// others through LDS.  A whole tile per wavefront instead (weights in LDS,
// nothing exchanged) left each SIMD one chain of 156 products and 192
// activations: 98 us for 72,000 samples, 41 for 8,192.
__global__ __launch_bounds__(256, 1) void k_train_tile(TrainArgs a) {
    __shared__ bf16x8 xch[2][8 * 64];
    __shared__ float sb[kNBias];
    __shared__ float sums[kNBiasParams + 1];
    const int lane = threadIdx.x & 63, g = lane >> 5, col = lane & 31;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int i = threadIdx.x; i < kNBias; i += 256)
        sb[i] = i < kBiasL2   ? a.params[kOffB1 + i]
                : i < kBiasL3 ? a.params[kOffB2 + i - kBiasL2]
                : i < kBiasL4 ? a.params[kOffB3 + i - kBiasL3]
                : i - kBiasL4 < kOut ? a.params[kOffB4 + i - kBiasL4] : 0.0f;
    bf16x8 w1[4], w2[8], w3[8], w4[8], b4, b3[8], b2[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        if (k < 4) w1[k] = a.frags[(kFragL1 + 4 * w + k) * 64 + lane];
        w2[k] = a.frags[(kFragL2 + 8 * w + k) * 64 + lane];
        w3[k] = a.frags[(kFragL3 + 8 * w + k) * 64 + lane];
        w4[k] = a.frags[(kFragL4 + k) * 64 + lane];
        b3[k] = a.frags[(kFragB3 + 8 * w + k) * 64 + lane];
        b2[k] = a.frags[(kFragB2 + 8 * w + k) * 64 + lane];
    }
    b4 = a.frags[(kFragB4 + w) * 64 + lane];
    __syncthreads();
    const int ntiles = (a.n + 31) >> 5;
    const float inv_n = 1.0f / (float)a.n;
    f32x16 s1 = zero16(), s2 = zero16(), s3 = zero16(), s4 = zero16();
    float loss = 0.0f;
    int buf = 0;
    // the wavefront's chunks of one layer: to memory, and to the others; a
    // buffer is written again two exchanges later, when the barrier between
    // has seen everyone's reads
    auto give = [&](const bf16x8 (&own)[2], bf16x8* out, int row, bool ok) {
        if (ok) {
            out[(size_t)row * 16 + 4 * w + g] = own[0];
            out[(size_t)row * 16 + 4 * w + 2 + g] = own[1];
        }
        buf ^= 1;
        xch[buf][(2 * w) * 64 + lane] = own[0];
        xch[buf][(2 * w + 1) * 64 + lane] = own[1];
        __syncthreads();
    };
    auto product = [&](const bf16x8 (&wt)[8]) {
        f32x16 acc = zero16();
#pragma unroll
        for (int k = 0; k < 8; ++k) acc = mfma(wt[k], xch[buf][k * 64 + lane], acc);
        return acc;
    };
    // z = acc + bias -> (silu(z) chunks, silu'(z))
    auto activate = [&](f32x16 acc, const float* bias, f32x16& gp, bf16x8 (&own)[2]) {
        f32x16 b;
        bias_init(b, bias + 32 * w, g);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const float z = acc[e] + b[e], s = sigmoid_f(z);
            gp[e] = s * (1.0f + z * (1.0f - s));
            acc[e] = z * s;
        }
        pack_tile(acc, own);
    };
    // a tile's inputs, loaded while the tile before it is worked on
    bf16x8 nx[4];
    uint32_t nL = 0u;
    float2 nvt = make_float2(0.0f, 0.0f);
    auto fetch = [&](int tile) {
        const int row = tile * 32 + col;
        const bool ok = row < a.n;
        const size_t src = ok ? (size_t)(a.perm ? a.perm[row] : row) : 0;
        nL = ok ? a.label[src] : 0u;
        nvt = ok ? a.v[src] : make_float2(0.0f, 0.0f);
#pragma unroll
        for (int k = 0; k < 4; ++k) nx[k] = a.x[src * 8 + 2 * k + g];
    };
    fetch(blockIdx.x);
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int row = tile * 32 + col;
        const bool ok = row < a.n;
        const uint32_t L = nL;
        const float2 vt = nvt;
        bf16x8 own[2];
        f32x16 g1, g2, g3;
        {
            f32x16 acc = zero16();
#pragma unroll
            for (int k = 0; k < 4; ++k) acc = mfma(w1[k], nx[k], acc);
            if (tile + (int)gridDim.x < ntiles) fetch(tile + gridDim.x);
            activate(acc, sb + kBiasL1, g1, own);
        }
        give(own, a.h1, row, ok);
        activate(product(w2), sb + kBiasL2, g2, own);
        give(own, a.h2, row, ok);
        activate(product(w3), sb + kBiasL3, g3, own);
        give(own, a.h3, row, ok);
        // The head, in every wavefront: logits in rows 0..13 (BCE with a
        // positive-class weight over the slots that exist), velocity in rows
        // 14 and 15 (squared error against the scaled LP solution), means
        // over the batch; each wavefront adds up two of a lane's eight losses
        f32x16 d = product(w4), b;
        bias_init(b, sb + kBiasL4, g);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int c = 8 * (e >> 2) + 4 * g + (e & 3);
            const float y = d[e] + b[e];
            d[e] = 0.0f;
            if (e >= 8) continue;                    // padding rows
            if (c < kSlots) {
                if ((L >> (kLabelValidShift + c)) & 1u) {
                    const float t = (float)((L >> c) & 1u);
                    if ((e & 3) == w) {
                        const float sp = fmaxf(y, 0.0f) + log1pf(expf(-fabsf(y)));      // softplus(y)
                        loss += (t * a.pos_w * (sp - y) + (1.0f - t) * sp) * inv_n;
                    }
                    const float s = sigmoid_f(y);
                    d[e] = (s * (1.0f - t + a.pos_w * t) - a.pos_w * t) * inv_n;
                }
            } else if (ok) {
                const float err = y - (c == kSlots ? vt.x : vt.y) * kVelScale;
                if ((e & 3) == w) loss += 0.5f * a.vel_w * err * err * inv_n;
                d[e] = a.vel_w * err * inv_n;
            }
        }
        s4 += d;
        pack_tile(d, own);
        if (ok && w == 0) a.dy[(size_t)row * 2 + g] = own[0];
        f32x16 dz = mfma(b4, own[0], zero16()) * g3;
        s3 += dz;
        pack_tile(dz, own);
        give(own, a.dz3, row, ok);
        dz = product(b3) * g2;
        s2 += dz;
        pack_tile(dz, own);
        give(own, a.dz2, row, ok);
        dz = product(b2) * g1;
        s1 += dz;
        pack_tile(dz, own);
        if (ok) {
            a.dz1[(size_t)row * 16 + 4 * w + g] = own[0];
            a.dz1[(size_t)row * 16 + 4 * w + 2 + g] = own[1];
        }
    }
    sum_rows(s1, lane, sums + 32 * w);
    sum_rows(s2, lane, sums + kHid + 32 * w);
    sum_rows(s3, lane, sums + 2 * kHid + 32 * w);
    if (w == 0) {
        float* tmp = sb;                             // the padding rows go nowhere
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        sum_rows(s4, lane, tmp);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (lane < kOut) sums[3 * kHid + lane] = tmp[lane];
    }
    __shared__ float wloss[4];
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) loss += __shfl_xor(loss, m);
    if (lane == 0) wloss[w] = loss;
    __syncthreads();
    if (threadIdx.x == 0) sums[kNBiasParams] = (wloss[0] + wloss[1]) + (wloss[2] + wloss[3]);
    __syncthreads();
    for (int i = threadIdx.x; i < kNBiasParams + 1; i += 256)
        a.bias_part[(size_t)blockIdx.x * (kNBiasParams + 1) + i] = sums[i];
}

// Weight gradients of one batch chunk: dW_l = dz_l^T h_{l-1}, job l in
// blockIdx.y.  Each step takes 64 samples of both operands (16-byte loads of
// their rows), turns them to [unit][sample] in LDS and multiplies, four
// 32-row m-tiles over the four wavefronts; the next step's loads are in
// flight meanwhile.
struct DwArgs {
    const int32_t* perm;
    const bf16x8 *x, *h1, *h2, *h3, *dz1, *dz2, *dz3, *dy;
    int n, chunk;             // batch rows, rows per chunk (a multiple of kDwStep)
    float* part;              // [chunks][kDwFloats]
};
constexpr int kDwStep = 64;
constexpr int kDwStride = 72;    // LDS row of 64 samples: 16-byte aligned

__global__ __launch_bounds__(256) void k_train_dw(DwArgs p) {
    __shared__ __attribute__((aligned(16))) __bf16 As[128 * kDwStride];
    __shared__ __attribute__((aligned(16))) __bf16 Bs[128 * kDwStride];
    const int job = blockIdx.y, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const bf16x8* A = job == 0 ? p.dz3 : (job == 1 ? p.dz2 : (job == 2 ? p.dz1 : p.dy));
    const bf16x8* B = job == 0 ? p.h2 : (job == 1 ? p.h1 : (job == 2 ? p.x : p.h3));
    const int ac = job == 3 ? 2 : 16, bc = job == 2 ? 8 : 16;     // 16-byte chunks per sample
    float* out = p.part + (size_t)blockIdx.x * kDwFloats +
                 (job == 0 ? kDwOff3 : (job == 1 ? kDwOff2 : (job == 2 ? kDwOff1 : kDwOff4)));
    if (job == 3)                                                  // rows 16..31 of the one m-tile
        for (int i = tid; i < 128 * kDwStride; i += 256) As[i] = (__bf16)0.0f;
    const int s = lane, c0 = w;                                    // sample, first chunk
    const int k0 = blockIdx.x * p.chunk, k1 = min(p.n, k0 + p.chunk);
    bf16x8 zero;
#pragma unroll
    for (int e = 0; e < 8; ++e) zero[e] = (__bf16)0.0f;
    bf16x8 ra[4], rb[4];
    auto fetch = [&](int k) {
        const int row = k + s;
        const bool ok = row < k1;
        const size_t xr = job == 2 && p.perm && ok ? (size_t)p.perm[row] : (size_t)row;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int c = c0 + 4 * u;
            ra[u] = ok && c < ac ? A[(size_t)row * ac + c] : zero;
            rb[u] = ok && c < bc ? B[xr * bc + c] : zero;
        }
    };
    f32x16 acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[t][e] = 0.0f;
    // job 3: one m-tile, the wavefronts take an n-tile each
    const int m0 = job == 3 ? 0 : 32 * w, n0 = job == 3 ? 32 * w : 0, nt = job == 3 ? 1 : (job == 2 ? 2 : 4);
    fetch(k0);
    for (int k = k0; k < k1; k += kDwStep) {
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int c = c0 + 4 * u;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if (c < ac) As[(8 * c + e) * kDwStride + s] = ra[u][e];
                if (c < bc) Bs[(8 * c + e) * kDwStride + s] = rb[u][e];
            }
        }
        __syncthreads();
        if (k + kDwStep < k1) fetch(k + kDwStep);
#pragma unroll
        for (int q = 0; q < kDwStep / 16; ++q) {
            const int at = 16 * q + 8 * (lane >> 5);
            const bf16x8 av = *reinterpret_cast<const bf16x8*>(&As[(m0 + (lane & 31)) * kDwStride + at]);
#pragma unroll
            for (int t = 0; t < 4; ++t)
                if (t < nt)
                    acc[t] = mfma(av, *reinterpret_cast<const bf16x8*>(
                                          &Bs[(n0 + 32 * t + (lane & 31)) * kDwStride + at]), acc[t]);
        }
    }
    const int N = job == 2 ? kInPad : kHid, M = job == 3 ? kOut : kHid;
#pragma unroll
    for (int t = 0; t < 4; ++t)
        if (t < nt)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = m0 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
                if (m < M) out[m * N + n0 + 32 * t + (lane & 31)] = acc[t][e];
            }
}

// The batch's gradient (its chunks' and blocks' partial sums added in order),
// and then either stored (loss_grad) or taken through one Adam step with the
// new weights packed for the next batch.
struct StepArgs {
    const float* part;        // [chunks][kDwFloats]
    int chunks;
    const float* bias_part;   // [blocks][kNBiasParams + 1]
    int blocks;
    float *w, *m, *v;         // parameters and moments
    float lr, b1, b2, eps, bc1, bc2;
    __bf16* frags;            // training fragments
    float* grad;              // not null: store the gradient, no Adam step
    bool first;               // the batch's loss starts the sum at loss
    float* loss;
};

// Fragment element of weight (row, position k along its packed K axis).
__device__ __forceinline__ int frag_at(int frag0, int nkc, int row, int k) {
    return ((frag0 + (row >> 5) * nkc + (k >> 4)) * 64 + (row & 31) + 32 * ((k >> 3) & 1)) * 8 + (k & 7);
}
__device__ __forceinline__ void adam(const StepArgs& a, int i, float gi, float& wi) {
    const float mi = a.b1 * a.m[i] + (1.0f - a.b1) * gi;
    const float vi = a.b2 * a.v[i] + (1.0f - a.b2) * gi * gi;
    a.m[i] = mi;
    a.v[i] = vi;
    wi = a.w[i] - a.lr * (mi / a.bc1) / (sqrtf(vi / a.bc2) + a.eps);
    a.w[i] = wi;
}

// Blocks [0, kDwFloats / 256): one weight per thread; the rest: 16 lanes per
// bias gradient (and the loss).
__global__ __launch_bounds__(256) void k_train_step(StepArgs a) {
    constexpr int kWBlocks = kDwFloats / 256;
    if (blockIdx.x < kWBlocks) {
        const int q = blockIdx.x * 256 + threadIdx.x;
        float gi = 0.0f;
#pragma unroll 8
        for (int c = 0; c < a.chunks; ++c) gi += a.part[(size_t)c * kDwFloats + q];
        int i, fwd, bwd = -1;
        __bf16* f = a.frags;
        if (q < kDwOff1) {                                       // W3 or W2
            const bool l3 = q < kDwOff2;
            const int r = l3 ? q : q - kDwOff2, row = r >> 7, col = r & 127;
            i = (l3 ? kOffW3 : kOffW2) + r;
            fwd = frag_at(l3 ? kFragL3 : kFragL2, 8, row, col);
            bwd = frag_at(l3 ? kFragB3 : kFragB2, 8, col, row);
        } else if (q < kDwOff4) {                                // W1
            const int r = q - kDwOff1;
            i = kOffW1 + r;
            fwd = frag_at(kFragL1, 4, r >> 6, r & 63);
        } else {                                                 // W4
            const int r = q - kDwOff4, row = r >> 7, col = r & 127;
            i = kOffW4 + r;
            fwd = frag_at(kFragL4, 8, row, col);
            bwd = frag_at(kFragB4, 1, col, row);
        }
        if (a.grad) { a.grad[i] = gi; return; }
        float wi;
        adam(a, i, gi, wi);
        f[fwd] = (__bf16)wi;
        if (bwd >= 0) f[bwd] = (__bf16)wi;
        return;
    }
    const int q = (blockIdx.x - kWBlocks) * 16 + threadIdx.x / 16, l = threadIdx.x & 15;
    float gi = 0.0f;
    if (q <= kNBiasParams)
        for (int b = l; b < a.blocks; b += 16) gi += a.bias_part[(size_t)b * (kNBiasParams + 1) + q];
#pragma unroll
    for (int m = 1; m < 16; m <<= 1) gi += __shfl_xor(gi, m);
    if (l != 0 || q > kNBiasParams) return;
    if (q == kNBiasParams) { *a.loss = a.first ? gi : *a.loss + gi; return; }
    const int i = q < kHid ? kOffB1 + q : (q < 2 * kHid ? kOffB2 + q - kHid : (q < 3 * kHid ? kOffB3 + q - 2 * kHid
                                                                                              : kOffB4 + q - 3 * kHid));
    if (a.grad) { a.grad[i] = gi; return; }
    float wi;
    adam(a, i, gi, wi);
}

// Training packing of the FP32 parameters (K axes in order): one fragment per
// block, 64 lanes.
__global__ void k_train_pack(const float* P, bf16x8* frags) {
    const int f = blockIdx.x, lane = threadIdx.x;
    int frag0, nkc, off, nin, rows;
    bool back = false;
    if (f < kFragL2) { frag0 = kFragL1; nkc = 4; off = kOffW1; nin = kInPad; rows = kHid; }
    else if (f < kFragL3) { frag0 = kFragL2; nkc = 8; off = kOffW2; nin = kHid; rows = kHid; }
    else if (f < kFragL4) { frag0 = kFragL3; nkc = 8; off = kOffW3; nin = kHid; rows = kHid; }
    else if (f < kFragB4) { frag0 = kFragL4; nkc = 8; off = kOffW4; nin = kHid; rows = kOut; }
    else if (f < kFragB3) { frag0 = kFragB4; nkc = 1; off = kOffW4; nin = kHid; rows = kHid; back = true; }
    else if (f < kFragB2) { frag0 = kFragB3; nkc = 8; off = kOffW3; nin = kHid; rows = kHid; back = true; }
    else { frag0 = kFragB2; nkc = 8; off = kOffW2; nin = kHid; rows = kHid; back = true; }
    const int mi = (f - frag0) / nkc, kc = (f - frag0) % nkc, row = 32 * mi + (lane & 31);
    bf16x8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int k = 16 * kc + 8 * (lane >> 5) + e;
        v[e] = (__bf16)(row < rows ? (back ? P[off + k * nin + row] : P[off + row * nin + k]) : 0.0f);
    }
    frags[f * 64 + lane] = v;
}

__global__ void k_fill_f32(float* p, float v, long n) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) p[i] = v;
}

__global__ void k_copy_f32(float* to, const float* from, long n) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) to[i] = from[i];
}

// Inference packing of the FP32 parameters (fragment layout in mlp.h).
__global__ void k_pack(const float* P, bf16x8* frags, float* bias) {
    const int f = blockIdx.x, lane = threadIdx.x;          // one fragment per block, 64 lanes
    int mi, kc, nin;
    const float* W;
    bool hidden_in;
    int rows;
    if (f < kFragL2) { const int q = f - kFragL1; mi = q / 4; kc = q % 4; W = P + kOffW1; nin = kInPad; hidden_in = false; rows = kHid; }
    else if (f < kFragL3) { const int q = f - kFragL2; mi = q / 8; kc = q % 8; W = P + kOffW2; nin = kHid; hidden_in = true; rows = kHid; }
    else if (f < kFragL4) { const int q = f - kFragL3; mi = q / 8; kc = q % 8; W = P + kOffW3; nin = kHid; hidden_in = true; rows = kHid; }
    else { const int q = f - kFragL4; mi = 0; kc = q; W = P + kOffW4; nin = kHid; hidden_in = true; rows = kOut; }
    const int row = 32 * mi + (lane & 31);
    bf16x8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int k = 16 * kc + 8 * (lane >> 5) + e;
        const int col = hidden_in ? hidden_perm(k) : k;
        v[e] = (__bf16)(row < rows ? W[row * nin + col] : 0.0f);
    }
    frags[f * 64 + lane] = v;
    if (f == 0) {
        for (int i = lane; i < kNBias; i += 64) {
            float b = 0.0f;
            if (i < kBiasL2) b = P[kOffB1 + i];
            else if (i < kBiasL3) b = P[kOffB2 + i - kBiasL2];
            else if (i < kBiasL4) b = P[kOffB3 + i - kBiasL3];
            else if (i - kBiasL4 < kOut) b = P[kOffB4 + i - kBiasL4];
            bias[i] = b;
        }
    }
}

// ------------------------------------------------------------- launchers
static inline int cdiv(long a, long b) { return (int)((a + b - 1) / b); }

hipError_t launch_mlp_infer(const void* feat, int in, const uint32_t* n_dev, int n_host, const void* frags,
                            const float* bias, float theta, uint32_t* mask, float2* vel, float* raw, int n_cu,
                            hipStream_t st) {
    InferArgs a{feat, n_dev, n_host, (const bf16x8*)frags, bias, theta, mask, vel, raw};
    // no more workgroups than tiles when the count is known here
    const dim3 g(n_dev ? n_cu : std::max(1, std::min(n_cu, cdiv(n_host, 32)))), b(1024);
    if (in == kF32 && ((uintptr_t)feat & 15u) == 0) hipLaunchKernelGGL(k_mlp_infer<kF32>, g, b, 0, st, a);
    else if (in == kF32) hipLaunchKernelGGL(k_mlp_infer<kF32Any>, g, b, 0, st, a);
    else if (in == kTiled) hipLaunchKernelGGL(k_mlp_infer<kTiled>, g, b, 0, st, a);
    else hipLaunchKernelGGL(k_mlp_infer<kRows>, g, b, 0, st, a);
    return hipGetLastError();
}

hipError_t launch_train_pack(const float* params, void* frags, hipStream_t st) {
    hipLaunchKernelGGL(k_train_pack, dim3(kNTrainFrags), dim3(64), 0, st, params, (bf16x8*)frags);
    return hipGetLastError();
}

hipError_t launch_train_batch(const TrainBatch& t, hipStream_t st) {
    const TrainArgs f{t.perm, (const bf16x8*)t.x, t.label, t.v, t.n, t.pos_w, t.vel_w, (const bf16x8*)t.frags, t.params,
                      (bf16x8*)t.h[0], (bf16x8*)t.h[1], (bf16x8*)t.h[2], (bf16x8*)t.dz[0], (bf16x8*)t.dz[1],
                      (bf16x8*)t.dz[2], (bf16x8*)t.dy, t.bias_part};
    const int blocks = std::min(t.max_blocks, cdiv(t.n, 32));
    hipLaunchKernelGGL(k_train_tile, dim3(blocks), dim3(256), 0, st, f);
    const int chunk = cdiv(cdiv(t.n, train_chunks(t.n)), kDwStep) * kDwStep, chunks = cdiv(t.n, chunk);
    const DwArgs d{t.perm, f.x, f.h1, f.h2, f.h3, f.dz1, f.dz2, f.dz3, f.dy, t.n, chunk, t.part};
    hipLaunchKernelGGL(k_train_dw, dim3(chunks, 4), dim3(256), 0, st, d);
    const StepArgs a{t.part, chunks, t.bias_part, blocks, t.w, t.m, t.v2, t.lr, t.b1, t.b2, t.eps, t.bc1, t.bc2,
                     (__bf16*)t.frags, t.grad, t.first, t.loss};
    static_assert(kDwFloats % 256 == 0, "one weight per thread");
    hipLaunchKernelGGL(k_train_step, dim3(kDwFloats / 256 + cdiv(kNBiasParams + 1, 16)), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_fill_f32(float* p, float v, long n, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill_f32, dim3(std::min(cdiv(n, 256), 4096)), dim3(256), 0, st, p, v, n);
    return hipGetLastError();
}

hipError_t launch_copy_f32(float* to, const float* from, long n, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_copy_f32, dim3(std::min(cdiv(n, 256), 4096)), dim3(256), 0, st, to, from, n);
    return hipGetLastError();
}

hipError_t launch_pack(const float* P, void* frags, float* bias, hipStream_t st) {
    hipLaunchKernelGGL(k_pack, dim3(kNFrags), dim3(64), 0, st, P, (bf16x8*)frags, bias);
    return hipGetLastError();
}

}  // namespace mlp
}  // namespace ecm
