// mlp_api.cpp -- host runtime behind include/ecm_mlp.h: parameters,
// dataset, the training loop (forward, backward and Adam on the GPU with
// the kernels of mlp_kernels.hip) and host-data entry points.
#include "mlp_host.h"
#include "stage.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <random>
#include <vector>

using namespace ecm;
using namespace ecm::mlp;

static inline __attribute__((always_inline)) uint16_t f32_to_bf16_rne(float f) {
    uint32_t u;
    std::memcpy(&u, &f, 4);
    const uint32_t r = (u + (((u >> 16) & 1u) + 0x7fffu)) >> 16;
    return (uint16_t)((u & 0x7fffffffu) > 0x7f800000u ? 0x7fc0u : r);          // NaN: quiet
}
// A row of them; with AVX2 where the CPU has it (8,192 samples: 200 us for the
// 4-wide baseline).
static void round_rows_base(const float* in, uint16_t* out, size_t n) {
    for (size_t i = 0; i < n; ++i) out[i] = f32_to_bf16_rne(in[i]);
}
#if !defined(__HIP_DEVICE_COMPILE__) && defined(__x86_64__)
__attribute__((target("avx2"))) static void round_rows_avx2(const float* in, uint16_t* out, size_t n) {
    for (size_t i = 0; i < n; ++i) out[i] = f32_to_bf16_rne(in[i]);
}
static void round_rows(const float* in, uint16_t* out, size_t n) {
    static const bool avx2 = __builtin_cpu_supports("avx2");
    (avx2 ? round_rows_avx2 : round_rows_base)(in, out, n);
}
#else
static void round_rows(const float* in, uint16_t* out, size_t n) { round_rows_base(in, out, n); }
#endif
static float bf16_to_f32(uint16_t h) {
    uint32_t u = (uint32_t)h << 16;
    float f;
    std::memcpy(&f, &u, 4);
    return f;
}

extern "C" int ecm_mlp_n_params(void) { return kNParams; }

extern "C" int ecm_mlp_create(uint64_t seed, ecm_mlp** out) {
    if (!out) return fail(ECM_E_ARG, "null argument");
    *out = nullptr;
    if (!ecm_device_available()) return fail(ECM_E_NOGPU, "no gfx950 device available");
    ecm_mlp* m = new ecm_mlp();
    (void)hipGetDevice(&m->dev);
    hipDeviceProp_t pr;
    if (hipGetDeviceProperties(&pr, m->dev) == hipSuccess && pr.multiProcessorCount > 0) m->n_cu = pr.multiProcessorCount;
    int rc = 0;
    if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess) rc = fail(ECM_E_HIP, "stream create failed");
    if (!rc) rc = m->params.alloc(kNParams);
    if (!rc) rc = m->grads.alloc(kNParams + 1);
    if (!rc) rc = m->adam_m.alloc(kNParams);
    if (!rc) rc = m->adam_v.alloc(kNParams);
    if (!rc) rc = m->tfrags.alloc((size_t)kNTrainFrags * 64);
    if (!rc) rc = m->frags.alloc((size_t)kNFrags * 64);
    if (!rc) rc = m->pbias.alloc(kNBias);
    if (!rc) rc = m->ds_count.alloc(1);
    if (rc) { ecm_mlp_destroy(m); return rc; }
    // seeded uniform(+-1/sqrt(fan_in)) init, the padding inputs of W1 zero
    std::vector<float> p(kNParams, 0.0f);
    std::mt19937_64 rng(seed);
    auto fill = [&](int off, int rows, int cols, int fan_in, int used_cols) {
        std::uniform_real_distribution<float> U(-1.0f / std::sqrt((float)fan_in), 1.0f / std::sqrt((float)fan_in));
        for (int r = 0; r < rows; ++r)
            for (int c = 0; c < cols; ++c) p[off + r * cols + c] = c < used_cols ? U(rng) : 0.0f;
    };
    fill(kOffW1, kHid, kInPad, kIn, kIn);
    fill(kOffB1, 1, kHid, kIn, kHid);
    fill(kOffW2, kHid, kHid, kHid, kHid);
    fill(kOffB2, 1, kHid, kHid, kHid);
    fill(kOffW3, kHid, kHid, kHid, kHid);
    fill(kOffB3, 1, kHid, kHid, kHid);
    fill(kOffW4, kOut, kHid, kHid, kHid);
    fill(kOffB4, 1, kOut, kHid, kOut);
    rc = ecm_mlp_set_params(m, p.data(), kNParams);
    if (rc) { ecm_mlp_destroy(m); return rc; }
    *out = m;
    return 0;
}

// A simulator step returns before its kernels finish, and a learned step
// reads the packed weights (frags, pbias) on the simulator's stream.  The
// calls that free or rewrite them therefore wait for the whole device.
extern "C" int ecm_mlp_destroy(ecm_mlp* m) {
    if (!m) return 0;
    (void)hipSetDevice(m->dev);
    (void)hipDeviceSynchronize();
    for (auto* b : {&m->params, &m->grads, &m->adam_m, &m->adam_v, &m->pbias, &m->y, &m->part, &m->bias_part})
        b->release();
    for (auto* b : {&m->frags, &m->tfrags, &m->ds_x, &m->xb, &m->h1, &m->h2, &m->h3, &m->dz1, &m->dz2, &m->dz3, &m->dy})
        b->release();
    m->ds_label.release(); m->ds_count.release(); m->lb.release();
    m->ds_v.release(); m->vb.release(); m->perm.release();
    if (m->stage) (void)hipHostFree(m->stage);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
    return 0;
}

extern "C" int ecm_mlp_get_params(ecm_mlp* m, float* out, int n) {
    if (!m || !out || n != kNParams) return fail(ECM_E_ARG, "expected %d parameters", kNParams);
    (void)hipSetDevice(m->dev);
    HIPCHK(hipMemcpyAsync(out, m->params.p, kNParams * sizeof(float), hipMemcpyDeviceToHost, m->stream));
    HIPCHK(hipStreamSynchronize(m->stream));
    return 0;
}

extern "C" int ecm_mlp_set_params(ecm_mlp* m, const float* in, int n) {
    if (!m || !in || n != kNParams) return fail(ECM_E_ARG, "expected %d parameters", kNParams);
    for (int i = 0; i < n; ++i)
        if (!std::isfinite(in[i])) return fail(ECM_E_ARG, "parameter %d is not finite", i);
    (void)hipSetDevice(m->dev);
    HIPCHK(hipDeviceSynchronize());          // a simulator step may still read the packed weights
    HIPCHK(hipMemcpyAsync(m->params.p, in, kNParams * sizeof(float), hipMemcpyHostToDevice, m->stream));
    HIPCHK(launch_fill_f32(m->adam_m.p, 0.0f, kNParams, m->stream));
    HIPCHK(launch_fill_f32(m->adam_v.p, 0.0f, kNParams, m->stream));
    m->adam_t = 0;
    m->tpacked = false;
    int rc = ecm_mlp_pack(m);
    if (rc) return rc;
    HIPCHK(hipStreamSynchronize(m->stream));
    return 0;
}

int ecm_mlp_pack(ecm_mlp* m) {
    HIPCHK(launch_pack(m->params.p, m->frags.p, m->pbias.p, m->stream));
    return 0;
}

// ----------------------------------------------------------------- dataset
extern "C" int ecm_mlp_dataset_reserve(ecm_mlp* m, int64_t capacity) {
    if (!m || capacity < 1 || capacity > (int64_t)0x7fffffff) return fail(ECM_E_ARG, "bad capacity");
    (void)hipSetDevice(m->dev);
    int64_t n = 0;
    int rc = ecm_mlp_dataset_size(m, &n);
    if (rc) return rc;
    if (capacity <= m->ds_cap) return 0;
    ecm::DBuf<bf16x8_t> x;
    ecm::DBuf<uint32_t> l;
    ecm::DBuf<float2> v;
    rc = x.alloc((size_t)capacity * 8);
    if (!rc) rc = l.alloc((size_t)capacity);
    if (!rc) rc = v.alloc((size_t)capacity);
    if (rc) { x.release(); l.release(); v.release(); return rc; }
    if (n > 0) {
        HIPCHK(hipMemcpyAsync(x.p, m->ds_x.p, (size_t)n * 8 * sizeof(bf16x8_t), hipMemcpyDeviceToDevice, m->stream));
        HIPCHK(hipMemcpyAsync(l.p, m->ds_label.p, (size_t)n * sizeof(uint32_t), hipMemcpyDeviceToDevice, m->stream));
        HIPCHK(hipMemcpyAsync(v.p, m->ds_v.p, (size_t)n * sizeof(float2), hipMemcpyDeviceToDevice, m->stream));
    }
    HIPCHK(hipStreamSynchronize(m->stream));
    m->ds_x.release(); m->ds_label.release(); m->ds_v.release();
    m->ds_x = x; m->ds_label = l; m->ds_v = v;
    x.p = nullptr; l.p = nullptr; v.p = nullptr;
    m->ds_cap = capacity;
    if (n == 0) return ecm_mlp_dataset_clear(m);
    return 0;
}

extern "C" int ecm_mlp_dataset_size(ecm_mlp* m, int64_t* n) {
    if (!m || !n) return fail(ECM_E_ARG, "null argument");
    (void)hipSetDevice(m->dev);
    uint32_t c = 0;
    HIPCHK(hipMemcpyAsync(&c, m->ds_count.p, sizeof(uint32_t), hipMemcpyDeviceToHost, m->stream));
    HIPCHK(hipStreamSynchronize(m->stream));
    *n = std::min<int64_t>(c, m->ds_cap);
    return 0;
}

extern "C" int ecm_mlp_dataset_clear(ecm_mlp* m) {
    if (!m) return fail(ECM_E_ARG, "null argument");
    (void)hipSetDevice(m->dev);
    const uint32_t z = 0;
    HIPCHK(hipMemcpyAsync(m->ds_count.p, &z, sizeof(uint32_t), hipMemcpyHostToDevice, m->stream));
    HIPCHK(hipStreamSynchronize(m->stream));
    return 0;
}

extern "C" int ecm_mlp_dataset_read(ecm_mlp* m, int64_t first, int n, float* x, uint32_t* label, float* v) {
    if (!m || n < 0 || first < 0) return fail(ECM_E_ARG, "bad arguments");
    int64_t have = 0;
    int rc = ecm_mlp_dataset_size(m, &have);
    if (rc) return rc;
    if (first + n > have) return fail(ECM_E_ARG, "samples [%lld, %lld) beyond the %lld logged", (long long)first,
                                      (long long)(first + n), (long long)have);
    if (n == 0) return 0;
    if (x) {
        std::vector<uint16_t> h((size_t)n * 64);
        HIPCHK(hipMemcpyAsync(h.data(), m->ds_x.p + first * 8, (size_t)n * 128, hipMemcpyDeviceToHost, m->stream));
        HIPCHK(hipStreamSynchronize(m->stream));
        for (size_t i = 0; i < h.size(); ++i) x[i] = bf16_to_f32(h[i]);
    }
    if (label) HIPCHK(hipMemcpyAsync(label, m->ds_label.p + first, (size_t)n * 4, hipMemcpyDeviceToHost, m->stream));
    if (v) HIPCHK(hipMemcpyAsync(v, m->ds_v.p + first, (size_t)n * 8, hipMemcpyDeviceToHost, m->stream));
    HIPCHK(hipStreamSynchronize(m->stream));
    return 0;
}

// ---------------------------------------------------------------- training
static int ensure_in(ecm_mlp* m, int B) {
    if (m->in_batch >= B) return 0;
    int rc = m->xb.alloc((size_t)B * 8);
    if (!rc) rc = m->lb.alloc(B);
    if (!rc) rc = m->vb.alloc(B);
    if (!rc) rc = m->y.alloc((size_t)B * kOut);
    m->in_batch = rc ? 0 : B;
    return rc;
}

static int ensure_ws(ecm_mlp* m, int B) {
    if (m->ws_batch >= B) return 0;
    m->ws_batch = 0;
    int rc = m->dy.alloc((size_t)B * 2);
    for (auto* b : {&m->h1, &m->h2, &m->h3, &m->dz1, &m->dz2, &m->dz3})
        if (!rc) rc = b->alloc((size_t)B * 16);
    if (!rc) rc = m->part.alloc((size_t)train_chunks(B) * kDwFloats);
    if (!rc) rc = m->bias_part.alloc((size_t)m->n_cu * (kNBiasParams + 1));
    if (rc) return rc;
    m->ws_batch = B;
    return 0;
}

// The training fragments of the current parameters: packed at the first use
// after the parameters were set, kept current by the Adam steps.
static int pack_train(ecm_mlp* m) {
    if (m->tpacked) return 0;
    HIPCHK(launch_train_pack(m->params.p, m->tfrags.p, m->stream));
    m->tpacked = true;
    return 0;
}

// The workspace and loss settings of a batch of B rows; the rows, the Adam
// constants and where the gradient goes are the caller's.
static TrainBatch train_batch(ecm_mlp* m, int B, float pos_w, float vel_w) {
    TrainBatch t{};
    t.n = B;
    t.pos_w = pos_w;
    t.vel_w = vel_w;
    t.frags = m->tfrags.p;
    t.params = m->params.p;
    t.h[0] = m->h1.p; t.h[1] = m->h2.p; t.h[2] = m->h3.p;
    t.dz[0] = m->dz1.p; t.dz[1] = m->dz2.p; t.dz[2] = m->dz3.p;
    t.dy = m->dy.p;
    t.bias_part = m->bias_part.p;
    t.max_blocks = m->n_cu;
    t.part = m->part.p;
    t.w = m->params.p;
    t.m = m->adam_m.p;
    t.v2 = m->adam_v.p;
    t.loss = m->grads.p + kNParams;
    return t;
}

// Host batches go through page-locked memory piece by piece (stage.h); results
// that fit into it come back through it, since the runtime's first touch
// of each result in pageable memory waits again.
constexpr size_t kStagePiece = 256 << 10, kStagePieces = 16;

// What a host call of n rows is staged through: the handle's page-locked
// pieces or, in a first call of few rows, ordinary memory with a piece for each
// of the three arrays.
struct Stage {
    unsigned char* mem = nullptr;
    size_t piece = kStagePiece, pieces = kStagePieces;
    std::unique_ptr<unsigned char[]> own;
    int open(ecm_mlp* m, size_t n) {
        const bool first = !m->host_called;
        m->host_called = true;
        if (!m->stage && !stage_page_locked(first, n)) {
            own.reset(new (std::nothrow) unsigned char[kFirstCallRows * 128 * 3]);
            if (own) {
                mem = own.get();
                piece = kFirstCallRows * 128;
                pieces = 3;
                return 0;
            }
        }
        if (!m->stage && hipHostMalloc((void**)&m->stage, piece * pieces, hipHostMallocDefault) != hipSuccess) {
            m->stage = nullptr;
            return fail(ECM_E_HIP, "hipHostMalloc of %zu bytes failed", piece * pieces);
        }
        mem = m->stage;
        return 0;
    }
};

struct StageQueue {
    hipStream_t st;
    int copy(void* dst, const void* src, size_t bytes) {
        HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st));
        return 0;
    }
    int wait() {
        HIPCHK(hipStreamSynchronize(st));
        return 0;
    }
};
using BatchStager = Stager<StageQueue>;

static int stage_host_batch(ecm_mlp* m, BatchStager& st, const float* x, const uint32_t* label, const float* v, int n) {
    int rc = st.put(m->xb.p, (size_t)n * 128, [&](void* to, size_t at, size_t len) {
        round_rows(x + at / 2, (uint16_t*)to, len / 2);
    });
    if (!rc && label) rc = st.put(m->lb.p, label, (size_t)n * 4);
    if (!rc && v) rc = st.put(m->vb.p, v, (size_t)n * 8);
    return rc;
}

// The result of a call: `bytes` of device memory, copied into the staging
// memory once the stream is there, or straight to the caller's when larger.
static int fetch(ecm_mlp* m, const Stage& stage, BatchStager& st, const void* dev, size_t bytes, void* out) {
    const bool staged = bytes <= stage.piece * stage.pieces;
    HIPCHK(hipMemcpyAsync(staged ? (void*)stage.mem : out, dev, bytes, hipMemcpyDeviceToHost, m->stream));
    HIPCHK(hipStreamSynchronize(m->stream));
    st.waited();
    if (staged) std::memcpy(out, stage.mem, bytes);
    return 0;
}

extern "C" int ecm_mlp_loss_grad(ecm_mlp* m, const float* x, const uint32_t* label, const float* v, int n,
                                 float pos_weight, float vel_weight, float* loss, float* grad) {
    if (!m || !x || !label || !v || n < 1 || !loss || !grad) return fail(ECM_E_ARG, "bad arguments");
    (void)hipSetDevice(m->dev);
    int rc = ensure_ws(m, n);
    if (!rc) rc = ensure_in(m, n);
    Stage stage;
    if (!rc) rc = stage.open(m, n);
    if (rc) return rc;
    StageQueue q{m->stream};
    BatchStager st(q, stage.mem, stage.piece, stage.pieces);
    if ((rc = stage_host_batch(m, st, x, label, v, n)) != 0) return rc;
    if ((rc = pack_train(m)) != 0) return rc;
    TrainBatch t = train_batch(m, n, pos_weight, vel_weight);
    t.first = true;
    t.x = m->xb.p;
    t.label = m->lb.p;
    t.v = m->vb.p;
    t.grad = m->grads.p;
    HIPCHK(launch_train_batch(t, m->stream));
    // the loss stands behind the gradient
    static_assert((kNParams + 1) * sizeof(float) <= 3 * kFirstCallRows * 128, "one fetch");
    HIPCHK(hipMemcpyAsync(stage.mem, m->grads.p, (kNParams + 1) * sizeof(float), hipMemcpyDeviceToHost, m->stream));
    HIPCHK(hipStreamSynchronize(m->stream));
    st.waited();
    std::memcpy(grad, stage.mem, kNParams * sizeof(float));
    std::memcpy(loss, stage.mem + kNParams * sizeof(float), sizeof(float));
    return 0;
}

extern "C" int ecm_mlp_forward(ecm_mlp* m, const float* x, int n, float* y) {
    if (!m || !x || !y || n < 1) return fail(ECM_E_ARG, "bad arguments");
    (void)hipSetDevice(m->dev);
    int rc = ensure_in(m, n);
    Stage stage;
    if (!rc) rc = stage.open(m, n);
    if (rc) return rc;
    StageQueue q{m->stream};
    BatchStager st(q, stage.mem, stage.piece, stage.pieces);
    if ((rc = stage_host_batch(m, st, x, nullptr, nullptr, n)) != 0) return rc;
    HIPCHK(launch_mlp_infer(m->xb.p, 0, nullptr, n, m->frags.p, m->pbias.p, 0.0f, m->lb.p, nullptr, m->y.p, m->n_cu,
                            m->stream));
    return fetch(m, stage, st, m->y.p, (size_t)n * kOut * sizeof(float), y);
}

// ------------------------------------------- forward without allocation
// Scratch of ecm_mlp_forward_noalloc: the proposal masks ([n]) and the output
// rows ([n][16] FP32, for a y that overlaps x) of up to
// ECM_MLP_NOALLOC_MAX_SAMPLES samples.  Every GPU holds its own copy until
// the process ends.  Nothing in it has to start at zero: the network writes
// every mask and every row.
constexpr size_t kNoAllocMaskBytes = (size_t)ECM_MLP_NOALLOC_MAX_SAMPLES * 4;
constexpr size_t kNoAllocBytes = kNoAllocMaskBytes + (size_t)ECM_MLP_NOALLOC_MAX_SAMPLES * kOut * 4;
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

// Device address of `scratch` on device `dev`, looked up once per device
// with that device current (each GPU holds the array at its own address).
static int scratch_address(int dev, unsigned char** out) {
    static std::mutex mu;
    static std::vector<unsigned char*> addr;
    std::lock_guard<std::mutex> lock(mu);
    if (dev < 0) return fail(ECM_E_ARG, "bad device %d", dev);
    if ((size_t)dev >= addr.size()) addr.resize((size_t)dev + 1, nullptr);
    if (!addr[dev]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(ECM_E_HIP, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
        addr[dev] = (unsigned char*)p;
    }
    *out = addr[dev];
    return 0;
}

extern "C" int ecm_mlp_forward_noalloc(ecm_mlp* m, const float* x, int n, float* y) {
    if (!m || !x || !y || n < 1) return fail(ECM_E_ARG, "bad arguments");
    if (n > ECM_MLP_NOALLOC_MAX_SAMPLES)
        return fail(ECM_E_ARG, "%d samples exceed the %d of the static scratch", n, ECM_MLP_NOALLOC_MAX_SAMPLES);
    HIPCHK(hipSetDevice(m->dev));
    unsigned char* base = nullptr;
    int rc = scratch_address(m->dev, &base);
    if (rc) return rc;
    // the network reads the FP32 rows itself, rounding as the host staging of
    // ecm_mlp_forward does; output rows over its input rows would reach tiles
    // that are yet to be read, and wait in the scratch
    const uintptr_t x0 = (uintptr_t)x, y0 = (uintptr_t)y;
    const size_t in_bytes = (size_t)n * kInPad * 4, out_bytes = (size_t)n * kOut * 4;
    const bool overlap = x0 < y0 + out_bytes && y0 < x0 + in_bytes;
    float* out = overlap ? reinterpret_cast<float*>(base + kNoAllocMaskBytes) : y;
    HIPCHK(launch_mlp_infer(x, 2, nullptr, n, m->frags.p, m->pbias.p, 0.0f, reinterpret_cast<uint32_t*>(base), nullptr,
                            out, m->n_cu, m->stream));
    if (overlap) HIPCHK(launch_copy_f32(y, out, (long)n * kOut, m->stream));
    HIPCHK(hipStreamSynchronize(m->stream));
    return 0;
}

extern "C" int ecm_mlp_train(ecm_mlp* m, int epochs, int batch, float lr, float pos_weight, float vel_weight,
                             uint64_t seed, float* losses) {
    if (!m || epochs < 0 || batch < 64 || !(lr > 0.0f)) return fail(ECM_E_ARG, "bad training arguments");
    (void)hipSetDevice(m->dev);
    HIPCHK(hipDeviceSynchronize());          // a simulator step may still read the packed weights
    int64_t n = 0;
    int rc = ecm_mlp_dataset_size(m, &n);
    if (rc) return rc;
    if (n < batch) return fail(ECM_E_STATE, "dataset holds %lld samples, fewer than one batch of %d", (long long)n, batch);
    rc = ensure_ws(m, batch);
    if (!rc && m->perm.n < (size_t)n) rc = m->perm.alloc((size_t)n);
    if (rc) return rc;
    // Fisher-Yates with the seeded generator (reproducible across hosts); the
    // next epoch's order is drawn while the GPU works on this one's
    std::vector<int32_t> order[2];      // (the capacity fits an int)
    std::mt19937_64 rng(seed);
    auto shuffle = [&](std::vector<int32_t>& p) {
        for (int64_t i = n - 1; i > 0; --i) {
            const int64_t j = (int64_t)(rng() % (uint64_t)(i + 1));
            std::swap(p[i], p[j]);
        }
    };
    order[0].resize((size_t)n);
    for (int64_t i = 0; i < n; ++i) order[0][i] = (int32_t)i;
    if (epochs > 0) shuffle(order[0]);
    const int64_t nb = n / batch;
    TrainBatch t = train_batch(m, batch, pos_weight, vel_weight);
    t.x = m->ds_x.p;
    t.label = m->ds_label.p;
    t.v = m->ds_v.p;
    t.lr = lr;
    t.b1 = 0.9f;
    t.b2 = 0.999f;
    t.eps = 1e-8f;
    if ((rc = pack_train(m)) != 0) return rc;
    for (int e = 0; e < epochs; ++e) {
        const std::vector<int32_t>& perm = order[e & 1];
        HIPCHK(hipMemcpyAsync(m->perm.p, perm.data(), (size_t)n * sizeof(int32_t), hipMemcpyHostToDevice, m->stream));
        for (int64_t b = 0; b < nb; ++b) {
            ++m->adam_t;
            t.first = b == 0;
            t.perm = m->perm.p + b * batch;
            t.bc1 = 1.0f - std::pow(t.b1, (float)m->adam_t);
            t.bc2 = 1.0f - std::pow(t.b2, (float)m->adam_t);
            HIPCHK(launch_train_batch(t, m->stream));
        }
        if (e + 1 < epochs) {
            order[(e + 1) & 1] = perm;
            shuffle(order[(e + 1) & 1]);
        }
        float L = 0.0f;
        HIPCHK(hipMemcpyAsync(&L, t.loss, sizeof(float), hipMemcpyDeviceToHost, m->stream));
        HIPCHK(hipStreamSynchronize(m->stream));      // also keeps `perm` alive for the upload
        if (losses) losses[e] = L / (float)nb;
    }
    rc = ecm_mlp_pack(m);
    if (rc) return rc;
    HIPCHK(hipStreamSynchronize(m->stream));
    return 0;
}
