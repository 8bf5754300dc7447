// arith_check.hip -- the device code's cheap roots, reciprocals, quotients and
// half-planes against sqrtf, `/`, atan_f and the branching half-plane, on the
// GPU.  Every check returns the operands that differ in out[0] and how many it
// compared in out[1].
#include "half_plane.h"

#include <cstring>

using namespace ecm;

namespace {

__device__ __forceinline__ bool same(float a, float b) { return __float_as_uint(a) == __float_as_uint(b); }

// Sums over the grid, one atomic per thread that has something.
__device__ __forceinline__ void add(unsigned long long* out, uint32_t bad, uint32_t n) {
    if (bad) atomicAdd(out, (unsigned long long)bad);
    if (n) atomicAdd(out + 1, (unsigned long long)n);
}

// All 2^23 mantissas of exponents lo .. hi - 1: thread t of the grid takes
// mantissa t at every exponent.  what 0: root_from; 1: recip_from of rcp; 2:
// recip_from of the rsq that the root came from (all-ones lengths excepted).
__global__ void k_unary(int what, int lo, int hi, unsigned long long* out) {
    const uint32_t m = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t bad = 0, n = 0;
    for (int e = lo; e < hi; ++e) {
        const float v = __uint_as_float((uint32_t)(e + 127) << 23 | m);
        if (what == 1) {
            bad += !same(recip_from(v, __builtin_amdgcn_rcpf(v)), 1.0f / v);
            ++n;
            continue;
        }
        const float y = __builtin_amdgcn_rsqf(v), l = root_from(v, y);
        if (what == 0) {
            bad += !same(l, sqrtf(v));
            ++n;
        } else if (!all_ones(l)) {
            bad += !same(recip_from(l, y), 1.0f / l);
            ++n;
        }
    }
    add(out, bad, n);
}

// atan_unit for the floats with bits [first, first + count), all in [0, 1].
__global__ void k_atan(uint32_t first, uint32_t count, unsigned long long* out) {
    uint32_t bad = 0, n = 0;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += gridDim.x * blockDim.x) {
        const float x = __uint_as_float(first + i);
        bad += !same(atan_unit(x), atan_f(x));
        ++n;
    }
    add(out, bad, n);
}

__device__ __forceinline__ uint32_t mix(uint32_t x) {
    x ^= x >> 16; x *= 0x7feb352du; x ^= x >> 15; x *= 0x846ca68bu; x ^= x >> 16;
    return x;
}

// quot over pairs: numerators of either sign, zero or with exponents -80 .. 59,
// lengths with exponents -60 .. 59; every fourth mantissa is one of the ends.
__global__ void k_quot(uint32_t seed, int rounds, unsigned long long* out) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t bad = 0, n = 0;
    for (int r = 0; r < rounds; ++r) {
        const uint32_t a = mix(seed + t * 2654435761u + r), b = mix(a ^ 0x9e3779b9u), c = mix(b ^ a);
        auto mant = [](uint32_t h) {
            const uint32_t ends[4] = {0u, 1u, 0x7fffffu, 0x7ffffeu};
            return (h & 3u) ? (h >> 9) : ends[(h >> 2) & 3u];
        };
        const float l = __uint_as_float((uint32_t)(127 - 60 + (int)(c % 120u)) << 23 | mant(a));
        float x = __uint_as_float((uint32_t)(127 - 80 + (int)((c >> 8) % 140u)) << 23 | mant(b));
        if ((c >> 20) % 61u == 0u) x = 0.0f;
        if (c >> 31) x = -x;
        const float y = recip_from(l, __builtin_amdgcn_rcpf(l));
        // a quotient below the normal numbers is not what the kernels form
        if (x != 0.0f && fabsf(x / l) < 0x1p-126f) continue;
        bad += !same(quot(x, l, y), x / l);
        ++n;
    }
    add(out, bad, n);
}

struct HalfPlane {
    float px, py, vx, vy, r;          // the agent
    float qx, qy, qr, qvx, qvy;       // the other
};
__global__ void k_half_plane(DevState s, const HalfPlane* in, int n, uint8_t* covered, unsigned long long* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const HalfPlane h = in[i];
    const float4 q = make_float4(h.qx, h.qy, h.qr, 0.0f);
    const float2 qv = make_float2(h.qvx, h.qvy);
    V2 p0, n0, p1, n1;
    agent_constraint(s, mk(h.px, h.py), mk(h.vx, h.vy), h.r, q, qv, p0, n0);
    const bool c = agent_constraint_common(s, mk(h.px, h.py), mk(h.vx, h.vy), h.r, q, qv, p1, n1);
    covered[i] = c ? 1 : 0;
    if (c) add(out, same(p0.x, p1.x) && same(p0.y, p1.y) && same(n0.x, n1.x) && same(n0.y, n1.y) ? 0u : 1u, 1u);
}

template <typename F>
int run(unsigned long long* out, F&& launch) {
    unsigned long long* d = nullptr;
    out[0] = out[1] = 0;
    if (hipMalloc((void**)&d, 16) != hipSuccess) return 1;
    int rc = hipMemcpy(d, out, 16, hipMemcpyHostToDevice) == hipSuccess ? 0 : 2;
    if (!rc) {
        launch(d);
        if (hipGetLastError() != hipSuccess || hipMemcpy(out, d, 16, hipMemcpyDeviceToHost) != hipSuccess) rc = 3;
    }
    (void)hipFree(d);
    return rc;
}

}  // namespace

extern "C" int check_unary(int what, int lo, int hi, unsigned long long* out) {
    if (what < 0 || what > 2 || lo < -126 || hi > 127 || lo >= hi) return 4;
    return run(out, [&](unsigned long long* d) { k_unary<<<(1 << 23) / 256, 256>>>(what, lo, hi, d); });
}

extern "C" int check_atan(unsigned long long* out) {
    const float one = 1.0f;
    uint32_t bits;
    std::memcpy(&bits, &one, 4);
    return run(out, [&](unsigned long long* d) { k_atan<<<4096, 256>>>(0u, bits + 1u, d); });
}

extern "C" int check_quot(uint32_t seed, int rounds, unsigned long long* out) {
    if (rounds < 1) return 4;
    return run(out, [&](unsigned long long* d) { k_quot<<<4096, 256>>>(seed, rounds, d); });
}

// T, dt as the handle's parameters; covered[n] receives which pairs the
// branch-free form took.
extern "C" int check_half_plane(float T, float inv_T, float dt, float inv_dt, const float* in, int n, uint8_t* covered,
                                unsigned long long* out) {
    static_assert(sizeof(HalfPlane) == 40, "ten floats");
    if (n < 1) return 4;
    DevState s;
    std::memset(&s, 0, sizeof(s));
    s.time_horizon = T; s.inv_time_horizon = inv_T; s.dt = dt; s.inv_dt = inv_dt;
    HalfPlane* d_in = nullptr;
    uint8_t* d_c = nullptr;
    int rc = 1;
    if (hipMalloc((void**)&d_in, (size_t)n * sizeof(HalfPlane)) == hipSuccess && hipMalloc((void**)&d_c, n) == hipSuccess &&
        hipMemcpy(d_in, in, (size_t)n * sizeof(HalfPlane), hipMemcpyHostToDevice) == hipSuccess) {
        rc = run(out, [&](unsigned long long* d) { k_half_plane<<<(n + 255) / 256, 256>>>(s, d_in, n, d_c, d); });
        if (!rc && hipMemcpy(covered, d_c, n, hipMemcpyDeviceToHost) != hipSuccess) rc = 3;
    }
    (void)hipFree(d_in);
    (void)hipFree(d_c);
    return rc;
}
