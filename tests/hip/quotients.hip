// quotients.hip -- the kernels' short forms of quotients and roots against the
// division operator and sqrtf on the device: every float, and seeded points.
// Each function returns the number of values that differ (a negative HIP error
// code if a call failed); *first is the first of them, if any.
#include <hip/hip_runtime.h>

#include "device.h"

namespace {

using namespace edxr;

struct Result {
    unsigned long long bad, first;
};

__device__ bool same(float a, float b) { return __float_as_uint(a) == __float_as_uint(b) || (a != a && b != b); }

struct Reciprocal {
    __device__ bool operator()(uint64_t i) const {
        const float x = __uint_as_float((uint32_t)i);
        return same(reciprocal(x), 1.0f / x) && (!in_range<-124, 125>(fabsf(x)) || same(rcp_normal(x), 1.0f / x));
    }
};
struct ReciprocalSqrt {
    __device__ bool operator()(uint64_t i) const {
        const float x = __uint_as_float((uint32_t)i);
        return same(reciprocal_sqrt(x), 1.0f / sqrtf(x));
    }
};
// A clip-space point whose coordinates' and w's exponents go beyond the range of the
// short projection on both sides, exponents and mantissas uniform; 0 among them.
struct Projection {
    uint64_t seed;
    __device__ static uint64_t mix(uint64_t z) {
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    }
    __device__ static float value(uint64_t z, int lo, int hi, bool sign) {
        const uint32_t e = (uint32_t)(127 + lo) + (uint32_t)((z >> 32 & 0xFFFFu) * (uint32_t)(hi - lo) >> 16);
        return __uint_as_float((sign ? (uint32_t)(z >> 63) << 31 : 0u) | e << 23 | (uint32_t)(z & 0x7FFFFFu));
    }
    __device__ bool operator()(uint64_t i) const {
        uint64_t z[4];
        for (int k = 0; k < 4; k++) z[k] = mix((4 * (i + seed) + k) * 0x9E3779B97F4A7C15ull);
        float4 c = make_float4(value(z[0], -104, 64, true), value(z[1], -104, 64, true), value(z[2], -104, 64, true),
                               value(z[3], -64, 64, false));
        if ((z[3] >> 48 & 0xFFu) == 0) c.x = 0.0f;
        if (!project_is_normal(c)) return true;
        const float4 a = project_normal(c), b = project_any(c);
        return same(a.x, b.x) && same(a.y, b.y) && same(a.z, b.z) && same(a.w, b.w);
    }
};
// The resolve's quotient of a byte.
struct Byte {
    __device__ bool operator()(uint64_t i) const {
        return same(quotient_normal((float)i, 255.0f, 1.0f / 255.0f), (float)i / 255.0f);
    }
};

template <class F>
__global__ __launch_bounds__(256) void k_check(F f, uint64_t n, Result* out) {
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256)
        if (!f(i)) {
            atomicAdd(&out->bad, 1ull);
            atomicMin(&out->first, (unsigned long long)i);
        }
}

template <class F>
long long run(F f, uint64_t n, uint64_t* first) {
    Result r{0, ~0ull}, *d = nullptr;
    hipError_t e = hipMalloc((void**)&d, sizeof(r));
    if (e == hipSuccess) e = hipMemcpy(d, &r, sizeof(r), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_check<F>, dim3(4096), dim3(256), 0, 0, f, n, d);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(&r, d, sizeof(r), hipMemcpyDeviceToHost);
    if (d) (void)hipFree(d);
    *first = r.first;
    return e == hipSuccess ? (long long)r.bad : -(long long)e;
}

}  // namespace

extern "C" {
long long check_reciprocal(uint64_t* first) { return run(Reciprocal{}, 1ull << 32, first); }
long long check_reciprocal_sqrt(uint64_t* first) { return run(ReciprocalSqrt{}, 1ull << 32, first); }
long long check_projection(uint64_t seed, uint64_t n, uint64_t* first) { return run(Projection{seed}, n, first); }
long long check_byte(uint64_t* first) { return run(Byte{}, 256, first); }
}
