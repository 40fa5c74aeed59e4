// short_operations.hip - the short reciprocal, root and quotient of the light
// importance (psx_path.h) against the correctly rounded operations on the
// device: every float of the stated ranges, and two random numerators for each
// denominator.  What remains of them needs no device: given the reciprocal,
// the quotient is proved on the host (tests/host/path_header_driver.cpp).
#include <hip/hip_runtime.h>

#include <cstdio>

#include "psx_path.h"

namespace {

constexpr uint32_t kMantissas = 1u << 23;
constexpr uint32_t kBlock = 256u;

__device__ uint32_t mixed(uint32_t v) {
    v ^= v >> 16;
    v *= 0x7feb352du;
    v ^= v >> 15;
    v *= 0x846ca68bu;
    return v ^ (v >> 16);
}

// one thread per mantissa; wrong[0..2]: reciprocals, roots, quotients
__global__ __launch_bounds__(kBlock) void check(unsigned long long *wrong) {
    const uint32_t m = blockIdx.x * kBlock + threadIdx.x;
    if (m >= kMantissas) return;
    unsigned long long bad[3] = {0ull, 0ull, 0ull};
    for (int e = -100; e < 100; ++e) {
        const float x = __uint_as_float((static_cast<uint32_t>(e + 127) << 23) | m);
        const float y = psx::lt_reciprocal(x);
        bad[0] += y != 1.0f / x;
        if (e >= -60) bad[1] += psx::lt_root(x) != sqrtf(x);
        if (e >= -60 && e < 60)
            for (uint32_t i = 0; i < 2u; ++i) {
                const uint32_t r = mixed(m * 401u + static_cast<uint32_t>(e + 100) * 2u + i);
                const int ea = e - 20 + static_cast<int>((r >> 23) % 41u);
                const float a = __uint_as_float((static_cast<uint32_t>(ea + 127) << 23) | (r & (kMantissas - 1u)));
                bad[2] += psx::lt_quotient(a, x, y) != a / x;
            }
    }
    for (int i = 0; i < 3; ++i)
        if (bad[i] != 0ull) atomicAdd(wrong + i, bad[i]);
}

}  // namespace

int main() {
    unsigned long long *device = nullptr, wrong[3] = {0ull, 0ull, 0ull};
    if (hipMalloc(reinterpret_cast<void **>(&device), sizeof(wrong)) != hipSuccess) {
        std::printf("no device\n");
        return 2;
    }
    bool ok = hipMemcpy(device, wrong, sizeof(wrong), hipMemcpyHostToDevice) == hipSuccess;
    if (ok) {
        hipLaunchKernelGGL(check, dim3(kMantissas / kBlock), dim3(kBlock), 0, nullptr, device);
        ok = hipGetLastError() == hipSuccess && hipDeviceSynchronize() == hipSuccess &&
             hipMemcpy(wrong, device, sizeof(wrong), hipMemcpyDeviceToHost) == hipSuccess;
    }
    ok = hipFree(device) == hipSuccess && ok;
    std::printf("wrong: %llu reciprocals, %llu roots, %llu quotients\n", wrong[0], wrong[1], wrong[2]);
    if (!ok || wrong[0] + wrong[1] + wrong[2] != 0ull) return 1;
    std::printf("ok\n");
    return 0;
}
