// psx_passes.hip - pass pixels from the film's sums, and the sampler's table
// (gfx950).
//
// The pass kernels do what a host loop over the downloaded film did, in the
// same order of float operations: three sums of 16 bytes a pixel and a count
// crossed the bus to give passes of 4 to 16 bytes, and the loop took longer
// than the frame of a small scene.  They are bound by the film's bytes: with
// the count check 68 read and 44 written a pixel for Combined, Normal, Albedo
// and Sample Count, 0.05 ms at 1920x1080.
#include "psx_device.h"
#include "psx_sobol.h"

#pragma clang fp contract(off)

namespace psx {
namespace {

constexpr uint32_t kPassBlock = 256;

// Cycles' safe_divide_even_color (src/luisa/path_tracer_common.cpp:516-548):
// channels with a zero denominator take the other channels' quotients.
__device__ __forceinline__ float4 divide_even_color(float4 n, float4 d) {
    float x = d.x != 0.0f ? n.x / d.x : 0.0f;
    float y = d.y != 0.0f ? n.y / d.y : 0.0f;
    float z = d.z != 0.0f ? n.z / d.z : 0.0f;
    if (d.x == 0.0f) {
        if (d.y == 0.0f) {
            x = z;
            y = z;
        } else if (d.z == 0.0f) {
            x = y;
            z = y;
        } else {
            x = 0.5f * (y + z);
        }
    } else if (d.y == 0.0f) {
        if (d.z == 0.0f) {
            y = x;
            z = x;
        } else {
            y = 0.5f * (x + z);
        }
    } else if (d.z == 0.0f) {
        z = 0.5f * (x + y);
    }
    return make_float4(x, y, z, 1.0f);
}

__device__ __forceinline__ float4 scaled(float4 v, float s) {
    return make_float4(v.x * s, v.y * s, v.z * s, v.w * s);
}
__device__ __forceinline__ float4 over(float4 v, float d) {
    return make_float4(v.x / d, v.y / d, v.z / d, v.w / d);
}

template <uint32_t CHANNELS>
__global__ __launch_bounds__(kPassBlock) void pass_kernel(FilmView film, uint64_t pixels, PassRule rule, uint32_t slot,
                                                          float exposure, float *out) {
    const uint64_t i = static_cast<uint64_t>(blockIdx.x) * kPassBlock + threadIdx.x;
    if (i >= pixels) return;
    const uint32_t count = film.sample_count[i];
    const float den = static_cast<float>(count > 1u ? count : 1u);
    const float4 *light = film.light ? reinterpret_cast<const float4 *>(film.light) + i * kLightPasses : nullptr;
    const float4 *albedo = reinterpret_cast<const float4 *>(film.albedo) + i;
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    switch (rule) {
    case PassRule::kCombined: {
        const float4 c = reinterpret_cast<const float4 *>(film.combined)[i];
        const float scale = exposure / den;
        float alpha = 1.0f - c.w / den;
        alpha = alpha < 0.0f ? 0.0f : alpha;
        alpha = 1.0f < alpha ? 1.0f : alpha;
        v = make_float4(c.x * scale, c.y * scale, c.z * scale, alpha);
        break;
    }
    case PassRule::kNormal:
        v = over(reinterpret_cast<const float4 *>(film.normal)[i], den);
        break;
    case PassRule::kAlbedo:
        v = over(*albedo, den);
        break;
    case PassRule::kSampleCount: {
        const float c = static_cast<float>(count);
        v = make_float4(c, c, c, c);
        break;
    }
    case PassRule::kLight:
        v = scaled(light[slot], exposure / den);
        break;
    case PassRule::kLightColor:
        v = over(light[slot], den);
        break;
    case PassRule::kOverAlbedo:
    case PassRule::kOverGlossy:
    case PassRule::kOverTransmission: {
        const float4 color = rule == PassRule::kOverAlbedo   ? *albedo
                             : rule == PassRule::kOverGlossy ? light[kLpGlossyColor]
                                                             : light[kLpTransmissionColor];
        v = divide_even_color(light[slot], color);
        v = make_float4(v.x * exposure, v.y * exposure, v.z * exposure, 1.0f);
        break;
    }
    case PassRule::kZero:
        break;
    }
    float *o = out + i * CHANNELS;
    o[0] = v.x;
    if (CHANNELS > 1u) o[1] = v.y;
    if (CHANNELS > 2u) o[2] = v.z;
    if (CHANNELS > 3u) o[3] = v.w;
}

// sets `wrong`, a word of host memory, when a pixel's count differs from `expected`
__global__ __launch_bounds__(kPassBlock) void count_check_kernel(const uint32_t *counts, uint64_t pixels,
                                                                 uint32_t expected, uint32_t *wrong) {
    const uint64_t i = static_cast<uint64_t>(blockIdx.x) * kPassBlock + threadIdx.x;
    const bool off = i < pixels && counts[i] != expected;
    if (__ballot(off) != 0ull && (threadIdx.x & 63u) == 0u) *wrong = 1u;
}

// One block per pattern.  Level n fills elements n ... 2n - 1 from the elements
// before them, so a level is parallel and the levels follow each other.
__global__ __launch_bounds__(256) void sobol_kernel(float4 *table, uint32_t size) {
    const uint32_t pattern = blockIdx.x;
    float *p = reinterpret_cast<float *>(table + static_cast<size_t>(pattern) * size);
    const uint32_t seed = sobol_pattern_seed(pattern);
    if (threadIdx.x < 4u) p[threadIdx.x] = hash_hp_float(seed + threadIdx.x);
    __syncthreads();
    uint32_t level = 0u;
    for (uint32_t n = 1u; n < size; ++level, n *= 2u) {
        const float strata = static_cast<float>(n * 2u);
        for (uint32_t j = threadIdx.x; j < 4u * n && (j >> 2) + n < size; j += 256u) {
            const uint32_t i = j >> 2, c = j & 3u;
            const uint32_t occupied = static_cast<uint32_t>(p[4u * (i ^ kSobolXors[c][level]) + c] * strata);
            p[4u * (n + i) + c] =
                (static_cast<float>(occupied ^ 1u) + hash_hp_float(seed + 4u * (n + i) + c)) / strata;
        }
        __syncthreads();
    }
}

}  // namespace

// `size` float4 per pattern, a power of two
hipError_t launch_sobol_table(float4 *table, uint32_t size, hipStream_t stream) {
    hipLaunchKernelGGL(sobol_kernel, dim3(kSobolPatterns), dim3(256), 0, stream, table, size);
    return hipGetLastError();
}

hipError_t launch_count_check(const uint32_t *counts, uint64_t pixels, uint32_t expected, uint32_t *wrong,
                              hipStream_t stream) {
    hipLaunchKernelGGL(count_check_kernel, dim3(static_cast<uint32_t>((pixels + kPassBlock - 1u) / kPassBlock)),
                       dim3(kPassBlock), 0, stream, counts, pixels, expected, wrong);
    return hipGetLastError();
}

// One pass of `channels` (1 to 4) floats a pixel into `out`.
hipError_t launch_pass(const FilmView &film, uint64_t pixels, PassRule rule, uint32_t slot, uint32_t channels,
                       float exposure, float *out, hipStream_t stream) {
    if (channels < 1u || channels > 4u) return hipErrorInvalidValue;
    using Fn = void (*)(FilmView, uint64_t, PassRule, uint32_t, float, float *);
    const Fn fns[4] = {pass_kernel<1>, pass_kernel<2>, pass_kernel<3>, pass_kernel<4>};
    hipLaunchKernelGGL(fns[channels - 1u], dim3(static_cast<uint32_t>((pixels + kPassBlock - 1u) / kPassBlock)),
                       dim3(kPassBlock), 0, stream, film, pixels, rule, slot, exposure, out);
    return hipGetLastError();
}

}  // namespace psx
