// psx_sobol.h - the tabulated Sobol sequence's constants and hash, shared by
// the host table (psx_host.cpp) and the device table (psx_passes.hip).
// (src/sampling/tabulated_sobol.cpp:93-199)
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace psx {

constexpr uint32_t kSobolPatterns = 256u;

constexpr uint32_t kSobolXors[4][32] = {
    {0u},
    {0x00000000u, 0x00000001u, 0x00000001u, 0x00000007u, 0x00000001u, 0x00000013u, 0x00000015u, 0x0000007fu,
     0x00000001u, 0x00000103u, 0x00000105u, 0x0000070fu, 0x00000111u, 0x00001333u, 0x00001555u, 0x00007fffu,
     0x00000001u, 0x00010003u, 0x00010005u, 0x0007000fu, 0x00010011u, 0x00130033u, 0x00150055u, 0x007f00ffu,
     0x00010101u, 0x01030303u, 0x01050505u, 0x070f0f0fu, 0x01111111u, 0x13333333u, 0x15555555u, 0x7fffffffu},
    {0x00000000u, 0x00000001u, 0x00000003u, 0x00000001u, 0x00000005u, 0x0000001fu, 0x0000002bu, 0x0000003du,
     0x00000011u, 0x00000133u, 0x00000377u, 0x00000199u, 0x00000445u, 0x00001ccfu, 0x00002ddbu, 0x0000366du,
     0x00000101u, 0x00010303u, 0x00030707u, 0x00010909u, 0x00051515u, 0x001f3f3fu, 0x002b6b6bu, 0x003dbdbdu,
     0x00101011u, 0x01303033u, 0x03707077u, 0x01909099u, 0x04515145u, 0x1cf3f3cfu, 0x2db6b6dbu, 0x36dbdb6du},
    {0x00000000u, 0x00000001u, 0x00000000u, 0x00000003u, 0x0000000du, 0x0000000cu, 0x00000005u, 0x0000004fu,
     0x00000014u, 0x000000e7u, 0x00000329u, 0x0000039cu, 0x00000011u, 0x00001033u, 0x00000044u, 0x000030bbu,
     0x0000d1cdu, 0x0000c2ecu, 0x00005415u, 0x0004fc3fu, 0x00015054u, 0x000e5c97u, 0x0032e5b9u, 0x0039725cu,
     0x00000101u, 0x01000303u, 0x00000404u, 0x03000b0bu, 0x0d001d1du, 0x0c002c2cu, 0x05004545u, 0x4f00cfcfu}};

__host__ __device__ inline uint32_t hash_hp(uint32_t v) {
    v ^= v >> 16u;
    v *= 0x21f0aaadu;
    v ^= v >> 15u;
    v *= 0xd35a2d97u;
    v ^= v >> 15u;
    return v ^ 0xe6fe3bebu;
}

__host__ __device__ inline float hash_hp_float(uint32_t v) {
    return static_cast<float>(hash_hp(v)) * (1.0f / 4294967808.0f);
}

// first hash input of a pattern: hash_hp_seeded_uint(pattern, 0x44605a73), the
// seed pre-mixed; element e takes inputs 4 e ... 4 e + 3 after it
__host__ __device__ inline uint32_t sobol_pattern_seed(uint32_t pattern) {
    uint32_t seed = 0x44605a73u;
    seed ^= seed << 19u;
    return hash_hp(pattern ^ seed);
}

}  // namespace psx
