// path_header_driver.cpp - parts of the device header psx_path.h that need no
// device, compiled for the host: the short reciprocal, quotient and root, and
// the traversal stack's bookkeeping.
//
// Usage: path_header_driver <reciprocal|root|quotient|stack>; prints "ok".
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <thread>
#include <vector>

// ---- what hipRTC provides to the header ---------------------------------------
namespace __hip_internal {
using std::int16_t;
using std::int32_t;
using std::int64_t;
using std::int8_t;
using std::uint16_t;
using std::uint32_t;
using std::uint64_t;
using std::uint8_t;
}  // namespace __hip_internal
struct float2 { float x, y; };
struct alignas(16) float4 { float x, y, z, w; };
struct uint2 { uint32_t x, y; };
struct alignas(16) uint4 { uint32_t x, y, z, w; };
static inline float2 make_float2(float x, float y) { return float2{x, y}; }
static inline float4 make_float4(float x, float y, float z, float w) { return float4{x, y, z, w}; }
static inline uint2 make_uint2(uint32_t x, uint32_t y) { return uint2{x, y}; }
static inline uint4 make_uint4(uint32_t x, uint32_t y, uint32_t z, uint32_t w) { return uint4{x, y, z, w}; }
template <typename To, typename From>
static inline To same_bits(From v) {
    To r;
    std::memcpy(&r, &v, sizeof(r));
    return r;
}
#define __float_as_uint(v) same_bits<uint32_t>(static_cast<float>(v))
#define __float_as_int(v) same_bits<int>(static_cast<float>(v))
#define __uint_as_float(v) same_bits<float>(static_cast<uint32_t>(v))
#define __int_as_float(v) same_bits<float>(static_cast<int>(v))
#define __brev(v) __builtin_bitreverse32(v)
#define __popcll(v) __builtin_popcountll(v)
#define __builtin_amdgcn_ballot_w64(v) ((v) ? 1ull : 0ull)
static struct { uint32_t x; } threadIdx, blockDim, blockIdx;
static inline void __syncthreads() {}

// The hardware's approximations are within one unit in the last place: one of
// the two floats around the value.  `upper` says which.
static thread_local bool upper = false;
static inline float around(double v) {
    float n = static_cast<float>(v);
    if (upper && static_cast<double>(n) < v) n = std::nextafterf(n, INFINITY);
    if (!upper && static_cast<double>(n) > v) n = std::nextafterf(n, 0.0f);
    return n;
}
#define __builtin_amdgcn_rcpf(v) around(1.0 / static_cast<double>(v))
#define __builtin_amdgcn_rsqf(v) around(1.0 / std::sqrt(static_cast<double>(v)))

using std::isfinite;
using std::isinf;
using std::isnan;
using std::max;
using std::min;
#define __device__
#define __host__
#define __shared__ static
#define __forceinline__ inline
#define __attribute__(x)
#define __HIPCC_RTC__
#include "psx_path.h"
#undef __attribute__

namespace {

constexpr uint32_t kOne = 1u << 23;  // mantissas are kOne ... 2 kOne - 1
float scaled(uint32_t mantissa, int e) { return std::ldexp(static_cast<float>(mantissa), e - 23); }

// every mantissa, from either float around 1 / x: exact but for the largest
// mantissa from below
int reciprocal() {
    int wrong = 0;
    for (bool u : {false, true}) {
        upper = u;
        for (uint32_t m = kOne; m < 2u * kOne; ++m) {
            const float x = scaled(m, 0);
            if (psx::lt_reciprocal(x) != 1.0f / x && (u || m != 2u * kOne - 1u)) ++wrong;
        }
    }
    return wrong;
}

// every mantissa and both parities of the exponent: exact but for one value
// from above
int root() {
    int wrong = 0;
    for (bool u : {false, true}) {
        upper = u;
        for (int e : {0, 1})
            for (uint32_t m = kOne; m < 2u * kOne; ++m) {
                const float x = scaled(m, e);
                if (psx::lt_root(x) != std::sqrt(x) && !(u && x == 0x1.dd26e4p+1f)) ++wrong;
            }
    }
    upper = false;
    return wrong + (psx::lt_root(0.0f) != 0.0f);
}

// With y the rounded 1 / x, q = a y is within 1.5 units of a / x, the residual
// and y add 2^-24 of it each, so before its rounding the quotient is within
// 2^-21 units of a / x.  It can round wrongly only where a / x is that near
// the middle of two floats: |2^(k+1) A - (2M + 1) X| <= 16 for the mantissas
// A, X and M of a, x and a / x.  All of those pairs are tried.
void quotients(uint32_t begin, uint32_t step, long &tried, long &wrong) {
    for (uint32_t X = kOne + begin; X < 2u * kOne; X += step) {
        const int twos = __builtin_ctz(X);
        if (twos > 4) continue;
        const uint32_t odd = X >> twos;
        uint32_t inverse = odd;  // modulo 2^32
        for (int i = 0; i < 5; ++i) inverse *= 2u - odd * inverse;
        const float x = scaled(X, 0), y = 1.0f / x;
        for (int k = 23; k <= 24; ++k) {
            const uint64_t modulus = 1ull << (k + 1 - twos);
            for (int d = -16; d <= 16; ++d) {
                if (d == 0 || __builtin_ctz(static_cast<uint32_t>(d < 0 ? -d : d)) != twos) continue;
                const int share = d / (1 << twos);
                uint64_t middle = (static_cast<uint32_t>(-share) * inverse) & (modulus - 1u);
                if (middle < 2u * kOne) middle += (2u * kOne - middle + modulus - 1u) / modulus * modulus;
                for (; middle < 4u * kOne; middle += modulus) {
                    const int64_t numerator = static_cast<int64_t>(middle) * X + d;
                    if ((middle & 1u) == 0u || (numerator & ((1ll << (k + 1)) - 1)) != 0) continue;
                    const int64_t A = numerator >> (k + 1);
                    if (A < kOne || A >= 2 * static_cast<int64_t>(kOne)) continue;
                    const float a = scaled(static_cast<uint32_t>(A), 0);
                    ++tried;
                    wrong += psx::lt_quotient(a, x, y) != a / x;
                }
            }
        }
    }
}
int quotient() {
    constexpr uint32_t kThreads = 4u;
    long tried[kThreads] = {}, wrong[kThreads] = {};
    std::vector<std::thread> threads;
    for (uint32_t i = 0; i < kThreads; ++i)
        threads.emplace_back([&, i] { quotients(i, kThreads, tried[i], wrong[i]); });
    long all = 0, bad = 0;
    for (uint32_t i = 0; i < kThreads; ++i) {
        threads[i].join();
        all += tried[i];
        bad += wrong[i];
    }
    std::printf("%ld pairs\n", all);
    return bad != 0 || all < 90000000 || psx::lt_quotient(0.0f, 3.0f, 1.0f / 3.0f) != 0.0f;
}

// Pushes in threes and pops as the traversal makes them.  Down to the depth
// that scene compilation allows, every entry comes back; whatever the depth,
// only this lane's kTraversalStackDepth spill words are touched.
int stack() {
    constexpr uint32_t kLanes = 4u, kLane = 2u, kGuard = 400u, kForeign = 0xdeadbeefu;
    const uint32_t depth = psx::kTraversalStackDepth, rows = depth + 2u * kGuard;
    for (uint32_t deepest : {3u, 16u, 17u, 40u, depth - 2u, depth, depth + 1u, depth + 20u, depth + 300u}) {
        std::vector<uint32_t> lds(psx::kTraversalLds * kLanes, kForeign), spill(rows * kLanes, kForeign);
        psx::Stack st = psx::make_stack(lds.data(), spill.data() + kGuard * kLanes, kLanes, kLane, kLane, kLanes);
        std::vector<uint32_t> model;
        uint32_t seed = deepest, next = 1u;
        auto random = [&] { return (seed = seed * 1664525u + 1013904223u) >> 16; };
        for (int step = 0; step < 20000; ++step) {
            const bool grow = (step / 500) % 2 == 0;
            if (model.size() + 3u <= deepest && random() % 4u < (grow ? 3u : 1u)) {
                st.reserve3();
                for (int i = 0; i < 3; ++i) {
                    const bool keep = random() % 4u != 0u;
                    st.push_if(next, keep);
                    if (keep) model.push_back(next);
                    ++next;
                }
            } else if (!model.empty()) {
                const uint32_t e = st.pop();
                if (e == kForeign || (deepest <= depth && e != model.back())) return 1;
                model.pop_back();
            }
            if (st.sp != static_cast<int>(model.size())) return 1;
        }
        for (uint32_t i = 0; i < spill.size(); ++i) {
            const bool own = i % kLanes == kLane && i / kLanes >= kGuard && i / kLanes < kGuard + depth;
            if (!own && spill[i] != kForeign) return 1;
        }
        for (uint32_t i = 0; i < lds.size(); ++i)
            if ((i % kLanes != kLane || i / kLanes >= psx::kShortStack) && lds[i] != kForeign) return 1;
    }
    return 0;
}

}  // namespace

int main(int argc, char **argv) {
    const std::string what = argc == 2 ? argv[1] : "";
    int rc = 2;
    if (what == "reciprocal") rc = reciprocal();
    if (what == "root") rc = root();
    if (what == "quotient") rc = quotient();
    if (what == "stack") rc = stack();
    if (rc != 0) return 1;
    std::printf("ok\n");
    return 0;
}
