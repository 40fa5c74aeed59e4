// psx_wavefront_kernels.h - device code of the wavefront integrator (gfx950):
// path-state loads and stores, camera-ray generation, the persistent trace
// kernel, the shade step and in-order accumulation, for single sessions and
// for server batches.  Included by psx_wavefront.hip (the compiled-in kernels
// and their launchers) and by the generated surface programs that psx_rtc.cpp
// compiles at run time.
#pragma once

#include "psx_path.h"

namespace psx {
namespace {

constexpr uint32_t kTraceBlock = 256;
constexpr uint32_t kShadeBlock = 256;
constexpr uint32_t kSkip = 0xffffffffu;  // queue/list entry of a padding lane
constexpr uint32_t kMaxWavesPerCu = 32u;
// Least reservation of a trace wave: a wave's lanes.  Spreading a short queue
// thinner (16 or 8 entries a wave) is not faster on any viewport frame.
constexpr uint32_t kLeastChunk = 64u;

// Pixel of entry `rem` of a dispatch's sample plane: tiles of
// (1 << shift) x (64 >> shift) pixels, one per wave, row-major over the window.
__device__ __forceinline__ void tile_pixel(uint32_t rem, uint32_t window_width, uint32_t shift, uint32_t &px,
                                           uint32_t &py) {
    const uint32_t tile = rem >> 6, lane = rem & 63u;
    const uint32_t tw = 1u << shift;
    const uint32_t tiles_x = (window_width + tw - 1u) >> shift;
    px = (tile % tiles_x) * tw + (lane & (tw - 1u));
    py = (tile / tiles_x) * (64u >> shift) + (lane >> shift);
}

__device__ __forceinline__ void add_counter(unsigned long long *dst, uint32_t value) {
    unsigned long long v = value;
    for (int offset = 32; offset > 0; offset >>= 1) v += __shfl_down(v, offset, 64);
    if ((threadIdx.x & 63) == 0 && v != 0ull) atomicAdd(dst, v);
}

// float4 number `word` of a path's and of a shadow ray's record
__device__ __forceinline__ float4 &path_word(const WavefrontView &w, uint32_t i, uint32_t word) {
    return w.path[static_cast<size_t>(i) * kPathWords + word];
}
__device__ __forceinline__ float4 &shadow_word(const WavefrontView &w, uint32_t i, uint32_t word) {
    return w.shadow[static_cast<size_t>(i) * kShadowWords + word];
}
__device__ __forceinline__ uint32_t bits_of(float v) { return __float_as_uint(v); }
__device__ __forceinline__ float4 bit_words(uint32_t x, uint32_t y, uint32_t z, uint32_t w) {
    return make_float4(__uint_as_float(x), __uint_as_float(y), __uint_as_float(z), __uint_as_float(w));
}

// What generation stores: the camera ray and the sample's identity, in the
// film sums' arrays.  The rest of a new path is constant (new_path_state).
__device__ __forceinline__ void store_camera_path(const WavefrontView &w, uint32_t i, const PathVars &p) {
    w.radiance[i] = make_float4(p.ray.o.x, p.ray.o.y, p.ray.o.z, p.ray.tmin);
    w.normal[i] = make_float4(p.ray.d.x, p.ray.d.y, p.ray.d.z, p.ray.tmax);
    w.albedo[i] = bit_words(p.sample, p.rng_hash, 0u, 0u);
}

// The state of a path that goes on.  The MIS normal is read only by light
// sampling and forward-hit MIS, so a scene without lights (MIS = false)
// neither loads nor stores it.
template <bool MIS>
__device__ __forceinline__ void store_step(const WavefrontView &w, uint32_t i, const PathVars &p) {
    path_word(w, i, kPathOrigin) = make_float4(p.ray.o.x, p.ray.o.y, p.ray.o.z, p.ray.tmin);
    path_word(w, i, kPathDirection) = make_float4(p.ray.d.x, p.ray.d.y, p.ray.d.z, p.ray.tmax);
    path_word(w, i, kPathSource) =
        bit_words(p.src_obj, p.src_prim, p.ps.flag | (p.ps.visibility << 20) | (p.bits << 25), p.step);
    path_word(w, i, kPathThroughput) = make_float4(p.throughput.x, p.throughput.y, p.throughput.z, p.prev_pdf);
    path_word(w, i, kPathIdentity) =
        bit_words(p.sample, p.rng_hash, p.ps.bounce | (p.ps.diffuse_bounce << 16),
                  p.ps.glossy_bounce | (p.ps.transmission_bounce << 16));
    path_word(w, i, kPathUv).z = __uint_as_float(p.ps.transparent_bounce);
    if (MIS) path_word(w, i, kPathMisNormal) = make_float4(p.mis_normal.x, p.mis_normal.y, p.mis_normal.z, 0.0f);
}

// light-pass sums of a path, field-major: field f of path i at f * capacity + i
__device__ __forceinline__ void store_lp(const WavefrontView &w, uint32_t i, const LightSums &lp) {
    const size_t n = w.capacity;
    const f3 v[10] = {lp.dd, lp.di, lp.gd, lp.gi, lp.td, lp.ti, lp.emission, lp.environment, lp.path_dw, lp.path_gw};
#pragma unroll
    for (int f = 0; f < 10; ++f) w.lp[f * n + i] = make_float4(v[f].x, v[f].y, v[f].z, 0.0f);
}

__device__ __forceinline__ LightSums load_lp(const WavefrontView &w, uint32_t i) {
    const size_t n = w.capacity;
    f3 v[10];
#pragma unroll
    for (int f = 0; f < 10; ++f) {
        const float4 q = w.lp[f * n + i];
        v[f] = V(q.x, q.y, q.z);
    }
    LightSums lp;
    lp.dd = v[0];
    lp.di = v[1];
    lp.gd = v[2];
    lp.gi = v[3];
    lp.td = v[4];
    lp.ti = v[5];
    lp.emission = v[6];
    lp.environment = v[7];
    lp.path_dw = v[8];
    lp.path_gw = v[9];
    return lp;
}

// A path's state for one shade step and the hit of its ray.  The first step
// (`first`) takes the constants of a new path; later ones leave the radiance
// where it is until something is added, and read the primary Albedo only at
// bounce 0, the only steps that change it.
template <bool MIS>
__device__ __forceinline__ PathVars load_path(const WavefrontView &w, uint32_t i, bool first, Hit &h) {
    PathVars p;
    const float4 o = first ? w.radiance[i] : path_word(w, i, kPathOrigin);
    const float4 d = first ? w.normal[i] : path_word(w, i, kPathDirection);
    const float4 id = first ? w.albedo[i] : path_word(w, i, kPathIdentity);
    const float4 hv = first ? w.first_hit[i] : path_word(w, i, kPathHit);
    const float4 uv = first ? make_float4(id.z, id.w, 0.0f, 0.0f) : path_word(w, i, kPathUv);
    p.ray.o = V(o.x, o.y, o.z);
    p.ray.tmin = o.w;
    p.ray.d = V(d.x, d.y, d.z);
    p.ray.tmax = d.w;
    p.sample = bits_of(id.x);
    p.rng_hash = bits_of(id.y);
    h.inst = h.object = bits_of(hv.x);
    h.valid = h.inst != kNone;
    h.prim = bits_of(hv.y);
    h.cprim = kNone;  // resolve_surface adds the mesh's offset to `prim`
    h.tri = bits_of(hv.z);
    h.t = hv.w;
    h.u = uv.x;
    h.v = uv.y;
    if (first) {
        new_path_state(p);
        return p;
    }
    const float4 a = path_word(w, i, kPathSource), t = path_word(w, i, kPathThroughput);
    p.src_obj = bits_of(a.x);
    p.src_prim = bits_of(a.y);
    p.ps.flag = bits_of(a.z) & 0xfffffu;
    p.ps.visibility = (bits_of(a.z) >> 20) & 0x1fu;
    p.bits = bits_of(a.z) >> 25;
    p.step = bits_of(a.w);
    p.throughput = V(t.x, t.y, t.z);
    p.prev_pdf = t.w;
    p.mis_normal = V(0.0f, 0.0f, 0.0f);
    if (MIS) {
        const float4 mn = path_word(w, i, kPathMisNormal);
        p.mis_normal = V(mn.x, mn.y, mn.z);
    }
    p.ps.bounce = bits_of(id.z) & 0xffffu;
    p.ps.diffuse_bounce = bits_of(id.z) >> 16;
    p.ps.glossy_bounce = bits_of(id.w) & 0xffffu;
    p.ps.transmission_bounce = bits_of(id.w) >> 16;
    p.ps.transparent_bounce = bits_of(uv.z);
    p.ps.rng_offset = 16u * (p.step + 1u);
    p.radiance = p.normal = p.albedo = V(0.0f, 0.0f, 0.0f);
    p.transparency = 0.0f;
    p.stored = w.radiance + i;
    if (p.ps.bounce == 0u) {
        const float4 al = w.albedo[i];
        p.albedo = V(al.x, al.y, al.z);
    }
    return p;
}

// film sums of a path that has none
__device__ __forceinline__ void store_empty_film(const WavefrontView &w, uint32_t i) {
    const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    w.radiance[i] = w.normal[i] = w.albedo[i] = zero;
}

__global__ void reset_kernel(WavefrontCounters *counters, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) counters[i] = WavefrontCounters{0u, 0u, 0u, 0u};
}

// camera rays for samples [first, first + count) of every window pixel;
// `first_at`, when given, holds `first` in device memory (a replayed graph
// renders whatever range the host stored there)
__global__ __launch_bounds__(kShadeBlock) void generate_kernel(KernelParams k, const float4 *sobol,
                                                                const float *filter, WavefrontView w, uint32_t first,
                                                                uint32_t count, const uint32_t *first_at) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t total = count * w.padded_pixels;
    if (first_at) first = *first_at;
    bool live = false;
    if (i < total) {
        const uint32_t sample = first + i / w.padded_pixels;
        uint32_t px, py;
        tile_pixel(i % w.padded_pixels, k.window_width, w.tile_shift, px, py);
        if (px < k.window_width && py < k.window_height) {
            PathVars p;
            init_path(k, sobol, filter, px + k.window_x, py + k.window_y, sample, p);
            live = (p.bits & PATH_DONE) == 0u;
            if (live) {
                store_camera_path(w, i, p);
            } else {
                store_empty_film(w, i);
            }
        }
        if (w.lp && !live) {
            LightSums z;
            z.dd = z.di = z.gd = z.gi = z.td = z.ti = z.emission = z.environment = z.path_dw = z.path_gw =
                V(0.0f, 0.0f, 0.0f);
            store_lp(w, i, z);
        }
    }
    // iteration 0 lists every path in order; padding lanes are skip markers
    if (i < total) {
        w.queue[0][i] = live ? (i << 1) : kSkip;
        w.list[0][i] = live ? i : kSkip;
    }
    if (i == 0u) {
        w.counters[0].trace_count = total;
        w.counters[0].shade_count = total;
    }
}

// Persistent trace kernel.  Each lane owns one query at a time; when at least
// w.refill lanes of a wave have finished, the idle lanes take entries from
// the wave's reserved chunk of the queue and start them while the others keep
// their traversal state (Aila & Laine, "Understanding the efficiency of ray
// traversal on GPUs", 2009: persistent threads with ray replacement).
template <bool COUNT, bool SEGMENTED = false>
__global__ __launch_bounds__(kTraceBlock, 4) void wf_trace_kernel(SceneView s, KernelParams k, WavefrontView w,
                                                               uint32_t it, Counters *counters, uint32_t *spill) {
    __shared__ uint32_t lds[kTraversalLds * kTraceBlock];
    Stack st = make_stack(lds, spill, kTraceBlock, threadIdx.x, blockIdx.x * kTraceBlock + threadIdx.x,
                          gridDim.x * kTraceBlock);
    WavefrontCounters *c = w.counters + it;
    const uint32_t count = c->trace_count;
    if (count == 0u) return;
    const uint32_t *queue = w.queue[it & 1u];
    const uint32_t lane = __lane_id();
    const unsigned long long below = (1ull << lane) - 1ull;
    uint32_t rays = 0u, nodes = 0u, tris = 0u;
    Traversal t;
    traversal_idle(t, st);
    // active: the lane owns a query; it is done once its traversal is no longer busy
    bool active = false, exhausted = false, shadow = false;
    uint32_t path = 0u, tdepth = 0u;
    f3 transmittance = V(1.0f, 1.0f, 1.0f);
    const f3 no_split = V(0.0f, 0.0f, 0.0f);
    // The wave's reservation [res, res_end) of queue entries.  One atomic on
    // the shared cursor reserves `chunk` entries, which the wave hands to its
    // idle lanes over several refills: a returning atomic on one address
    // stalls the whole wave, and claiming per refill made it the largest
    // cost per ray.  `exhausted`: no chunk is left to reserve.
    uint32_t res = 0u, res_end = 0u;
    const uint32_t refill = w.refill;
    // A wave's first reservation is its own by its number, with no atomic:
    // 4096 waves that open with one on the same word take 49 us, the whole
    // time of an iteration with few rays.  A short queue is dealt out evenly
    // in the same way, down to kLeastChunk entries a wave, and then needs no
    // cursor at all.  Neighbouring reservations go to different blocks.
    // Device time of a dispatch: Cornell 256x256x1 1.61 -> 0.60 ms, instanced
    // 640x400x4 6.2 -> 4.9, Cornell 640x400x16 5.7 -> 4.9.  A reservation is
    // two trace_chunks: the cursor serves one wave in 12 ns, and much larger
    // ones spread the rays in flight over too much of the scene (device time
    // at 128, 256 and 1024 entries: instanced frame 86.9, 85.7, 89.5 ms;
    // Cornell 640x400x16 4.23, 3.89, 3.89).
    const uint32_t waves = gridDim.x * (kTraceBlock / 64u);
    const uint32_t share = (count + waves - 1u) / waves;
    uint32_t chunk = 2u * w.trace_chunk;
    const uint32_t own = min(chunk, max(share, kLeastChunk));
    const uint32_t dealt = waves * own;
    if (!SEGMENTED) {
        const uint32_t at = ((threadIdx.x >> 6) * gridDim.x + blockIdx.x) * own;
        res = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(at < count ? at : count)));
        res_end = count - res > own ? res + own : count;
        exhausted = dealt >= count;
        if (exhausted && res == res_end) return;
    }
    // SEGMENTED (w.segments = 8): the queue is cut into 8 contiguous
    // segments, each with its own cursor.  A wave starts on the segment of
    // its block's XCD (workgroups are dispatched to the 8 XCDs round-robin),
    // so each XCD's L2 sees the rays of one region of the queue, and moves to
    // the next segment when its own is drained.
    constexpr uint32_t segments = SEGMENTED ? 8u : 1u;
    uint32_t seg = blockIdx.x % segments, tried = 0u;
    for (;;) {
        if (!exhausted || res < res_end) {
            const unsigned long long idle = __ballot(!active);
            const uint32_t want = static_cast<uint32_t>(__popcll(idle));
            if (res == res_end && !exhausted && want > 0u) {
                const uint32_t leader = static_cast<uint32_t>(__ffsll(static_cast<long long>(idle)) - 1);
                if (!SEGMENTED) {
                    uint32_t b = 0u;
                    if (lane == leader) b = dealt + atomicAdd(&c->trace_fetch, chunk);
                    b = static_cast<uint32_t>(
                        __builtin_amdgcn_readlane(static_cast<int>(b), static_cast<int>(leader)));
                    if (b < count) {
                        res = b;
                        res_end = count - b > chunk ? b + chunk : count;
                    }
                    exhausted = b >= count || count - b <= chunk;
                    // smaller reservations near the end, so that the waves
                    // run out of work together
                    const uint32_t rest = exhausted ? 0u : (count - b) / (2u * waves);
                    chunk = min(chunk, max(rest, kLeastChunk));
                } else {
                    uint32_t b = 0u, e = 0u;
                    if (lane == leader) {
                        for (;;) {
                            const uint32_t begin = static_cast<uint32_t>(
                                static_cast<unsigned long long>(count) * seg / segments);
                            const uint32_t end = static_cast<uint32_t>(
                                static_cast<unsigned long long>(count) * (seg + 1u) / segments);
                            const uint32_t got = atomicAdd(&c->segment_fetch[seg], chunk);
                            if (got < end - begin) {
                                b = begin + got;
                                e = end - b > chunk ? b + chunk : end;
                                break;
                            }
                            if (++tried == segments) break;
                            seg = seg + 1u == segments ? 0u : seg + 1u;
                        }
                    }
                    const int l = static_cast<int>(leader);
                    res = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(b), l));
                    res_end = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(e), l));
                    seg = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(seg), l));
                    tried = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(tried), l));
                    exhausted = tried == segments;
                }
            }
            const uint32_t avail = res_end - res;
            const uint32_t rank = static_cast<uint32_t>(__popcll(idle & below));
            const uint32_t qi = res + rank;
            res += want < avail ? want : avail;
            if (!active && rank < avail) {
                const uint32_t entry = queue[qi];
                if (entry != kSkip) {
                    path = entry >> 1;
                    shadow = (entry & 1u) != 0u;
                    Ray ray;
                    TraceQuery q;
                    if (shadow) {
                        const float4 o = shadow_word(w, path, kShadowOrigin), d = shadow_word(w, path, kShadowDirection);
                        const float4 sq = shadow_word(w, path, kShadowIdentity);
                        ray = Ray{V(o.x, o.y, o.z), V(d.x, d.y, d.z), 0.0f, o.w};
                        q = TraceQuery{VIS_SHADOW, bits_of(sq.x), bits_of(sq.y), bits_of(sq.z), bits_of(sq.w)};
                        tdepth = bits_of(shadow_word(w, path, kShadowLight).w);
                        transmittance = V(1.0f, 1.0f, 1.0f);
                    } else {
                        const float4 o = it == 0u ? w.radiance[path] : path_word(w, path, kPathOrigin);
                        const float4 d = it == 0u ? w.normal[path] : path_word(w, path, kPathDirection);
                        ray = Ray{V(o.x, o.y, o.z), V(d.x, d.y, d.z), o.w, d.w};
                        q = TraceQuery{contract_visibility(CVIS_CAMERA), kNone, kNone, kNone, kNone};
                        if (it > 0u) {
                            const float4 a = path_word(w, path, kPathSource);
                            q.visibility = contract_visibility((bits_of(a.z) >> 20) & 0x1fu);
                            q.src_obj = bits_of(a.x);
                            q.src_prim = bits_of(a.y);
                        }
                    }
                    traversal_begin(s, t, st, ray, q);
                    active = true;
                }
            }
        }
        const unsigned long long owned = __ballot(active);
        if (owned == 0ull) {
            if (exhausted && res == res_end) break;
            continue;
        }
        // Traverse until enough lanes are idle to refill.  With nothing left
        // to refill from, stop when half of the owned lanes are done, so that
        // a shadow ray past a transparent surface does not wait for the
        // longest ray of its wave.
        const uint32_t busy_min = !exhausted || res < res_end ? 64u - refill
                                                              : static_cast<uint32_t>(__popcll(owned)) >> 1u;
        do {
            traversal_advance<COUNT>(s, t, st, nodes, tris);
        } while (static_cast<uint32_t>(__popcll(__ballot(traversal_busy(t, st)))) > busy_min);
        if (active && !traversal_busy(t, st)) {
            ++rays;
            const Hit h = traversal_result(t, st);
            if (!shadow) {
                float4 *hit = it == 0u ? w.first_hit + path : &path_word(w, path, kPathHit);
                float2 *uv = it == 0u ? reinterpret_cast<float2 *>(w.albedo + path) + 1
                                      : reinterpret_cast<float2 *>(&path_word(w, path, kPathUv));
                *hit = bit_words(h.inst, h.prim, h.tri, __float_as_uint(h.t));
                *uv = make_float2(h.u, h.v);
                active = false;
            } else {
                Ray rest;
                if (shadow_hit(s, k.transparent_max, h, rest, tdepth, transmittance)) {
                    if (w.shadow_t) {
                        // light passes: the next shade step applies it
                        w.shadow_t[path] = make_float4(transmittance.x, transmittance.y, transmittance.z, 0.0f);
                    } else {
                        // the path's radiance is not touched between the
                        // shade steps, so the light joins it here, in the
                        // order of the path: after this step's emission and
                        // before the next one's
                        const float4 L = shadow_word(w, path, kShadowLight);
                        PathVars sum;
                        sum.stored = w.radiance + path;
                        apply_shadow<false>(k, sum, V(L.x, L.y, L.z),
                                            bits_of(shadow_word(w, path, kShadowDirection).w), transmittance, no_split,
                                            no_split);
                        if (!sum.stored)
                            w.radiance[path] =
                                make_float4(sum.radiance.x, sum.radiance.y, sum.radiance.z, sum.transparency);
                    }
                    active = false;
                } else {
                    // past a transparent surface: same shadow ray from the next float
                    traversal_resume(s, t, st, rest.tmin);
                }
            }
        }
    }
    add_counter(&counters->rays, rays);
    if (COUNT) {
        add_counter(&counters->nodes, nodes);
        add_counter(&counters->tris, tris);
    }
}

// The block's shade entries sorted by the shade class of their hit (miss
// first, then one class per closure structure), with skip entries last: a
// counting sort in LDS.  Paths of one class run the same closure code, so a
// wave diverges less; the order within a class is arbitrary, and no path's
// result depends on it.  Every thread of the block calls it.
__device__ __forceinline__ uint32_t sort_block(const SceneView &s, const WavefrontView &w, uint32_t entry,
                                               bool first, uint32_t *slot, uint32_t *counts) {
    uint32_t key = 0u;
    if (entry != kSkip) {
        const uint32_t inst = bits_of(first ? w.first_hit[entry].x : path_word(w, entry, kPathHit).x);
        key = inst < s.instance_count ? s.instances[inst].shade_class : 0u;
        key = key < kShadeKeys ? key : kShadeKeys - 1u;
    }
    if (threadIdx.x < kShadeKeys) counts[threadIdx.x] = 0u;
    __syncthreads();
    const uint32_t rank = entry != kSkip ? atomicAdd(&counts[key], 1u) : 0u;
    __syncthreads();
    uint32_t offset = 0u, valid = 0u;
#pragma unroll
    for (uint32_t c = 0; c < kShadeKeys; ++c) {
        const uint32_t n = counts[c];
        offset += c < key ? n : 0u;
        valid += n;
    }
    if (entry != kSkip) slot[offset + rank] = entry;
    __syncthreads();
    const uint32_t out = threadIdx.x < valid ? slot[threadIdx.x] : kSkip;
    __syncthreads();
    return out;
}

// One shade launch: the body of wf_shade_kernel and of the shade kernels of
// generated surface programs.
template <bool LP, bool LIGHTS>
__device__ __forceinline__ void shade_launch(const SceneView &s, const KernelParams &k, const float4 *sobol,
                                             const WavefrontView &w, uint32_t it) {
    __shared__ float4 lamp_sphere[LIGHTS ? kLampCache : 1u];
    __shared__ uint32_t lamp_bits[LIGHTS ? kLampCache : 1u];
    LampView lv{lamp_sphere, lamp_bits, 0u};
    if (LIGHTS) lv = stage_lamps(s, lamp_sphere, lamp_bits);
    const WavefrontCounters *c = w.counters + it;
    WavefrontCounters *next = w.counters + it + 1u;
    const uint32_t count = c->shade_count;
    const uint32_t *list = w.list[it & 1u];
    uint32_t *next_queue = w.queue[(it + 1u) & 1u];
    uint32_t *next_list = w.list[(it + 1u) & 1u];
    const uint32_t stride = gridDim.x * blockDim.x;
    const uint32_t lane = __lane_id();
    const unsigned long long below = (1ull << lane) - 1ull;
    // this wave's reservations [q_pos, q_end) in next_queue and [l_pos, l_end)
    // in next_list: a returning atomic on the shared counters per step would
    // stall the wave, as it did the trace kernel's refill
    uint32_t q_pos = 0u, q_end = 0u, l_pos = 0u, l_end = 0u;
    __shared__ uint32_t sort_slot[kShadeBlock];
    __shared__ uint32_t sort_count[kShadeKeys];
    const bool sorted = w.shade_sort != 0u;
    const bool first = it == 0u;
    // the block steps over the list together (the sort is block-wide)
    for (uint32_t base = blockIdx.x * blockDim.x; base < count; base += stride) {
        const uint32_t i = base + threadIdx.x;
        uint32_t entry = i < count ? list[i] : kSkip;
        if (sorted) entry = sort_block(s, w, entry, first, sort_slot, sort_count);
        bool cont = false, shadow = false, live = false;
        uint32_t path = 0u;
        if (entry != kSkip) {
            path = entry;
            Hit h;
            PathVars p = load_path<LIGHTS>(w, path, first, h);
            const bool aov = p.ps.bounce == 0u;
            const uint32_t flag = p.ps.flag;
            if (LP && !first) p.lp = load_lp(w, path);
            if (LP && (p.bits & PATH_SHADOW_PENDING) != 0u) {
                const float4 L = shadow_word(w, path, kShadowLight);
                const float4 tr = w.shadow_t[path];
                const float4 a = w.shadow_split[path], b = w.shadow_split[w.capacity + path];
                apply_shadow<LP>(k, p, V(L.x, L.y, L.z), bits_of(shadow_word(w, path, kShadowDirection).w),
                                 V(tr.x, tr.y, tr.z), V(a.x, a.y, a.z), V(b.x, b.y, b.z));
                p.bits &= ~PATH_SHADOW_PENDING;
            }
            if (!LP || (p.bits & PATH_FINISHING) == 0u) {
                ShadowRay sr;
                cont = path_step<false, LP, LIGHTS>(s, lv, k, sobol, p, h, sr, nullptr);
                shadow = sr.active;
                if (shadow) {
                    shadow_word(w, path, kShadowOrigin) = make_float4(sr.ray.o.x, sr.ray.o.y, sr.ray.o.z, sr.ray.tmax);
                    shadow_word(w, path, kShadowDirection) =
                        make_float4(sr.ray.d.x, sr.ray.d.y, sr.ray.d.z, __uint_as_float(sr.depth));
                    shadow_word(w, path, kShadowIdentity) =
                        bit_words(sr.q.src_obj, sr.q.src_prim, sr.q.light_obj, sr.q.light_prim);
                    shadow_word(w, path, kShadowLight) =
                        make_float4(sr.L.x, sr.L.y, sr.L.z, __uint_as_float(sr.tdepth));
                    if (LP) {
                        w.shadow_split[path] = make_float4(sr.dw.x, sr.dw.y, sr.dw.z, 0.0f);
                        w.shadow_split[w.capacity + path] = make_float4(sr.gw.x, sr.gw.y, sr.gw.z, 0.0f);
                        p.bits |= PATH_SHADOW_PENDING;
                    }
                }
                if (LP && !cont) p.bits |= shadow ? PATH_FINISHING : PATH_DONE;
            }
            // A path that ended leaves its film sums only; what its last
            // shadow ray brings is added by the trace kernel, except to the
            // light passes, which the next shade step completes.
            live = cont || (LP && shadow);
            if (live) store_step<LIGHTS>(w, path, p);
            if (!p.stored) w.radiance[path] = make_float4(p.radiance.x, p.radiance.y, p.radiance.z, p.transparency);
            if (aov) w.albedo[path] = make_float4(p.albedo.x, p.albedo.y, p.albedo.z, 0.0f);
            if (first || ((flag ^ p.ps.flag) & FLAG_SINGLE_PASS_DONE) != 0u)
                w.normal[path] = make_float4(p.normal.x, p.normal.y, p.normal.z, 0.0f);
            if (LP) store_lp(w, path, p.lp);
        }
        // the wave's continuation entries, then its shadow entries, into its
        // queue reservation, and its live paths into its list reservation;
        // an append that overflows a reservation continues in a new chunk
        const unsigned long long cm = __ballot(cont), sm = __ballot(shadow), lm = __ballot(live);
        if ((cm | sm) != 0ull) {
            const uint32_t nc = static_cast<uint32_t>(__popcll(cm)), ns = static_cast<uint32_t>(__popcll(sm));
            const uint32_t nq = nc + ns, nl = static_cast<uint32_t>(__popcll(lm));
            // The next reservation: the entries needed now, and while steps
            // of the list lie ahead of this wave as many as they may append,
            // up to a chunk.  A short list then leaves few unused entries for
            // the next iteration to skip, and a long one takes few turns at
            // the counters, which serve one wave in 12 ns.  Device time:
            // Cornell 640x400x16 4.24 -> 3.73 ms, instanced 640x400x4 4.67 ->
            // 4.24; counting on a quarter of the paths ahead to go on costs
            // turns (4.22 ms), on twice as many leaves more unused (3.90).
            const uint32_t ahead = ((count - 1u - base) / stride) * 64u;
            const uint32_t q_old = q_pos, q_avail = q_end - q_pos;
            uint32_t q_new = 0u;
            if (nq > q_avail) {
                const uint32_t size = max(nq - q_avail, min(ahead, w.queue_chunk));
                if (lane == 0u) q_new = atomicAdd(&next->trace_count, size);
                q_new = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(q_new)));
                q_pos = q_new + (nq - q_avail);
                q_end = q_new + size;
            } else {
                q_pos += nq;
            }
            const uint32_t l_old = l_pos, l_avail = l_end - l_pos;
            uint32_t l_new = 0u;
            if (nl > l_avail) {
                const uint32_t size = max(nl - l_avail, min(ahead, kListScale * w.list_chunk));
                if (lane == 0u) l_new = atomicAdd(&next->shade_count, size);
                l_new = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(l_new)));
                l_pos = l_new + (nl - l_avail);
                l_end = l_new + size;
            } else {
                l_pos += nl;
            }
            const uint32_t qr = cont ? static_cast<uint32_t>(__popcll(cm & below))
                                     : nc + static_cast<uint32_t>(__popcll(sm & below));
            const uint32_t qs = qr < q_avail ? q_old + qr : q_new + (qr - q_avail);
            if (cont) next_queue[qs] = path << 1;
            if (shadow && !cont) next_queue[qs] = (path << 1) | 1u;
            if (cont && shadow) {
                const uint32_t r2 = nc + static_cast<uint32_t>(__popcll(sm & below));
                next_queue[r2 < q_avail ? q_old + r2 : q_new + (r2 - q_avail)] = (path << 1) | 1u;
            }
            const uint32_t lr = static_cast<uint32_t>(__popcll(lm & below));
            if (live) next_list[lr < l_avail ? l_old + lr : l_new + (lr - l_avail)] = path;
        }
    }
    // the unused ends of this wave's reservations become skip entries
    for (uint32_t j = q_pos + lane; j < q_end; j += 64u) next_queue[j] = kSkip;
    for (uint32_t j = l_pos + lane; j < l_end; j += 64u) next_list[j] = kSkip;
}

template <bool LP, bool LIGHTS>
__global__ __launch_bounds__(kShadeBlock, 2) void wf_shade_kernel(SceneView s, KernelParams k, const float4 *sobol,
                                                               WavefrontView w, uint32_t it) {
    shade_launch<LP, LIGHTS>(s, k, sobol, w, it);
}

// in-order film accumulation of the batch, one lane per window pixel
// adds one sample's light passes to a pixel's sums (w counts samples)
__device__ __forceinline__ void add_light_passes(float4 *sums, const WavefrontView &w, uint32_t path) {
    const size_t n = w.capacity;
    // LightSums fields in LightPassBuffer order; volume and colour passes stay zero
    const int field[kLightPasses] = {0, 1, 2, 3, 4, 5, -1, -1, 6, 7, -1, -1};
#pragma unroll
    for (uint32_t b = 0; b < kLightPasses; ++b) {
        float4 v = sums[b];
        if (field[b] >= 0) {
            const float4 q = w.lp[field[b] * n + path];
            v.x += q.x;
            v.y += q.y;
            v.z += q.z;
        } else {
            v.x += 0.0f;
            v.y += 0.0f;
            v.z += 0.0f;
        }
        v.w += 1.0f;
        sums[b] = v;
    }
}

__global__ __launch_bounds__(256) void accumulate_kernel(KernelParams k, WavefrontView w, FilmView film,
                                                         uint32_t count) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= w.padded_pixels) return;
    uint32_t px, py;
    tile_pixel(i, k.window_width, w.tile_shift, px, py);
    if (px >= k.window_width || py >= k.window_height) return;
    const size_t index = (size_t)py * k.window_width + px;
    float4 c = reinterpret_cast<float4 *>(film.combined)[index];
    float4 n = reinterpret_cast<float4 *>(film.normal)[index];
    float4 a = reinterpret_cast<float4 *>(film.albedo)[index];
    uint32_t completed = film.sample_count[index];
    float4 *light = film.light ? reinterpret_cast<float4 *>(film.light) + index * kLightPasses : nullptr;
    for (uint32_t s = 0; s < count; ++s) {
        const uint32_t path = s * w.padded_pixels + i;
        if (light) add_light_passes(light, w, path);
        const float4 r = w.radiance[path];
        const float4 pn = w.normal[path];
        const float4 pa = w.albedo[path];
        f3 rad = V(r.x, r.y, r.z);
        if (any_nan(rad)) rad = V(0.0f, 0.0f, 0.0f);
        c.x += rad.x;
        c.y += rad.y;
        c.z += rad.z;
        c.w += r.w;
        n.x += pn.x;
        n.y += pn.y;
        n.z += pn.z;
        n.w += 1.0f;
        a.x += pa.x;
        a.y += pa.y;
        a.z += pa.z;
        a.w += 1.0f;
        completed += 1u;
    }
    reinterpret_cast<float4 *>(film.combined)[index] = c;
    reinterpret_cast<float4 *>(film.normal)[index] = n;
    reinterpret_cast<float4 *>(film.albedo)[index] = a;
    film.sample_count[index] = completed;
}


// item of a batch-wide index: the last item whose base is <= i (bases rise)
template <bool PIXELS>
__device__ __forceinline__ uint32_t batch_item(const BatchItem *items, uint32_t n, uint32_t i) {
    uint32_t lo = 0u, len = n;
    while (len > 1u) {
        const uint32_t half = len >> 1;
        const uint32_t base = PIXELS ? items[lo + half].pixel_base : items[lo + half].path_base;
        if (base <= i) {
            lo += half;
            len -= half;
        } else {
            len = half;
        }
    }
    // every lane of a wave lies in the same item
    return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(lo)));
}

// camera rays for every item of a server batch
__global__ __launch_bounds__(kShadeBlock) void generate_batch_kernel(const BatchItem *items, uint32_t n_items,
                                                                      WavefrontView w, uint32_t total) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0u) {
        w.counters[0].trace_count = total;
        w.counters[0].shade_count = total;
    }
    if (i - threadIdx.x % 64u >= total) return;
    const BatchItem &it = items[batch_item<false>(items, n_items, i)];
    const KernelParams &k = it.k;
    const uint32_t local = i - it.path_base;
    const uint32_t sample = it.first + local / it.padded;
    const uint32_t rem = local % it.padded;
    const uint32_t tile = rem >> 6, lane = rem & 63u;
    const uint32_t tiles_x = (k.window_width + 7u) >> 3;
    const uint32_t px = (tile % tiles_x) * 8u + (lane & 7u);
    const uint32_t py = (tile / tiles_x) * 8u + (lane >> 3);
    bool live = false;
    if (px < k.window_width && py < k.window_height) {
        PathVars p;
        init_path(k, it.sobol, it.filter, px + k.window_x, py + k.window_y, sample, p);
        live = (p.bits & PATH_DONE) == 0u;
        if (live) {
            store_camera_path(w, i, p);
        } else {
            store_empty_film(w, i);
        }
    }
    w.queue[0][i] = live ? (i << 1) : kSkip;
    w.list[0][i] = live ? i : kSkip;
}

// in-order film accumulation of every item of a server batch
__global__ __launch_bounds__(256) void accumulate_batch_kernel(const BatchItem *items, uint32_t n_items,
                                                               WavefrontView w, uint32_t total_pixels) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i - threadIdx.x % 64u >= total_pixels) return;
    const BatchItem &it = items[batch_item<true>(items, n_items, i)];
    const KernelParams &k = it.k;
    const uint32_t local = i - it.pixel_base;
    const uint32_t tile = local >> 6, lane = local & 63u;
    const uint32_t tiles_x = (k.window_width + 7u) >> 3;
    const uint32_t px = (tile % tiles_x) * 8u + (lane & 7u);
    const uint32_t py = (tile / tiles_x) * 8u + (lane >> 3);
    if (px >= k.window_width || py >= k.window_height) return;
    const size_t index = (size_t)py * k.window_width + px;
    const FilmView &film = it.film;
    float4 c = reinterpret_cast<float4 *>(film.combined)[index];
    float4 n = reinterpret_cast<float4 *>(film.normal)[index];
    float4 a = reinterpret_cast<float4 *>(film.albedo)[index];
    uint32_t completed = film.sample_count[index];
    for (uint32_t s = 0; s < it.count; ++s) {
        const uint32_t path = it.path_base + s * it.padded + local;
        const float4 r = w.radiance[path];
        const float4 pn = w.normal[path];
        const float4 pa = w.albedo[path];
        f3 rad = V(r.x, r.y, r.z);
        if (any_nan(rad)) rad = V(0.0f, 0.0f, 0.0f);
        c.x += rad.x;
        c.y += rad.y;
        c.z += rad.z;
        c.w += r.w;
        n.x += pn.x;
        n.y += pn.y;
        n.z += pn.z;
        n.w += 1.0f;
        a.x += pa.x;
        a.y += pa.y;
        a.z += pa.z;
        a.w += 1.0f;
        completed += 1u;
    }
    reinterpret_cast<float4 *>(film.combined)[index] = c;
    reinterpret_cast<float4 *>(film.normal)[index] = n;
    reinterpret_cast<float4 *>(film.albedo)[index] = a;
    film.sample_count[index] = completed;
}

}  // namespace
}  // namespace psx
