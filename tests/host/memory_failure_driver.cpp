// memory_failure_driver.cpp - libpsx.so on a device that is only pretended:
// this program defines the HIP runtime's functions itself, so the library's
// host code runs without a GPU and allocations can be made to fail.
//
// "Device" memory is host memory, kernels do nothing but check that the
// tables, films and path state they are given are live and large enough, and
// the render and pass kernels move just enough data to follow pixels from the
// film to a sink.  Usage: memory_failure_driver <scenario>; prints "ok".
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "psx.h"
#include "psx_device.h"

namespace {

struct Fake {
    std::map<const void *, std::string> kernels;  // host stub -> device name
    std::map<const char *, size_t> live;
    size_t refuse_bytes = ~static_cast<size_t>(0);  // device allocations of at least this fail
    long fail_in = -1;                              // the allocation after this many fails
    long break_in = -1;                             // the wait for an event after this many fails
    int launches = 0;
    std::vector<std::string> faults;
};
// first used by the library's static constructors, before this program's own
Fake &fake() {
    static Fake *f = new Fake;
    return *f;
}

void fault(const std::string &what) {
    if (fake().faults.size() < 8u) fake().faults.push_back(what);
}

void need(const char *kernel, const char *what, const void *p, size_t bytes) {
    const auto &live = fake().live;
    auto it = live.upper_bound(static_cast<const char *>(p));
    if (p && it != live.begin()) {
        --it;
        if (static_cast<const char *>(p) + bytes <= it->first + it->second) return;
    }
    fault(std::string(kernel) + ": " + what);
}

template <typename T>
const T &arg(void **args, int i) {
    return *static_cast<const T *>(args[i]);
}

void need_tables(const char *kernel, const psx::KernelParams &k, const float4 *sobol, const float *filter) {
    need(kernel, "sampler table", sobol, static_cast<size_t>(k.sequence_size) * 256u * 16u);
    need(kernel, "filter table", filter, 1024u * 4u);
}

// the tables of the scene's parameter version
void need_scene(const char *kernel, const psx::SceneView &s) {
    need(kernel, "parameters", s.params, 4u);
    need(kernel, "materials", s.materials, s.material_count * sizeof(psx::Material));
    need(kernel, "material shadow", s.material_shadow, s.material_count * 16u);
    need(kernel, "material emission", s.material_emission, s.material_count * 16u);
    need(kernel, "instance opacity", s.instance_opaque, s.instance_count * 4u);
    if (s.emitter_count == 0u) return;
    need(kernel, "emitters", s.emitters, s.emitter_count * sizeof(psx::Emitter));
    need(kernel, "distribution", s.distribution, s.distribution_count * sizeof(psx::DistEntry));
    need(kernel, "tree nodes", s.tree_nodes, s.tree_node_count * sizeof(psx::TreeNode));
    need(kernel, "tree emitters", s.tree_emitters, s.tree_emitter_count * sizeof(psx::TreeEmitter));
    need(kernel, "tree mapping", s.tree_mapping, s.tree_emitter_count * 8u);
    need(kernel, "emitter primitives", s.emitter_cprim, s.emitter_count * 4u);
    need(kernel, "node measures", s.node_measures, s.tree_node_count * sizeof(psx::LightMeasure));
    need(kernel, "emitter measures", s.emitter_measures, s.tree_emitter_count * sizeof(psx::LightMeasure));
}

void need_film(const char *kernel, const psx::FilmView &f, size_t n) {
    need(kernel, "combined", f.combined, n * 16u);
    need(kernel, "normal", f.normal, n * 16u);
    need(kernel, "albedo", f.albedo, n * 16u);
    need(kernel, "sample count", f.sample_count, n * 4u);
    if (f.light) need(kernel, "light", f.light, n * psx::kLightPasses * 16u);
}

void need_paths(const char *kernel, const psx::WavefrontView &w) {
    const size_t n = w.capacity;
    need(kernel, "path", w.path, n * psx::kPathWords * 16u);
    need(kernel, "shadow", w.shadow, n * psx::kShadowWords * 16u);
    need(kernel, "radiance", w.radiance, n * 16u);
    need(kernel, "normal", w.normal, n * 16u);
    need(kernel, "albedo", w.albedo, n * 16u);
    need(kernel, "first hit", w.first_hit, n * 16u);
    for (int i = 0; i < 2; ++i) {
        need(kernel, "queue", w.queue[i], n * 8u);
        need(kernel, "list", w.list[i], n * 4u);
    }
    need(kernel, "counters", w.counters, sizeof(psx::WavefrontCounters));
    if (w.lp) {
        need(kernel, "light sums", w.lp, n * 160u);
        need(kernel, "shadow split", w.shadow_split, n * 32u);
        need(kernel, "shadow transmittance", w.shadow_t, n * 16u);
    }
}

// a film whose float number i holds i (in 24 bits) and whose counts are right
void fill_film(const psx::FilmView &f, size_t pixels, uint32_t samples) {
    for (size_t i = 0; i < 4u * pixels; ++i) {
        const float v = static_cast<float>(i & 0xffffffu);
        f.combined[i] = f.normal[i] = f.albedo[i] = v;
    }
    for (size_t i = 0; i < pixels; ++i) f.sample_count[i] += samples;
}

void run(const std::string &name, void **args) {
    const char *k = name.c_str();
    auto is = [&](const char *part) { return name.find(part) != std::string::npos; };
    if (is("render_kernel")) {
        const auto &p = arg<psx::KernelParams>(args, 1);
        const auto &film = arg<psx::FilmView>(args, 4);
        const size_t n = static_cast<size_t>(p.window_width) * p.window_height;
        need_scene(k, arg<psx::SceneView>(args, 0));
        need_tables(k, p, arg<const float4 *>(args, 2), arg<const float *>(args, 3));
        need_film(k, film, n);
        if (fake().faults.empty()) fill_film(film, n, arg<uint32_t>(args, 6));
    } else if (is("generate_kernel")) {
        need_tables(k, arg<psx::KernelParams>(args, 0), arg<const float4 *>(args, 1), arg<const float *>(args, 2));
        need_paths(k, arg<psx::WavefrontView>(args, 3));
    } else if (is("wf_trace_kernel")) {
        need_paths(k, arg<psx::WavefrontView>(args, 2));
    } else if (is("wf_shade_kernel")) {
        need_paths(k, arg<psx::WavefrontView>(args, 3));
    } else if (is("accumulate_kernel")) {
        const auto &p = arg<psx::KernelParams>(args, 0);
        const auto &film = arg<psx::FilmView>(args, 2);
        const size_t n = static_cast<size_t>(p.window_width) * p.window_height;
        need_paths(k, arg<psx::WavefrontView>(args, 1));
        need_film(k, film, n);
        if (fake().faults.empty()) fill_film(film, n, arg<uint32_t>(args, 3));
    } else if (is("count_check_kernel")) {
        const auto *counts = arg<const uint32_t *>(args, 0);
        for (uint64_t i = 0; i < arg<uint64_t>(args, 1); ++i)
            if (counts[i] != arg<uint32_t>(args, 2)) *arg<uint32_t *>(args, 3) = 1u;
    } else if (is("pass_kernel")) {
        const auto &film = arg<psx::FilmView>(args, 0);
        const uint64_t n = arg<uint64_t>(args, 1);
        const uint32_t channels = static_cast<uint32_t>(k[name.find("pass_kernelILj") + 14u] - '0');
        const float *from = arg<psx::PassRule>(args, 2) == psx::PassRule::kCombined ? film.combined : film.normal;
        auto *out = arg<float *>(args, 5);
        need(k, "film", from, n * 16u);
        need(k, "pixels", out, n * channels * 4u);
        for (uint64_t i = 0; fake().faults.empty() && i < n; ++i)
            for (uint32_t c = 0; c < channels; ++c) out[i * channels + c] = from[4u * i + c];
    } else if (is("sobol_kernel")) {
        need(k, "table", arg<float4 *>(args, 0), static_cast<size_t>(arg<uint32_t>(args, 1)) * 256u * 16u);
    } else if (is("sampler_kernel")) {
        need(k, "sampler table", arg<const float4 *>(args, 1),
             static_cast<size_t>(arg<psx::KernelParams>(args, 0).sequence_size) * 256u * 16u);
    }
}

hipError_t take(void **p, size_t bytes, bool device) {
    Fake &f = fake();
    *p = nullptr;
    if (device && (bytes >= f.refuse_bytes || (f.fail_in >= 0 && f.fail_in-- == 0))) return hipErrorOutOfMemory;
    *p = std::calloc(bytes, 1u);
    if (!*p) return hipErrorOutOfMemory;
    f.live[static_cast<char *>(*p)] = bytes;
    return hipSuccess;
}
hipError_t give(void *p) {
    if (p && fake().live.erase(static_cast<char *>(p)) == 0u) fault("freed twice");
    std::free(p);
    return hipSuccess;
}
template <typename H>
hipError_t handle(H *h) {
    *h = reinterpret_cast<H>(std::malloc(1u));
    return hipSuccess;
}

}  // namespace

// ---- the HIP runtime ---------------------------------------------------------
extern "C" {
void **__hipRegisterFatBinary(const void *) {
    static void *module = nullptr;
    return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *stub, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
    fake().kernels[stub] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
namespace {
struct Config {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
} config;
}  // namespace
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
    config = Config{grid, block, shared, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream) {
    *grid = config.grid;
    *block = config.block;
    *shared = config.shared;
    *stream = config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *stub, dim3, dim3, void **args, size_t, hipStream_t) {
    ++fake().launches;
    run(fake().kernels[stub], args);
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t bytes) { return take(p, bytes, true); }
hipError_t hipMallocAsync(void **p, size_t bytes, hipStream_t) { return take(p, bytes, true); }
hipError_t hipFree(void *p) { return give(p); }
hipError_t hipFreeAsync(void *p, hipStream_t) { return give(p); }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { return take(p, bytes, false); }
hipError_t hipHostFree(void *p) { return give(p); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void *p, int v, size_t n) {
    need("hipMemset", "target", p, n);
    if (fake().faults.empty()) std::memset(p, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) { return hipMemset(p, v, n); }
hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
    *v = 256;
    return hipSuccess;
}
hipError_t hipFuncGetAttributes(hipFuncAttributes *a, const void *) {
    std::memset(a, 0, sizeof(*a));
    a->numRegs = 128;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
    *n = 4;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static char word[16];
    *p = word;
    return hipSuccess;
}
const char *hipGetErrorName(hipError_t) { return "pretended"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t *s) { return handle(s); }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t s) {
    std::free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return handle(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
    std::free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) {
    Fake &f = fake();
    return f.break_in >= 0 && f.break_in-- == 0 ? hipErrorUnknown : hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 1.0f;
    return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *) { return hipSuccess; }
}  // extern "C"

// ---- scenarios -----------------------------------------------------------------
namespace {

bool expect(bool ok, const char *what) {
    if (!ok) std::printf("failed: %s\n", what);
    return ok;
}
#define EXPECT(x) \
    if (!expect((x), #x)) return 1

struct World {
    psx_backend *backend = nullptr;
    psx_scene *scene = nullptr;
    psx_session *session = nullptr;
    psx_render_settings settings{};
    std::vector<uint32_t> passes, channels;
    uint32_t samples_per_dispatch = 1u;
    bool emissive = false;

    psx_render_settings sized(uint32_t width, uint32_t height) {
        psx_render_settings s = settings;
        s.width = width;
        s.height = height;
        return s;
    }
    bool make(uint32_t integrator, std::vector<uint32_t> kinds) {
        psx_backend_options o{1u, samples_per_dispatch, integrator, PSX_BACKEND_NO_GRAPHS};
        if (psx_backend_create(0, &o, &backend) != PSX_OK) return false;
        static const float positions[9] = {0, 0, 0, 1, 0, 0, 0, 1, 0};
        static const uint32_t triangle[3] = {0, 1, 2}, slot[1] = {0};
        static const float parameters[4] = {0.5f, 0.5f, 0.5f, 0.0f};
        psx_closure_instr diffuse{};
        diffuse.op = emissive ? PSX_CLOSURE_EMISSION : PSX_CLOSURE_DIFFUSE;
        (emissive ? diffuse.strength : diffuse.roughness) = 3u;
        static const float glow[4] = {0.5f, 0.5f, 0.5f, 1.0f};
        psx_material material{&diffuse, 1u, 0u, emissive ? glow : parameters, 4u,
                              emissive ? PSX_EMISSION_SAMPLING_FRONT_BACK : PSX_EMISSION_SAMPLING_NONE};
        psx_mesh mesh{positions, 3u, triangle, 1u, nullptr, nullptr, slot, 1u, nullptr};
        psx_instance instance{};
        instance.visibility_mask = PSX_VISIBILITY_ALL;
        psx_scene_desc d{};
        d.abi_version = PSX_ABI_VERSION;
        for (int i = 0; i < 4; ++i) instance.transform[5 * i] = d.camera.transform[5 * i] = 1.0f;
        d.materials = &material;
        d.material_count = 1u;
        d.meshes = &mesh;
        d.mesh_count = 1u;
        d.instances = &instance;
        d.instance_count = 1u;
        d.camera.field_of_view = d.camera.horizontal_field_of_view = 0.8f;
        d.camera.near_clip = 1.0e-3f;
        d.camera.far_clip = 100.0f;
        if (psx_scene_compile(backend, &d, nullptr, nullptr, &scene) != PSX_OK) return false;
        psx_render_settings_default(&settings);
        passes = std::move(kinds);
        channels.assign(passes.size(), 4u);
        settings.passes = passes.data();
        settings.pass_channels = channels.data();
        settings.pass_count = static_cast<uint32_t>(passes.size());
        const psx_render_settings s = sized(64, 48);
        return psx_session_create(scene, &s, &session) == PSX_OK;
    }
    ~World() {
        if (session) psx_session_destroy(session);
        if (scene) psx_scene_destroy(scene);
        if (backend) psx_backend_destroy(backend);
    }
};

// a larger sampler table that cannot be had, then the first one again
int table(uint32_t integrator) {
    World w;
    EXPECT(w.make(integrator, {PSX_PASS_COMBINED}));
    const psx_render_settings s = w.sized(64, 48);
    EXPECT(psx_session_render_device(w.session, 0, 1, 16) == PSX_OK);
    EXPECT(psx_session_reset(w.session, &s) == PSX_OK);
    fake().refuse_bytes = 8192u * 256u * 16u;
    EXPECT(psx_session_render_device(w.session, 0, 1, 8192) == PSX_ERROR_OUT_OF_MEMORY);
    psx_tuning_report report;
    if (integrator == PSX_INTEGRATOR_WAVEFRONT)
        EXPECT(psx_session_autotune(w.session, 1u, &report) == PSX_ERROR_OUT_OF_MEMORY);
    EXPECT(psx_session_reset(w.session, &s) == PSX_OK);
    EXPECT(psx_session_render_device(w.session, 0, 1, 16) == PSX_OK);
    fake().refuse_bytes = ~static_cast<size_t>(0);
    EXPECT(psx_session_reset(w.session, &s) == PSX_OK);
    EXPECT(psx_session_render_device(w.session, 0, 1, 8192) == PSX_OK);
    return 0;
}

// more samples a dispatch than fit, any of the arrays failing, then as many
// as before; with light passes or without
int path_state(std::vector<uint32_t> kinds) {
    for (long nth = 0; nth < 64; ++nth) {
        World w;
        w.samples_per_dispatch = 4u;
        EXPECT(w.make(PSX_INTEGRATOR_WAVEFRONT, kinds));
        EXPECT(psx_session_render_device(w.session, 0, 2, 64) == PSX_OK);
        fake().fail_in = nth;
        const int rc = psx_session_render_device(w.session, 2, 4, 64);
        const bool all_tried = fake().fail_in >= 0;
        fake().fail_in = -1;
        EXPECT(rc == (all_tried ? PSX_OK : PSX_ERROR_OUT_OF_MEMORY));
        const uint32_t first = all_tried ? 6u : 2u;
        EXPECT(psx_session_render_device(w.session, first, 1, 64) == PSX_OK);
        EXPECT(psx_session_render_device(w.session, first + 1u, 4, 64) == PSX_OK);
        if (all_tried) return 0;
    }
    return 1;
}

// a reset to a larger window, any of the film's arrays failing: the session
// renders nothing until a reset has succeeded
int film(std::vector<uint32_t> kinds) {
    for (long nth = 0; nth < 16; ++nth) {
        World w;
        EXPECT(w.make(PSX_INTEGRATOR_MEGAKERNEL, kinds));
        const psx_render_settings small = w.sized(64, 48), large = w.sized(96, 64);
        EXPECT(psx_session_render_device(w.session, 0, 1, 16) == PSX_OK);
        fake().fail_in = nth;
        const int rc = psx_session_reset(w.session, &large);
        const bool all_tried = fake().fail_in >= 0;
        fake().fail_in = -1;
        EXPECT(rc == (all_tried ? PSX_OK : PSX_ERROR_OUT_OF_MEMORY));
        if (!all_tried) {
            std::vector<float> out(96u * 64u * 64u * 12u);
            std::vector<uint32_t> words(96u * 64u * PSX_TRACE_EVENTS * PSX_TRACE_WORDS);
            EXPECT(psx_session_render_device(w.session, 0, 1, 16) == PSX_ERROR_INCOMPLETE);
            EXPECT(psx_session_render(w.session, 0, 1, 0, 16, nullptr) == PSX_ERROR_INCOMPLETE);
            EXPECT(psx_session_read_film(w.session, out.data(), nullptr, nullptr, nullptr) == PSX_ERROR_INCOMPLETE);
            EXPECT(psx_session_primary_hits(w.session, 0, 16, words.data()) == PSX_ERROR_INCOMPLETE);
            EXPECT(psx_session_trace_events(w.session, 0, 16, words.data()) == PSX_ERROR_INCOMPLETE);
            EXPECT(psx_session_path_trace(w.session, 1, 1, 0, 16, out.data(), nullptr) == PSX_ERROR_INCOMPLETE);
            EXPECT(psx_session_sampler_probe(w.session, 0, 16, 0, 4, words.data()) == PSX_ERROR_INCOMPLETE);
            psx_tuning_report report;
            EXPECT(psx_session_autotune(w.session, 1, &report) == PSX_ERROR_INCOMPLETE);
        }
        EXPECT(psx_session_reset(w.session, &small) == PSX_OK);
        EXPECT(psx_session_render_device(w.session, 0, 1, 16) == PSX_OK);
        EXPECT(psx_session_reset(w.session, &large) == PSX_OK);
        EXPECT(psx_session_render_device(w.session, 0, 1, 16) == PSX_OK);
        if (all_tried) return 0;
    }
    return 1;
}

// new parameters of which a table cannot be had: the scene keeps its old ones,
// and takes the new ones when there is memory again
int parameters(bool emissive) {
    for (long nth = 0; nth < 32; ++nth) {
        World w;
        w.emissive = emissive;
        EXPECT(w.make(PSX_INTEGRATOR_MEGAKERNEL, {PSX_PASS_COMBINED}));
        EXPECT(psx_session_render_device(w.session, 0, 1, 16) == PSX_OK);
        const float other[4] = {0.25f, 0.5f, 0.75f, emissive ? 2.0f : 0.0f};
        fake().fail_in = nth;
        const int rc = psx_scene_update_parameters(w.scene, 0u, other, 4u);
        const bool all_tried = fake().fail_in >= 0;
        fake().fail_in = -1;
        EXPECT(rc == (all_tried ? PSX_OK : PSX_ERROR_OUT_OF_MEMORY));
        EXPECT(psx_session_render_device(w.session, 1, 1, 16) == PSX_OK);
        EXPECT(psx_scene_update_parameters(w.scene, 0u, other, 4u) == PSX_OK);
        EXPECT(psx_session_render_device(w.session, 2, 1, 16) == PSX_OK);
        if (all_tried) return 0;
    }
    return 1;
}

struct Collected {
    int begun = 0, ended = 0, cancelled = 0;
    std::vector<uint32_t> kinds;
    bool right = true;
};
psx_sink collect(Collected &c) {
    psx_sink sink{};
    sink.user = &c;
    sink.begin = [](void *u, const psx_render_settings *) { static_cast<Collected *>(u)->begun++; };
    sink.write = [](void *u, uint32_t kind, uint32_t channels, uint32_t, uint32_t, uint32_t w, uint32_t h, uint32_t,
                    uint32_t, const float *p) {
        auto &c = *static_cast<Collected *>(u);
        c.kinds.push_back(kind);
        for (size_t i = 0; i < static_cast<size_t>(w) * h; ++i)
            for (uint32_t k = 0; k < channels; ++k)
                c.right &= p[i * channels + k] == static_cast<float>((4u * i + k) & 0xffffffu);
    };
    sink.end = [](void *u, int cancelled) {
        static_cast<Collected *>(u)->ended++;
        static_cast<Collected *>(u)->cancelled = cancelled;
    };
    return sink;
}

// every pass reaches the sink whole, with device memory left or without
int passes(uint32_t width, uint32_t height, std::vector<uint32_t> channels) {
    for (bool full : {false, true}) {
        World w;
        EXPECT(w.make(PSX_INTEGRATOR_MEGAKERNEL,
                      std::vector<uint32_t>(channels.size(), static_cast<uint32_t>(PSX_PASS_COMBINED))));
        w.channels = channels;
        w.settings.pass_channels = w.channels.data();
        const psx_render_settings s = w.sized(width, height);
        EXPECT(psx_session_reset(w.session, &s) == PSX_OK);
        EXPECT(psx_session_render_device(w.session, 0, 1, 16) == PSX_OK);
        if (full) fake().refuse_bytes = 0u;
        Collected c;
        const psx_sink sink = collect(c);
        EXPECT(psx_session_render(w.session, 1, 1, 0, 16, &sink) == PSX_OK);
        fake().refuse_bytes = ~static_cast<size_t>(0);
        EXPECT(c.begun == 1 && c.ended == 1 && c.cancelled == 0 && c.right && c.kinds.size() == channels.size());
    }
    return 0;
}

// a device that fails between a sink's begin and its end
int broken(uint32_t width, uint32_t height) {
    World w;
    EXPECT(w.make(PSX_INTEGRATOR_MEGAKERNEL, {PSX_PASS_COMBINED, PSX_PASS_NORMAL, PSX_PASS_ALBEDO}));
    const psx_render_settings s = w.sized(width, height);
    for (long nth = 0;; ++nth) {
        EXPECT(nth < 32);
        EXPECT(psx_session_reset(w.session, &s) == PSX_OK);
        Collected c;
        const psx_sink sink = collect(c);
        fake().break_in = nth;
        const int rc = psx_session_render(w.session, 0, 1, 0, 16, &sink);
        const bool whole = fake().break_in >= 0;
        fake().break_in = -1;
        EXPECT(rc == (whole ? PSX_OK : PSX_ERROR_DEVICE));
        EXPECT(c.begun == (nth > 0) && c.ended == c.begun && c.cancelled == (nth > 0 && !whole) && c.right);
        if (whole) return 0;
    }
}

}  // namespace

int main(int argc, char **argv) {
    if (argc != 2) return 2;
    const std::string scenario = argv[1];
    int rc = 2;
    if (scenario == "table") rc = table(PSX_INTEGRATOR_MEGAKERNEL) || table(PSX_INTEGRATOR_WAVEFRONT);
    if (scenario == "path-state")
        rc = path_state({PSX_PASS_COMBINED}) || path_state({PSX_PASS_COMBINED, PSX_PASS_DIFFUSE_DIRECT});
    if (scenario == "film") rc = film({PSX_PASS_COMBINED}) || film({PSX_PASS_COMBINED, PSX_PASS_DIFFUSE_DIRECT});
    if (scenario == "passes")
        rc = passes(64, 48, {4u, 1u, 3u, 9u}) || passes(1920, 1090, {4u, 2u, 4u}) || passes(4352, 4000, {1u, 4u, 4u, 2u});
    if (scenario == "parameters") rc = parameters(false) || parameters(true);
    if (scenario == "broken") rc = broken(64, 48) || broken(4352, 4000);
    for (const std::string &f : fake().faults) std::printf("fault: %s\n", f.c_str());
    if (rc != 0 || !fake().faults.empty() || fake().launches == 0) return 1;
    std::printf("ok\n");
    return 0;
}
