// Edge validation, pose checks and FK dumps on gfx950, plus the C ABI for
// them (include/prrtc.h).
//
// Edge validation replaces the per-edge block of the reference planner
// (src/planning/pRRTC.cu:430-445): there one CUDA thread per interpolated
// pose runs fkcc<Robot> and a shared-memory atomicOr folds the verdict.
// Here one wave64 validates one edge: each pass puts up to 64 poses on the
// lanes (poses interleaved across passes so the first pass already spans the
// whole edge), the robot's check sequence runs with the obstacle tables in
// LDS, and a ballot after every check group ends the pass -- and the edge --
// at the first collision.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>

#include "host_common.h"

namespace prrtc {

// ------------------------------------------------------------------ kernels

template <class Robot>
__global__ __launch_bounds__(kWave) void k_fk_spheres(const float *__restrict__ poses, int n,
                                                      float *__restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float q[Robot::DOF];
#pragma unroll
    for (int d = 0; d < Robot::DOF; d++) q[d] = poses[(size_t)i * Robot::DOF + d];
    Robot::fk_spheres(q, out + (size_t)i * Robot::NSPHERES * 3);
}

// Lane l of a wave takes pose base + l.  Ctx: CheckCtx where the poses of a
// wave lie together (a path's), SpreadCtx where they have nothing to do with
// each other (samples); the verdicts are the same (see launch_check).
template <class Robot, class Ctx>
__global__ __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(2))) void k_check_poses(const float *__restrict__ scene, int scene_f4,
                                                       const float *__restrict__ poses, int n,
                                                       uint8_t *__restrict__ out) {
    extern __shared__ float4 lds_scene[];
    Ctx ctx;
    ctx.independent = true;
    ctx.key = 0;
    bind_scene(scene, scene_f4, lds_scene, ctx.obs);
    for (int base = blockIdx.x * kWave; base < n; base += gridDim.x * kWave) {
        const int i = base + threadIdx.x;
        const int src = i < n ? i : n - 1;
        float q[Robot::DOF];
#pragma unroll
        for (int d = 0; d < Robot::DOF; d++) q[d] = poses[(size_t)src * Robot::DOF + d];
        ctx.coll = false;
        ctx.dead = i >= n;
        Robot::check(q, ctx);
        if (i < n) out[i] = ctx.coll ? 0 : 1;
    }
}

// One wave per edge (grid-stride over edges).  Pass p of P = ceil(g/64)
// gives lane l the pose k = l*P + p; pose k is a + (k+1) * ((b-a)/g).
template <class Robot>
__global__ __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(2))) void k_validate_edges(const float *__restrict__ scene, int scene_f4,
                                                          const float *__restrict__ edges, int n, int g,
                                                          uint8_t *__restrict__ out) {
    extern __shared__ float4 lds_scene[];
    constexpr int D = Robot::DOF;
    CheckCtx ctx;
    ctx.independent = false;
    bind_scene(scene, scene_f4, lds_scene, ctx.obs);
    const int lane = threadIdx.x;
    const int passes = (g + kWave - 1) / kWave;
    const float gf = (float)g;
    const XcdRange range(n);   // edges are 4*2*D bytes and straddle lines
    for (int e = range.first; e < range.end; e += range.stride) {
        const float *a = edges + (size_t)e * 2 * D;
        const float *b = a + D;
        float av[D], dv[D];
#pragma unroll
        for (int d = 0; d < D; d++) {
            av[d] = a[d];
            dv[d] = (b[d] - av[d]) / gf;
        }
        bool bad = false;
        for (int p = 0; p < passes && !bad; p++) {
            const int k = lane * passes + p;
            const float kk = (float)((k < g ? k : g - 1) + 1);
            float q[D];
#pragma unroll
            for (int d = 0; d < D; d++) q[d] = fmaf(kk, dv[d], av[d]);
            ctx.coll = false;
            ctx.dead = k >= g;
            ctx.key = 0;
            Robot::check(q, ctx);
            bad = ballot(ctx.coll) != 0;
        }
        if (lane == 0) out[e] = bad ? 0 : 1;
    }
}

// ------------------------------------------------------------------ helpers

static thread_local std::string g_error;

void set_error(const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_error = buf;
}

int robot_dof(int robot) {
    switch (robot) {
#define PRRTC_DOF_CASE(ID, R) case ID: return R::DOF;
        PRRTC_FOR_EACH_ROBOT(PRRTC_DOF_CASE)
#undef PRRTC_DOF_CASE
        default: return -1;
    }
}

int robot_num_spheres(int robot) {
    switch (robot) {
#define PRRTC_NSPH_CASE(ID, R) case ID: return R::NSPHERES;
        PRRTC_FOR_EACH_ROBOT(PRRTC_NSPH_CASE)
#undef PRRTC_NSPH_CASE
        default: return -1;
    }
}

bool scene_valid(const prrtc_scene *s) {
    if (!s) return false;
    const int n[5] = {s->n_spheres, s->n_capsules, s->n_z_capsules, s->n_cuboids, s->n_z_cuboids};
    const float *p[5] = {s->spheres, s->capsules, s->z_capsules, s->cuboids, s->z_cuboids};
    const int w[5] = {4, 8, 8, 15, 15};
    for (int t = 0; t < 5; t++) {
        if (n[t] < 0 || (n[t] > 0 && !p[t])) return false;
        for (int i = 0; i < n[t] * w[t]; i++)
            if (!std::isfinite(p[t][i])) return false;
    }
    return true;
}

// Cull radius of a cuboid with half-extents h: its half-diagonal |h| (the box
// lies inside the ball of that radius about its centre), padded by 2^-16
// relative and 1 mm absolute.  A robot sphere (radius r) whose centre is
// farther than r + cull from the box centre is at least 1 mm from the box,
// so the box test's value is positive by a margin far above the rounding
// of either computation: skipping the test cannot change a verdict.  A
// non-finite extent gives a non-finite radius, which never culls.
static float cuboid_cull_radius(const float *h) {
    const double R = std::sqrt((double)h[0] * h[0] + (double)h[1] * h[1] + (double)h[2] * h[2]);
    return (float)(R * (1.0 + 1.0 / 65536.0) + 1e-3);
}

size_t scene_packed_floats(const prrtc_scene *s) {
    return 8 + 4 * (size_t)scene_payload_f4(s->n_spheres, s->n_capsules, s->n_z_capsules, s->n_cuboids,
                                            s->n_z_cuboids);
}

int scene_lds_f4(const prrtc_scene *s) {
    return scene_lds_f4(s->n_spheres, s->n_capsules, s->n_z_capsules, s->n_cuboids, s->n_z_cuboids);
}

void scene_pack(const prrtc_scene *s, float *out) {
    const int nf4 = scene_payload_f4(s->n_spheres, s->n_capsules, s->n_z_capsules, s->n_cuboids, s->n_z_cuboids);
    int32_t hdr[8] = {s->n_spheres, s->n_capsules, s->n_z_capsules, s->n_cuboids, s->n_z_cuboids, nf4, 0, 0};
    std::memcpy(out, hdr, sizeof hdr);
    float *o = out + 8;
    for (int i = 0; i < s->n_spheres; i++, o += 4) std::memcpy(o, s->spheres + 4 * i, 4 * sizeof(float));
    auto caps = [&](const float *c, int n) {
        for (int i = 0; i < n; i++, o += 8) {
            const float *r = c + 8 * i;  // x1 y1 z1 xv yv zv r rdv
            const float v[8] = {r[0], r[1], r[2], r[6], r[3], r[4], r[5], r[7]};
            std::memcpy(o, v, sizeof v);
        }
    };
    caps(s->capsules, s->n_capsules);
    caps(s->z_capsules, s->n_z_capsules);
    auto cubs = [&](const float *c, int n) {
        for (int i = 0; i < n; i++, o += 16) {
            const float *r = c + 15 * i;  // x y z a1 a2 a3 r1 r2 r3
            const float v[16] = {r[0], r[1], r[2], r[12], r[3], r[4], r[5], r[13],
                                 r[6], r[7], r[8], r[14], r[9], r[10], r[11], cuboid_cull_radius(r + 12)};
            std::memcpy(o, v, sizeof v);
        }
    };
    cubs(s->cuboids, s->n_cuboids);
    cubs(s->z_cuboids, s->n_z_cuboids);
}

int num_cus() {
    static int cus = 0;
    static std::once_flag once;
    std::call_once(once, [] {
        int dev = 0;
        hipDeviceProp_t prop;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
            cus = prop.multiProcessorCount;
        if (cus <= 0) cus = 256;
    });
    return cus;
}

template <class... KArgs, class... Args>
static void launch_scene_kernel(void (*k)(KArgs...), dim3 grid, int lds_f4, hipStream_t st, Args... args) {
    hipLaunchKernelGGL(k, grid, dim3(kWave), lds_f4 * sizeof(float4), st, args...);
    PRRTC_HIP(hipGetLastError());
}

template <class Robot>
static void launch_validate(const float *d_scene, size_t scene_f4, int lds_f4, const float *d_edges, int n, int g,
                            uint8_t *d_out, hipStream_t st) {
    // three workgroups for each of the eight waves a CU holds: edges take
    // uneven time, and the last ones even out; each workgroup stages the
    // scene, so many more would cost.  Against two: 10k Fetch edges 82 -> 79
    // us (139 -> 131 on another scene), 30k Baxter edges 260 -> 249 us.
    const int grid = std::max(1, std::min(n, num_cus() * 24));
    launch_scene_kernel(k_validate_edges<Robot>, dim3(grid), lds_f4, st, d_scene, (int)scene_f4, d_edges,
                        n, g, d_out);
}

// Whether the poses (on the host) are samples rather than paths: most blocks of
// 64, at most 64 of them asked, hold a pose farther than `apart` (2-norm over
// the joints) from their first, among three of them.
static bool poses_apart(const float *poses, int n, int dof, float apart) {
    const int blocks = (n + kWave - 1) / kWave, asked = std::min(blocks, 64);
    int far = 0;
    for (int j = 0; j < asked; j++) {
        const size_t first = (size_t)((long long)blocks * j / asked) * kWave;
        const size_t last = std::min(first + kWave, (size_t)n) - 1;
        float most = 0.0f;
        for (int k = 1; k <= 3; k++) {
            const float *p = poses + first * dof, *q = poses + (first + (last - first) * k / 3) * dof;
            float d2 = 0.0f;
            for (int d = 0; d < dof; d++) d2 += (q[d] - p[d]) * (q[d] - p[d]);
            most = std::max(most, d2);
        }
        far += most > apart * apart;
    }
    return 2 * far > asked;
}

// Poses of a path are checked like an edge's, by balls over the wave; samples
// pose by pose (SpreadCtx), since balls around them rule out little and cost
// their own forming and a branch per gate and obstacle.  kSpread is the length
// of a 64-pose path at which both take the same time: Panda 2 to 2.5, Fetch
// 1.5 to 2, Baxter 4 to 5, UR5 3 to 5, over scenes of 12 to 4096 obstacles
// (the point robot 4, in metres).
// 4096 uniform poses by balls and pose by pose: Panda, 72 obstacles 207 and 157
// us, 1000 spheres 1182 and 860; Baxter, 32 boxes 73 and 50 us, 1000 spheres
// 1084 and 648.  64 paths of 0.5 rad: Panda, 72 obstacles 26 and 48 us, 1000
// spheres 73 and 236.  65536 uniform positions of the point robot among 1000
// spheres: 149 and 32 us.
template <class Robot>
static void launch_check(const float *d_scene, size_t scene_f4, int lds_f4, const float *d_poses, int n, bool apart,
                         uint8_t *d_out, hipStream_t st) {
    const int blocks = std::max(1, std::min((n + kWave - 1) / kWave, num_cus() * 16));
    launch_scene_kernel(apart ? k_check_poses<Robot, SpreadCtx> : k_check_poses<Robot, CheckCtx>, dim3(blocks), lds_f4,
                        st, d_scene, (int)scene_f4, d_poses, n, d_out);
}

template <class Robot>
static void spread_of(float &out) { out = Robot::kSpread; }

// Scenes are staged whole into LDS: at most kMaxLdsScene bytes of tables
// (4096 float4: e.g. 1024 cuboids or 4096 spheres).
static bool scene_fits(size_t scene_f4) { return scene_f4 * sizeof(float4) <= kMaxLdsScene; }

template <class Robot>
static void launch_fk(const float *d_poses, int n, float *d_out, hipStream_t st) {
    hipLaunchKernelGGL(k_fk_spheres<Robot>, dim3((n + kWave - 1) / kWave), dim3(kWave), 0, st, d_poses, n, d_out);
    PRRTC_HIP(hipGetLastError());
}

// FN<Robot>(args...) for the robot id, over every robot of
// PRRTC_FOR_EACH_ROBOT (the arguments reach each case through a lambda)
#define PRRTC_DISPATCH_CASE(ID, R) \
    case ID: call_(RobotTag<R>{}); break;
#define PRRTC_DISPATCH(robot, FN, ...)                                              \
    do {                                                                            \
        auto call_ = [&](auto tag) { FN<typename decltype(tag)::type>(__VA_ARGS__); }; \
        switch (robot) { PRRTC_FOR_EACH_ROBOT(PRRTC_DISPATCH_CASE) }                 \
    } while (0)

static bool all_finite(const float *p, size_t n) {
    for (size_t i = 0; i < n; i++)
        if (!std::isfinite(p[i])) return false;
    return true;
}

// Copies n floats and says whether all are finite (one pass, without an
// early exit, so that it vectorizes).
static bool copy_finite(float *dst, const float *src, size_t n) {
    uint32_t bad = 0;
    for (size_t i = 0; i < n; i++) {
        uint32_t b;
        std::memcpy(&b, src + i, sizeof b);
        std::memcpy(dst + i, &b, sizeof b);
        bad |= (uint32_t)((b & 0x7f800000u) == 0x7f800000u);
    }
    return bad == 0;
}

static HostCall &host_call() {
    static thread_local HostCall hc;
    return hc;
}

// One verdict call on host buffers: packed scene and n_floats of input go up
// in one copy, `launch` queues the kernel on the stream, n verdict bytes come
// back.  Returns false, with nothing launched, if the input is not finite.
template <class Launch>
static bool verdict_call(const prrtc_scene *scene, const float *in, size_t n_floats, int n, uint8_t *out,
                         Launch &&launch) {
    const size_t scene_bytes = (sizeof(float) * scene_packed_floats(scene) + 255) & ~size_t(255);
    const size_t in_bytes = (sizeof(float) * n_floats + 255) & ~size_t(255);
    const size_t up = scene_bytes + in_bytes, total = up + (size_t)n;
    if (total > HostCall::kMost) {
        // the copies outweigh the allocations, and pinning as much would not pay
        if (!all_finite(in, n_floats)) return false;
        std::vector<float> packed(scene_packed_floats(scene));
        scene_pack(scene, packed.data());
        DevBuf<float> ds(packed.size()), di(n_floats);
        DevBuf<uint8_t> dout(n);
        PRRTC_HIP(hipMemcpy(ds.p, packed.data(), sizeof(float) * packed.size(), hipMemcpyHostToDevice));
        PRRTC_HIP(hipMemcpy(di.p, in, sizeof(float) * n_floats, hipMemcpyHostToDevice));
        launch(ds.p, di.p, dout.p, (hipStream_t)0);
        PRRTC_HIP(hipMemcpy(out, dout.p, n, hipMemcpyDeviceToHost));
        return true;
    }
    HostCall &hc = host_call();
    hc.need(total);
    if (!copy_finite(reinterpret_cast<float *>(hc.host + scene_bytes), in, n_floats)) return false;
    const hipStream_t s = nullptr;
    struct Drain {   // a call that fails half way leaves nothing queued on the buffers
        bool done = false;
        ~Drain() {
            if (!done) (void)hipStreamSynchronize(nullptr);
        }
    } drain;
    scene_pack(scene, reinterpret_cast<float *>(hc.host));
    PRRTC_HIP(hipMemcpyAsync(hc.dev, hc.host, scene_bytes + sizeof(float) * n_floats, hipMemcpyHostToDevice, s));
    launch(reinterpret_cast<const float *>(hc.dev), reinterpret_cast<const float *>(hc.dev + scene_bytes),
           reinterpret_cast<uint8_t *>(hc.dev + up), s);
    PRRTC_HIP(hipMemcpyAsync(hc.host + up, hc.dev + up, (size_t)n, hipMemcpyDeviceToHost, s));
    PRRTC_HIP(hipStreamSynchronize(s));
    drain.done = true;
    std::memcpy(out, hc.host + up, (size_t)n);
    return true;
}

}  // namespace prrtc

using namespace prrtc;

// ------------------------------------------------------------------ C ABI

extern "C" {

int prrtc_version(void) { return 1; }

const char *prrtc_last_error(void) { return g_error.c_str(); }

void prrtc_settings_default(prrtc_settings *s) {
    if (!s) return;
    // pRRTC_settings.hh:4-16
    s->max_samples = 1000000;
    s->max_iters = 1000000;
    s->num_new_configs = 600;
    s->granularity = 64;
    s->range = 0.5f;
    s->balance = 1;
    s->tree_ratio = 0.5f;
    s->dynamic_domain = 1;
    s->dd_alpha = 0.0001f;
    s->dd_radius = 4.0f;
    s->dd_min_radius = 1.0f;
    s->seed = 1;
}

int prrtc_robot_dof(int robot) { return robot_dof(robot); }

int prrtc_robot_num_spheres(int robot) { return robot_num_spheres(robot); }

size_t prrtc_scene_packed_floats(const prrtc_scene *scene) {
    if (!scene) return 0;
    return scene_packed_floats(scene);
}

int prrtc_scene_pack(const prrtc_scene *scene, float *out, size_t cap_floats) {
    if (!scene_valid(scene) || !out) {
        set_error("prrtc_scene_pack: invalid scene or output");
        return PRRTC_EINVAL;
    }
    if (cap_floats < scene_packed_floats(scene)) {
        set_error("prrtc_scene_pack: output holds %zu floats, %zu needed", cap_floats, scene_packed_floats(scene));
        return PRRTC_EOVERFLOW;
    }
    scene_pack(scene, out);
    return PRRTC_OK;
}

int prrtc_fk_spheres(int robot, const float *poses, int n, float *out_centres) {
    return guarded("prrtc_fk_spheres", [&]() -> int {
        const int D = robot_dof(robot), S = robot_num_spheres(robot);
        if (D < 0 || n < 0 || (n > 0 && (!poses || !out_centres))) {
            set_error("prrtc_fk_spheres: invalid argument");
            return PRRTC_EINVAL;
        }
        if (n == 0) return PRRTC_OK;
        DevBuf<float> dq((size_t)n * D), dc((size_t)n * S * 3);
        PRRTC_HIP(hipMemcpy(dq.p, poses, sizeof(float) * n * D, hipMemcpyHostToDevice));
        PRRTC_DISPATCH(robot, launch_fk, dq.p, n, dc.p, (hipStream_t)0);
        PRRTC_HIP(hipMemcpy(out_centres, dc.p, sizeof(float) * (size_t)n * S * 3, hipMemcpyDeviceToHost));
        return PRRTC_OK;
    });
}

int prrtc_check_poses(int robot, const prrtc_scene *scene, const float *poses, int n, uint8_t *out_free) {
    return guarded("prrtc_check_poses", [&]() -> int {
        const int D = robot_dof(robot);
        if (D < 0 || n < 0 || !scene_valid(scene) || (n > 0 && (!poses || !out_free))) {
            set_error("prrtc_check_poses: invalid argument");
            return PRRTC_EINVAL;
        }
        if (n == 0) return PRRTC_OK;
        const size_t f4 = (scene_packed_floats(scene) - 8) / 4;
        const bool fits = scene_fits(f4);
        const bool finite = fits ? verdict_call(scene, poses, (size_t)n * D, n, out_free,
                                                [&](const float *ds, const float *dq, uint8_t *dout, hipStream_t st) {
                                                    float spread = 0.0f;
                                                    PRRTC_DISPATCH(robot, spread_of, spread);
                                                    const bool apart = poses_apart(poses, n, D, spread);
                                                    PRRTC_DISPATCH(robot, launch_check, ds, f4, scene_lds_f4(scene), dq, n, apart,
                                                                   dout, st);
                                                })
                                 : all_finite(poses, (size_t)n * D);
        if (!finite) {
            set_error("prrtc_check_poses: non-finite pose");
            return PRRTC_EINVAL;
        }
        if (!fits) {
            set_error("prrtc_check_poses: scene tables exceed %zu bytes", kMaxLdsScene);
            return PRRTC_EINVAL;
        }
        return PRRTC_OK;
    });
}

int prrtc_validate_edges(int robot, const prrtc_scene *scene, const float *edges, int n, int granularity,
                         uint8_t *out_free) {
    return guarded("prrtc_validate_edges", [&]() -> int {
        const int D = robot_dof(robot);
        if (D < 0 || n < 0 || granularity < 1 || !scene_valid(scene) || (n > 0 && (!edges || !out_free))) {
            set_error("prrtc_validate_edges: invalid argument");
            return PRRTC_EINVAL;
        }
        if (n == 0) return PRRTC_OK;
        const size_t f4 = (scene_packed_floats(scene) - 8) / 4;
        const bool fits = scene_fits(f4);
        const bool finite = fits ? verdict_call(scene, edges, (size_t)n * 2 * D, n, out_free,
                                                [&](const float *ds, const float *de, uint8_t *dout, hipStream_t st) {
                                                    PRRTC_DISPATCH(robot, launch_validate, ds, f4, scene_lds_f4(scene), de, n,
                                                                   granularity, dout, st);
                                                })
                                 : all_finite(edges, (size_t)n * 2 * D);
        if (!finite) {
            set_error("prrtc_validate_edges: non-finite edge endpoint");
            return PRRTC_EINVAL;
        }
        if (!fits) {
            set_error("prrtc_validate_edges: scene tables exceed %zu bytes", kMaxLdsScene);
            return PRRTC_EINVAL;
        }
        return PRRTC_OK;
    });
}

int prrtc_validate_edges_async(int robot, const float *d_scene, size_t scene_floats, const float *d_edges, int n,
                               int granularity, uint8_t *d_out_free, void *stream) {
    return guarded("prrtc_validate_edges_async", [&]() -> int {
        const int D = robot_dof(robot);
        if (D < 0 || n < 0 || granularity < 1 || !d_scene || scene_floats < 8 || (scene_floats - 8) % 4 ||
            (n > 0 && (!d_edges || !d_out_free))) {
            set_error("prrtc_validate_edges_async: invalid argument");
            return PRRTC_EINVAL;
        }
        if (n == 0) return PRRTC_OK;
        if (!scene_fits((scene_floats - 8) / 4)) {
            set_error("prrtc_validate_edges_async: scene tables exceed %zu bytes", kMaxLdsScene);
            return PRRTC_EINVAL;
        }
        const size_t f4 = (scene_floats - 8) / 4;
        PRRTC_DISPATCH(robot, launch_validate, d_scene, f4, scene_lds_f4_most((int)f4), d_edges, n, granularity,
                       d_out_free, (hipStream_t)stream);
        return PRRTC_OK;
    });
}

}  // extern "C"
