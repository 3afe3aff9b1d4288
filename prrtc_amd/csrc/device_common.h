// Device building blocks of the pRRTC hot path for gfx950 (CDNA4, wave64).
//
//  * packed scene layout (float4 tables) and its LDS staging;
//  * sphere-vs-obstacle tests in the reference's squared form
//    (src/planning/utils.cuh:58-208): value < 0 means collision;
//  * check contexts that the generated robot code drives, with the
//    wavefront-level early exit (ballot after every check group);
//  * robot dispatch (Sphere / Panda / Fetch / Baxter).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "robots/baxter.gen.h"
#include "robots/fetch.gen.h"
#include "robots/panda.gen.h"
#include "robots/ur5.gen.h"

namespace prrtc {

constexpr int kWave = 64;
constexpr int kXcds = 8;   // MI355X: 8 XCDs, workgroups dispatched to them round-robin
constexpr int kMaxDof = 14;
// Largest obstacle table set staged into LDS per workgroup.
constexpr size_t kMaxLdsScene = 64 * 1024;

// ---------------------------------------------------------------------------
// packed scene: a header of two float4 (int counts), then the tables
//   spheres  : 1 float4 each   (x, y, z, r)
//   capsules : 2 float4 each   (x1, y1, z1, r) (xv, yv, zv, rdv)
//   z-caps   : 2 float4 each
//   cuboids  : 4 float4 each   (x, y, z, r1) (a1, r2) (a2, r3) (a3, cull)
//   z-cuboids: 4 float4 each   (cull: padded half-diagonal, set by the host pack)
struct SceneHeader {
    int32_t n_sph, n_cap, n_zcap, n_cub, n_zcub, n_f4, pad0, pad1;
};
static_assert(sizeof(SceneHeader) == 32, "header is two float4");

__host__ __device__ inline int scene_payload_f4(int n_sph, int n_cap, int n_zcap, int n_cub, int n_zcub) {
    return n_sph + 2 * (n_cap + n_zcap) + 4 * (n_cub + n_zcub);
}

// Obstacle tables as seen by one workgroup: counts in registers (uniform),
// payload in LDS (staged).  `ball` holds a bounding ball (centre, padded
// radius) of every obstacle that is not a sphere, in table order (capsules,
// z-capsules, cuboids, z-cuboids); a sphere's row is its own ball.  An
// obstacle is named by its index in the whole scene, spheres first.
struct Obstacles {
    const float4 *sph, *cap, *zcap, *cub, *zcub, *ball;
    int n_sph, n_cap, n_zcap, n_cub, n_zcub;

    __device__ void bind(const SceneHeader &h, const float4 *payload) {
        n_sph = h.n_sph; n_cap = h.n_cap; n_zcap = h.n_zcap; n_cub = h.n_cub; n_zcub = h.n_zcub;
        sph = payload;
        cap = sph + n_sph;
        zcap = cap + 2 * n_cap;
        cub = zcap + 2 * n_zcap;
        zcub = cub + 4 * n_cub;
        ball = zcub + 4 * n_zcub;
    }
    __device__ __forceinline__ int count() const { return n_sph + n_cap + n_zcap + n_cub + n_zcub; }
};

// Part `part` of 2^shift of a scene's obstacles: i with i mod 2^shift ==
// part.  Planner waves that share a pass's poses each take one.
struct Share {
    int part = 0, shift = 0;
};

// LDS float4 of a staged scene: its tables and a ball for every obstacle that
// is not a sphere.  Where the host sees only a device copy (scene_f4 float4 of
// tables): the most it can be, one ball per two float4 of tables.  What a
// workgroup asks for and does not use costs resident waves: 65536 Baxter poses
// against 4096 spheres, asked for 96 KiB and for the 64 they need, 10.5 and 5.8
// ms; 1024 boxes, 96 and 80 KiB, 5.1 and 2.8 ms.
__host__ __device__ constexpr int scene_lds_f4(int n_sph, int n_cap, int n_zcap, int n_cub, int n_zcub) {
    return n_sph + 3 * (n_cap + n_zcap) + 5 * (n_cub + n_zcub);
}
__host__ __device__ constexpr int scene_lds_f4_most(int scene_f4) { return scene_f4 + scene_f4 / 2; }

// Read a packed scene's header.  `cap_f4` is the payload size the host
// allocated; a header that does not fit it (or is inconsistent) is read as an
// empty scene, so no access leaves the buffer.
__device__ inline void read_header(const float *packed, int cap_f4, SceneHeader &h) {
    const int4 *hdr = reinterpret_cast<const int4 *>(packed);
    const int4 h0 = hdr[0], h1 = hdr[1];
    h.n_sph = h0.x; h.n_cap = h0.y; h.n_zcap = h0.z; h.n_cub = h0.w;
    h.n_zcub = h1.x; h.n_f4 = h1.y; h.pad0 = 0; h.pad1 = 0;
    const bool ok = h.n_sph >= 0 && h.n_cap >= 0 && h.n_zcap >= 0 && h.n_cub >= 0 && h.n_zcub >= 0 &&
                    h.n_f4 == scene_payload_f4(h.n_sph, h.n_cap, h.n_zcap, h.n_cub, h.n_zcub) && h.n_f4 <= cap_f4;
    if (!ok) h = SceneHeader{0, 0, 0, 0, 0, 0, 0, 0};
}

__host__ __device__ __forceinline__ float sq3(float dx, float dy, float dz) {
#pragma clang fp contract(off)
    return fmaf(dx, dx, fmaf(dy, dy, dz * dz));
}

// Ball about a segment's midpoint that holds the capsule of rows (p, r) and
// (v, .): radius |v|/2 + |r| (a test squares r + the sphere's radius, so a
// negative one reaches as far), padded by 2^-16 relative, 1 mm absolute and
// 2^-20 of the midpoint's coordinates.  The pads cover the rounding of sqrtf,
// of the midpoint and of the tests they replace many times over (the midpoint
// and a test's nearest point on the segment are rounded to 2^-24 of their
// coordinates, more than 1 mm beyond 16 km).
__host__ __device__ __forceinline__ float4 capsule_ball(const float4 &p, float vx, float vy, float vz) {
#pragma clang fp contract(off)
    const float x = fmaf(0.5f, vx, p.x), y = fmaf(0.5f, vy, p.y), z = fmaf(0.5f, vz, p.z);
    const float far = fmaxf(fmaxf(fabsf(x), fabsf(y)), fabsf(z));
    return make_float4(x, y, z, fmaf(0.5f * sqrtf(sq3(vx, vy, vz)) + fabsf(p.w), 1.0f + 0x1p-16f,
                                     fmaf(0x1p-20f, far, 1e-3f)));
}

// Copy a packed scene's payload into LDS and append the balls
// (scene_lds_f4 of it in all); every lane of the workgroup helps.
__device__ inline void stage_scene(const float *packed, int cap_f4, float4 *lds, SceneHeader &h) {
#pragma clang fp contract(off)
    read_header(packed, cap_f4, h);
    const float4 *src = reinterpret_cast<const float4 *>(packed) + 2;
    for (int i = threadIdx.x; i < h.n_f4; i += blockDim.x) lds[i] = src[i];
    const float4 *cap = src + h.n_sph, *cub = cap + 2 * (h.n_cap + h.n_zcap);
    const int n_caps = h.n_cap + h.n_zcap, n_balls = n_caps + h.n_cub + h.n_zcub;
    for (int i = threadIdx.x; i < n_balls; i += blockDim.x) {
        float4 b;
        if (i < n_caps) {
            const float4 p = cap[2 * i];
            float4 v = cap[2 * i + 1];
            if (i >= h.n_cap) v.x = v.y = 0.0f;   // a z-capsule's test reads v.z alone
            b = capsule_ball(p, v.x, v.y, v.z);
        } else {
            const float4 *row = cub + 4 * (i - n_caps);
            b = row[0];
            b.w = row[3].w;   // the cull radius of the host pack
        }
        lds[h.n_f4 + i] = b;
    }
    __syncthreads();
}

// Stage a packed scene for a workgroup.
__device__ inline void bind_scene(const float *packed, int cap_f4, float4 *lds, Obstacles &obs) {
    SceneHeader h;
    stage_scene(packed, cap_f4, lds, h);
    obs.bind(h, lds);
}

// The items 0 .. n - 1 of a launch that workgroup blockIdx.x takes, by first,
// end and stride.  Workgroups reach the XCDs round-robin (workgroup b runs on
// XCD b % 8) and each XCD has its own L2, so each XCD's workgroups share one
// contiguous range: what neighbouring items read (an edge list's lines, a
// tree) comes into one L2 instead of all eight.
struct XcdRange {
    int first, end, stride;
    __device__ __forceinline__ explicit XcdRange(int n) {
        first = blockIdx.x;
        end = n;
        stride = gridDim.x;
        if ((int)gridDim.x >= kXcds) {
            const int x = blockIdx.x % kXcds;
            first = (int)((long long)n * x / kXcds) + blockIdx.x / kXcds;
            end = (int)((long long)n * (x + 1) / kXcds);
            stride = ((int)gridDim.x - x + kXcds - 1) / kXcds;   // workgroups on this XCD
        }
    }
};

__device__ __forceinline__ uint64_t ballot(bool p) { return __ballot(p); }

// Obstacle table read.  LOCAL: the tables are known to be staged in LDS, so
// the generic pointer is narrowed to an LDS address (its low 32 bits) and
// read with an LDS instruction, where the compiler cannot see the pointer's
// origin (a caller that is not inlined into the kernel) and would otherwise
// emit a flat load.
template <bool LOCAL>
__device__ __forceinline__ float4 ld_obs(const float4 *p) {
    if constexpr (LOCAL) {
        typedef float f4v __attribute__((ext_vector_type(4)));
        typedef const __attribute__((address_space(3))) f4v local_f4v;
        const f4v v = *reinterpret_cast<local_f4v *>((uint32_t)(uintptr_t)p);
        return make_float4(v.x, v.y, v.z, v.w);
    } else {
        return *p;
    }
}

// ---- broad phase -----------------------------------------------------------
// The poses of one wave lie close together (one edge, or neighbouring
// sub-edges of a chain), so a robot sphere's 64 positions fit a small ball.
// Before any exact test the wave forms that ball and tests it against 64
// obstacles at once, one obstacle per lane; the ballot is the list of
// obstacles any lane can touch.  The exact tests then run over that list
// alone, with scalar control flow.  Measured against a cull and a branch per
// sphere and obstacle (the form before; a free 64-pose Panda pass took 9.4k
// VALU instructions and 975 branches, and a wave alone on its SIMD spent half
// its cycles waiting on ballot-to-branch chains): 1M C1 edges 17.5 -> 8.2 ms,
// 10k free Fetch edges 220 -> 95 us, 64 Panda edges 50 -> 26 us, an uneven
// batch of 128 problems 270 -> 219 ms, the same verdicts bit for bit.

// Largest value over the wave (unsigned order), on every lane.  All 64 lanes
// must be active.
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
#define PRRTC_DPP_MAX(CTRL, ROWS)                                                                        \
    {                                                                                                    \
        const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);     \
        v = v > o ? v : o;                                                                               \
    }
    PRRTC_DPP_MAX(0x111, 0xf)   // row_shr:1, 2, 4, 8: lane 15 of a row holds the row's
    PRRTC_DPP_MAX(0x112, 0xf)
    PRRTC_DPP_MAX(0x114, 0xf)
    PRRTC_DPP_MAX(0x118, 0xf)
    PRRTC_DPP_MAX(0x142, 0xa)   // row_bcast:15 into rows 1 and 3
    PRRTC_DPP_MAX(0x143, 0xc)   // row_bcast:31 into rows 2 and 3
#undef PRRTC_DPP_MAX
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

__device__ __forceinline__ float lane_value(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// A ball that holds one point per live lane; the same on every lane.
struct WaveBall {
    float x, y, z, r;
};

__host__ __device__ __forceinline__ float padded_root(float d2) {
#pragma clang fp contract(off)
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_sqrtf(d2) * (1.0f + 0x1p-16f);
#else
    return sqrtf(d2) * (1.0f + 0x1p-16f);
#endif
}

// Centre of the ball: midway between the first and the last live lane's
// point (the ends of the wave's stretch of the path).
__device__ __forceinline__ WaveBall ball_centre(float x, float y, float z, uint64_t live) {
#pragma clang fp contract(off)
    const int a = __builtin_ctzll(live), b = 63 - __builtin_clzll(live);
    return WaveBall{0.5f * (lane_value(x, a) + lane_value(x, b)), 0.5f * (lane_value(y, a) + lane_value(y, b)),
                    0.5f * (lane_value(z, a) + lane_value(z, b)), 0.0f};
}

// Radius from the live lanes' squared distances: padded by 2^-16 relative,
// far above the rounding of the distances and of the raw square root (1
// ulp).  The maximum is taken over the bit patterns, where a NaN is above
// every number: a lane without a position then makes the radius NaN, and a
// NaN ball is near every obstacle (in_reach).
__device__ __forceinline__ float ball_radius(float d2, bool live) {
#pragma clang fp contract(off)
    const uint32_t m = wave_max(live ? (uint32_t)__float_as_int(d2) : 0u);
    return padded_root(__int_as_float((int)m));
}

// Point (x, y, z) of every live lane in one ball (`live`: the ballot of the
// live lanes, not empty).  All 64 lanes call it.
__device__ __forceinline__ WaveBall wave_ball(float x, float y, float z, bool on, uint64_t live) {
#pragma clang fp contract(off)
    WaveBall c = ball_centre(x, y, z, live);
    c.r = ball_radius(sq3(x - c.x, y - c.y, z - c.z), on);
    return c;
}

__host__ __device__ __forceinline__ float sphere_ball_radius(float r) {
#pragma clang fp contract(off)
    return fmaf(fabsf(r), 1.0f + 0x1p-16f, 1e-3f);
}

// One obstacle's ball on each lane: obstacle i of the scene.  A sphere's is
// padded like the others (2^-16 relative, 1 mm).
template <bool LOCAL>
__device__ __forceinline__ float4 obstacle_ball(const Obstacles &o, int i) {
#pragma clang fp contract(off)
    const bool s = i < o.n_sph;
    float4 b = ld_obs<LOCAL>(s ? o.sph + i : o.ball + (i - o.n_sph));
    if (s) b.w = sphere_ball_radius(b.w);
    return b;
}

// Whether anything within `reach` of the ball's centre can touch the
// obstacle ball `b`.  Both radii are padded, so an obstacle out of reach is
// at least about 1 mm from every live lane's sphere: its exact test would be
// positive, and skipping it cannot change a verdict.  NaN counts as in reach.
__host__ __device__ __forceinline__ bool in_reach(const float4 &b, const WaveBall &c, float reach) {
#pragma clang fp contract(off)
    const float rb = reach + b.w;
    return !(sq3(b.x - c.x, b.y - c.y, b.z - c.z) > rb * rb);
}

// ---- exact tests -----------------------------------------------------------
// The reference's squared forms (utils.cuh:58-208): value < 0 means
// collision.  Rounding is pinned: every multiply-add is an explicit fmaf in a
// fixed association (and contraction is off), so the CPU oracle can reproduce
// each verdict bit for bit in its "fused" mode.

__host__ __device__ __forceinline__ float sphere_test(const float4 &s, float x, float y, float z, float r) {   // utils.cuh:58-81
#pragma clang fp contract(off)
    const float rs = s.w + r;
    return fmaf(-rs, rs, sq3(s.x - x, s.y - y, s.z - z));
}
__host__ __device__ __forceinline__ float capsule_test(const float4 &p, const float4 &v, float x, float y, float z,
                                              float r) {                                                // utils.cuh:113-126
#pragma clang fp contract(off)
    const float dot = fmaf(x - p.x, v.x, fmaf(y - p.y, v.y, (z - p.z) * v.z));
    const float cdf = fmaxf(fminf(dot * v.w, 1.0f), 0.0f);
    const float rs = r + p.w;
    return fmaf(-rs, rs, sq3(x - fmaf(v.x, cdf, p.x), y - fmaf(v.y, cdf, p.y), z - fmaf(v.z, cdf, p.z)));
}
__host__ __device__ __forceinline__ float z_capsule_test(const float4 &p, const float4 &v, float x, float y, float z,
                                                float r) {                                              // utils.cuh:135-148
#pragma clang fp contract(off)
    const float dot = (z - p.z) * v.z;
    const float cdf = fmaxf(fminf(dot * v.w, 1.0f), 0.0f);
    const float rs = r + p.w;
    return fmaf(-rs, rs, sq3(x - p.x, y - p.y, z - fmaf(v.z, cdf, p.z)));
}
__host__ __device__ __forceinline__ float cuboid_test(const float4 &c, const float4 &a1, const float4 &a2, const float4 &a3,
                                             float x, float y, float z, float r) {                      // utils.cuh:158-175
#pragma clang fp contract(off)
    const float xs = x - c.x, ys = y - c.y, zs = z - c.z;
    const float d1 = fmaxf(0.0f, fabsf(fmaf(a1.x, xs, fmaf(a1.y, ys, a1.z * zs))) - c.w);
    const float d2 = fmaxf(0.0f, fabsf(fmaf(a2.x, xs, fmaf(a2.y, ys, a2.z * zs))) - a1.w);
    const float d3 = fmaxf(0.0f, fabsf(fmaf(a3.x, xs, fmaf(a3.y, ys, a3.z * zs))) - a2.w);
    return fmaf(-r, r, sq3(d1, d2, d3));
}
__host__ __device__ __forceinline__ float z_cuboid_test(const float4 &c, const float4 &a1, const float4 &a2, float x, float y,
                                               float z, float r) {                                      // utils.cuh:184-201
#pragma clang fp contract(off)
    const float xs = x - c.x, ys = y - c.y, zs = z - c.z;
    const float d1 = fmaxf(0.0f, fabsf(fmaf(a1.x, xs, a1.y * ys)) - c.w);
    const float d2 = fmaxf(0.0f, fabsf(fmaf(a2.x, xs, a2.y * ys)) - a1.w);
    const float d3 = fmaxf(0.0f, fabsf(zs) - a2.w);
    return fmaf(-r, r, sq3(d1, d2, d3));
}

// Smallest test value of obstacle i (wave-uniform) against N spheres per
// lane, lowered into m[n] (ANY: into m[0], for callers that want only
// whether some sphere hits).  A NaN test value is dropped by fminf as it
// would fail `< 0`.  far(n, ball) says (wave-uniformly) that sphere n is out
// of the obstacle's reach on every lane; the obstacle's rows are read once
// for all N.  ASK_ALL: asking costs no vector instruction, so it is asked for
// spheres and z-capsules too, whose tests are as cheap as a cull.
template <int N, bool LOCAL, bool ANY, bool ASK_ALL, class Far>
__device__ __forceinline__ void test_obstacle(const Obstacles &o, int i, const float *x, const float *y,
                                              const float *z, const float *r, float *m, Far far) {
#pragma clang fp contract(off)
    auto each = [&](auto cheap, auto test) {
#pragma unroll
        for (int n = 0; n < N; n++) {
            if ((ASK_ALL || !cheap.value) && far(n)) continue;
            m[ANY ? 0 : n] = fminf(m[ANY ? 0 : n], test(x[n], y[n], z[n], r[n]));
        }
    };
    if (i < o.n_sph) {
        const float4 s = ld_obs<LOCAL>(o.sph + i);
        each(std::true_type{}, [&](float a, float b, float c, float d) { return sphere_test(s, a, b, c, d); });
        return;
    }
    i -= o.n_sph;
    if (i < o.n_cap) {
        const float4 p = ld_obs<LOCAL>(o.cap + 2 * i), v = ld_obs<LOCAL>(o.cap + 2 * i + 1);
        each(std::false_type{}, [&](float a, float b, float c, float d) { return capsule_test(p, v, a, b, c, d); });
        return;
    }
    i -= o.n_cap;
    if (i < o.n_zcap) {
        const float4 p = ld_obs<LOCAL>(o.zcap + 2 * i), v = ld_obs<LOCAL>(o.zcap + 2 * i + 1);
        each(std::true_type{}, [&](float a, float b, float c, float d) { return z_capsule_test(p, v, a, b, c, d); });
        return;
    }
    i -= o.n_zcap;
    if (i < o.n_cub) {
        const float4 p = ld_obs<LOCAL>(o.cub + 4 * i), a1 = ld_obs<LOCAL>(o.cub + 4 * i + 1),
                     a2 = ld_obs<LOCAL>(o.cub + 4 * i + 2), a3 = ld_obs<LOCAL>(o.cub + 4 * i + 3);
        each(std::false_type{}, [&](float a, float b, float c, float d) { return cuboid_test(p, a1, a2, a3, a, b, c, d); });
        return;
    }
    i -= o.n_cub;
    const float4 p = ld_obs<LOCAL>(o.zcub + 4 * i), a1 = ld_obs<LOCAL>(o.zcub + 4 * i + 1),
                 a2 = ld_obs<LOCAL>(o.zcub + 4 * i + 2);
    each(std::false_type{}, [&](float a, float b, float c, float d) { return z_cuboid_test(p, a1, a2, a, b, c, d); });
}

// sphere_environment_in_collision (utils.cuh:211-242) for N spheres per
// lane, whose answer is wanted sphere by sphere: hit[n] on each live lane.
// All 64 lanes call it; `on` marks the live ones (at least one).  The ball of
// sphere n's positions is left on lane k0 + n of `balls`.
template <int N, bool LOCAL>
__device__ __forceinline__ void env_hits(const Obstacles &o, Share sh, const float (&x)[N], const float (&y)[N],
                                         const float (&z)[N], const float (&r)[N], bool on, bool (&hit)[N],
                                         int k0, WaveBall &balls) {
#pragma clang fp contract(off)
    const uint64_t live = ballot(on);
    const int lane = threadIdx.x & (kWave - 1);
    const int mine = (o.count() - sh.part + (1 << sh.shift) - 1) >> sh.shift;   // obstacles of the share
    float m[N];
#pragma unroll
    for (int n = 0; n < N; n++) m[n] = __builtin_huge_valf();
    int base = 0;
    do {   // at least once: the balls are wanted in an empty scene too
        const int j = base + lane;
        const bool have = j < mine;
        float4 b = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (mine > 0) b = obstacle_ball<LOCAL>(o, have ? (j << sh.shift) + sh.part : 0);
        uint64_t near[N];
#pragma unroll
        for (int n = 0; n < N; n++) {
            const WaveBall c = wave_ball(x[n], y[n], z[n], on, live);
            near[n] = ballot(have && in_reach(b, c, c.r + r[n]));
            int ln = lane;
            asm volatile("" : "+v"(ln));   // compared here: kept across the edge loop, a mask per gate spills SGPRs
            if (ln == k0 + n) balls = c;
        }
        // obstacle by obstacle, each against the spheres that list it
        uint64_t w = 0;
#pragma unroll
        for (int n = 0; n < N; n++) w |= near[n];
        for (; w; w &= w - 1) {
            const int bit = __builtin_ctzll(w);
            const int i = __builtin_amdgcn_readfirstlane(((base + bit) << sh.shift) + sh.part);
            test_obstacle<N, LOCAL, false, true>(o, i, x, y, z, r, m, [&](int n) { return !((near[n] >> bit) & 1); });
        }
        base += kWave;
    } while (base < mine);
#pragma unroll
    for (int n = 0; n < N; n++) hit[n] = m[n] < 0.0f;
}

// The same for poses that have nothing to do with each other (SpreadCtx):
// their balls would rule out little, so every obstacle is tested in turn, a
// capsule or cuboid unless it is out of a sphere's reach on every live lane.
template <int N, bool LOCAL>
__device__ __forceinline__ void env_hits_each(const Obstacles &o, const float (&x)[N], const float (&y)[N],
                                              const float (&z)[N], const float (&r)[N], bool on, bool (&hit)[N]) {
#pragma clang fp contract(off)
    float m[N];
#pragma unroll
    for (int n = 0; n < N; n++) m[n] = __builtin_huge_valf();
    auto far = [&](const float4 &b, int n) {   // on every active lane
        const float rb = r[n] + b.w;
        return ballot(!(sq3(x[n] - b.x, y[n] - b.y, z[n] - b.z) > rb * rb)) == 0;
    };
    if (on) {
        for (int i = 0; i < o.n_sph; i++) {
            const float4 s = ld_obs<LOCAL>(o.sph + i);
#pragma unroll
            for (int n = 0; n < N; n++) m[n] = fminf(m[n], sphere_test(s, x[n], y[n], z[n], r[n]));
        }
        for (int i = 0; i < o.n_cap; i++) {
            const float4 p = ld_obs<LOCAL>(o.cap + 2 * i), v = ld_obs<LOCAL>(o.cap + 2 * i + 1),
                         b = ld_obs<LOCAL>(o.ball + i);
#pragma unroll
            for (int n = 0; n < N; n++) {
                if (far(b, n)) continue;
                m[n] = fminf(m[n], capsule_test(p, v, x[n], y[n], z[n], r[n]));
            }
        }
        for (int i = 0; i < o.n_zcap; i++) {
            const float4 p = ld_obs<LOCAL>(o.zcap + 2 * i), v = ld_obs<LOCAL>(o.zcap + 2 * i + 1);
#pragma unroll
            for (int n = 0; n < N; n++) m[n] = fminf(m[n], z_capsule_test(p, v, x[n], y[n], z[n], r[n]));
        }
        for (int i = 0; i < o.n_cub; i++) {
            const float4 p = ld_obs<LOCAL>(o.cub + 4 * i), a1 = ld_obs<LOCAL>(o.cub + 4 * i + 1),
                         a2 = ld_obs<LOCAL>(o.cub + 4 * i + 2), a3 = ld_obs<LOCAL>(o.cub + 4 * i + 3);
            const float4 b = make_float4(p.x, p.y, p.z, a3.w);
#pragma unroll
            for (int n = 0; n < N; n++) {
                if (far(b, n)) continue;
                m[n] = fminf(m[n], cuboid_test(p, a1, a2, a3, x[n], y[n], z[n], r[n]));
            }
        }
        for (int i = 0; i < o.n_zcub; i++) {
            const float4 p = ld_obs<LOCAL>(o.zcub + 4 * i), a1 = ld_obs<LOCAL>(o.zcub + 4 * i + 1),
                         a2 = ld_obs<LOCAL>(o.zcub + 4 * i + 2);
            const float4 b = make_float4(p.x, p.y, p.z, ld_obs<LOCAL>(o.zcub + 4 * i + 3).w);
#pragma unroll
            for (int n = 0; n < N; n++) {
                if (far(b, n)) continue;
                m[n] = fminf(m[n], z_cuboid_test(p, a1, a2, x[n], y[n], z[n], r[n]));
            }
        }
    }
#pragma unroll
    for (int n = 0; n < N; n++) hit[n] = m[n] < 0.0f;
}

// Whether any of N spheres (the leaves of one link) hits an obstacle, on each
// live lane.  The spheres of every lane lie in one ball about `c`, `reach`
// its radius.  One running minimum serves the group (some value < 0 iff their
// minimum is).  EARLY: the wave leaves once every live lane has a hit.
// skip(ball) says (wave-uniformly) that an obstacle on the list is out of the
// whole group's reach all the same.
template <int N, bool EARLY, bool LOCAL, class Skip>
__device__ __forceinline__ bool env_group(const Obstacles &o, Share sh, const float (&x)[N], const float (&y)[N],
                                          const float (&z)[N], const float (&r)[N], bool on, const WaveBall &c,
                                          float reach, Skip skip) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & (kWave - 1);
    const int mine = (o.count() - sh.part + (1 << sh.shift) - 1) >> sh.shift;
    float m[1] = {__builtin_huge_valf()};
    for (int base = 0; base < mine; base += kWave) {
        const int j = base + lane;
        const bool have = j < mine;
        const float4 b = obstacle_ball<LOCAL>(o, have ? (j << sh.shift) + sh.part : 0);
        for (uint64_t w = ballot(have && in_reach(b, c, reach)); w; w &= w - 1) {
            const int i = __builtin_amdgcn_readfirstlane(((base + __builtin_ctzll(w)) << sh.shift) + sh.part);
            // of a link's spheres near an obstacle most are out of its reach
            // on every lane; the exact test costs three times this one
            const float4 ob = obstacle_ball<LOCAL>(o, i);
            if (skip(ob)) continue;
            test_obstacle<N, LOCAL, true, false>(o, i, x, y, z, r, m, [&](int n) {
                const float rb = r[n] + ob.w;
                return ballot(!(sq3(x[n] - ob.x, y[n] - ob.y, z[n] - ob.z) > rb * rb)) == 0;
            });
            if (EARLY && ballot(on && !(m[0] < 0.0f)) == 0) return true;
        }
    }
    return m[0] < 0.0f;
}

// env_group for spheres without a bound of their own: the ball is taken
// about the first sphere's stretch and holds all of them.
template <int N, bool EARLY, bool LOCAL>
__device__ __forceinline__ bool env_leaves(const Obstacles &o, Share sh, const float (&x)[N], const float (&y)[N],
                                           const float (&z)[N], const float (&r)[N], bool on) {
#pragma clang fp contract(off)
    WaveBall c = ball_centre(x[0], y[0], z[0], ballot(on));
    uint32_t d = 0;
    float rmax = 0.0f;
#pragma unroll
    for (int n = 0; n < N; n++) {
        // bit patterns of non-negative floats order like the floats, a NaN above all
        const uint32_t e = (uint32_t)__float_as_int(sq3(x[n] - c.x, y[n] - c.y, z[n] - c.z));
        d = e > d ? e : d;
        rmax = fmaxf(rmax, r[n]);
    }
    c.r = ball_radius(__int_as_float((int)d), on);
    return env_group<N, EARLY, LOCAL>(o, sh, x, y, z, r, on, c, c.r + rmax, [](const float4 &) { return false; });
}

// env_group for spheres that lie in the ball (gx, gy, gz; gr) on every lane
// -- the leaves of one link, bounded about the link's gate centre with a
// 1 mm pad by the generator.  SPREAD: the lanes' balls lie far apart, so the
// ball around them lists most obstacles; each is asked of the lanes' own first.
template <int N, bool EARLY, bool LOCAL, bool SPREAD = false>
__device__ __forceinline__ bool env_leaves_bounded(const Obstacles &o, Share sh, const float (&x)[N],
                                                   const float (&y)[N], const float (&z)[N], const float (&r)[N],
                                                   bool on, float gx, float gy, float gz, float gr) {
#pragma clang fp contract(off)
    const WaveBall c = wave_ball(gx, gy, gz, on, ballot(on));
    return env_group<N, EARLY, LOCAL>(o, sh, x, y, z, r, on, c, c.r + gr, [&](const float4 &b) {
        return SPREAD && ballot(on && in_reach(b, WaveBall{gx, gy, gz, 0.0f}, gr)) == 0;
    });
}

// sphere_sphere_self_collision (utils.cuh:83-86) with the radius sum folded.
__device__ __forceinline__ bool self_hit(float ax, float ay, float az, float bx, float by, float bz, float rs) {
#pragma clang fp contract(off)
    return fmaf(-rs, rs, sq3(ax - bx, ay - by, az - bz)) < 0.0f;
}

// Self-collision groups by the same balls.  A group is a pair of gate spheres
// (a link's each); `pairs` packs one group per word: the gates' numbers and
// the sum of their radii, padded and rounded up to binary16 by the
// generator.  With the ball of gate k's positions on lane k, every lane takes
// one group: when the two balls stay apart by more than the radii, no live
// lane's gates touch and the group needs no test at all.  (A gate test costs
// some 30 instructions and a branch, and Baxter has 355; here 64 groups cost
// as much as one.  30k Baxter edges 542 -> 284 us, an uneven batch of 128
// problems 219 -> 163 ms, a served burst 105 -> 63 ms.)  near[w] gets the
// groups 64 w .. 64 w + 63 that do, of those whose number is sh.part mod
// 2^sh.shift (the wave's own).
// Words of 64 for the robot that has the most groups; a robot's check touches
// the words of its own only.
constexpr int kSelfWords = (std::max({gen::panda::SELF_GROUPS, gen::fetch::SELF_GROUPS, gen::baxter::SELF_GROUPS,
                                      gen::ur5::SELF_GROUPS}) + 63) / 64;

template <int NS>
__device__ __forceinline__ void self_groups_own(Share sh, uint64_t (&near)[kSelfWords]) {
    static_assert(NS <= 64 * kSelfWords, "a robot is missing in kSelfWords");
    const int lane = threadIdx.x & (kWave - 1);
    const uint64_t own = ballot((lane & ((1 << sh.shift) - 1)) == sh.part);   // 64 is a multiple of 2^shift
#pragma unroll
    for (int w = 0; w < (NS + 63) / 64; w++) near[w] = own;
}

template <int NS>
__device__ __forceinline__ void self_groups_near(Share sh, const uint32_t *pairs, const WaveBall &balls,
                                                 uint64_t (&near)[kSelfWords]) {
#pragma clang fp contract(off)
    static_assert(NS <= 64 * kSelfWords, "a robot is missing in kSelfWords");
    const int lane = threadIdx.x & (kWave - 1);
    const bool own = (lane & ((1 << sh.shift) - 1)) == sh.part;
    auto from = [](float v, uint32_t k) {
        return __int_as_float(__builtin_amdgcn_ds_bpermute((int)(k << 2), __float_as_int(v)));
    };
    uint32_t p[(NS + 63) / 64];
#pragma unroll
    for (int w = 0; w < (NS + 63) / 64; w++) p[w] = pairs[64 * w + lane < NS ? 64 * w + lane : NS - 1];
#pragma unroll
    for (int w = 0; w < (NS + 63) / 64; w++) {
#pragma clang fp contract(off)
        const uint32_t a = p[w] & 0xff, b = (p[w] >> 8) & 0xff;
        const float dx = from(balls.x, a) - from(balls.x, b), dy = from(balls.y, a) - from(balls.y, b),
                    dz = from(balls.z, a) - from(balls.z, b);
        const uint16_t h = (uint16_t)(p[w] >> 16);
        const float reach = (from(balls.r, a) + from(balls.r, b)) + (float)__builtin_bit_cast(_Float16, h);
        near[w] = ballot(own && 64 * w + lane < NS && !(sq3(dx, dy, dz) > reach * reach));
    }
}

// ---------------------------------------------------------------------------
// Check context driven by the generated robot code, for a pass of up to 64
// poses (one per lane).
//
// Path mode (independent == false): `key` orders the lanes' poses into groups
// (sub-edges, non-decreasing with the lane index).  Lanes whose key is >= the
// key of the lowest colliding lane can no longer change the answer, so they
// stop; the wavefront leaves once no lane is live.  With one key for the
// whole wave (one edge) the first collision anywhere ends the pass.
//
// Pose mode (independent == true): every lane is its own question; a lane
// stops only on its own collision.
struct CheckCtx {
    Obstacles obs;
    bool coll;
    bool dead;
    bool independent;
    int key;
    WaveBall balls;                   // lane k: the ball of gate k's positions
    uint64_t near[kSelfWords];        // self-collision groups to test

    __device__ __forceinline__ bool live() const { return !coll && !dead; }
    __device__ __forceinline__ bool any(bool p) const { return ballot(p) != 0; }
    // Self-collision group j (numbered in check order) is this wave's to
    // test: its own, and not ruled out by the gates' balls.
    __device__ __forceinline__ bool mine(int j) const { return (near[j >> 6] >> (j & 63)) & 1; }
    // Any of the groups j .. j + n - 1 (of one 64-group word).
    __device__ __forceinline__ bool mine_any(int j, int n) const {
        return ((near[j >> 6] >> (j & 63)) & ((1ull << n) - 1)) != 0;
    }
    template <int NS>
    __device__ __forceinline__ void self_own() { self_groups_own<NS>(Share{}, near); }
    template <int NS>
    __device__ __forceinline__ void self_near(const uint32_t *pairs) {
        self_groups_near<NS>(Share{}, pairs, balls, near);
    }
    // The ball of a gate that never moves, at number k.
    __device__ __forceinline__ void fixed_gate(int k, float x, float y, float z) {
        if ((int)(threadIdx.x & (kWave - 1)) == k) balls = WaveBall{x, y, z, 0.0f};
    }
    // Gate spheres k0 .. k0 + N - 1 against the obstacles, hit[n] on each
    // live lane; called by the whole wave while some lane is live.
    template <int N>
    __device__ __forceinline__ void env_gates(int k0, const float (&x)[N], const float (&y)[N], const float (&z)[N],
                                              const float (&r)[N], bool (&hit)[N]) {
        env_hits<N, false>(obs, Share{}, x, y, z, r, live(), hit, k0, balls);
    }
    // Whether any of the N spheres of a leaf group hits an obstacle, on the
    // lanes with `on` (at least one); called by the whole wave.
    template <int N, bool EARLY>
    __device__ __forceinline__ bool env_any(const float (&x)[N], const float (&y)[N], const float (&z)[N],
                                            const float (&r)[N], bool on) const {
        return env_leaves<N, EARLY, false>(obs, Share{}, x, y, z, r, on);
    }
    // The same for N spheres that lie inside the ball (gx, gy, gz; gr) on
    // every lane.
    template <int N, bool EARLY>
    __device__ __forceinline__ bool env_any_bounded(const float (&x)[N], const float (&y)[N], const float (&z)[N],
                                                    const float (&r)[N], bool on, float gx, float gy, float gz,
                                                    float gr) const {
        return env_leaves_bounded<N, EARLY, false>(obs, Share{}, x, y, z, r, on, gx, gy, gz, gr);
    }
    __device__ __forceinline__ bool self(float ax, float ay, float az, float bx, float by, float bz, float rs) const {
        return self_hit(ax, ay, az, bx, by, bz, rs);
    }
    __device__ __forceinline__ bool near_point(float ax, float ay, float az, float bx, float by, float bz,
                                               float d2) const {
#pragma clang fp contract(off)
        return !(sq3(ax - bx, ay - by, az - bz) > d2);
    }
    __device__ __forceinline__ void hit() { coll = true; }
    // Gate bits of this lane's pose after the gate pass.  A context whose
    // waves split the obstacle tables ORs them across its waves; here every
    // wave sees every obstacle, so there is nothing to share.
    __device__ __forceinline__ void share_gates(uint64_t &) const {}
    __device__ __forceinline__ bool stop() {
        if (!independent) {
            const uint64_t cm = ballot(coll);
            if (cm) {
                const int l = __builtin_ctzll(cm);
                const int stop_key = __builtin_amdgcn_readlane(key, l);
                dead = dead || key >= stop_key;
            }
        }
        return ballot(!coll && !dead) == 0;
    }
};

// Check context of a pass of poses that have nothing to do with each other:
// no balls over the wave, neither for the gates nor for the self-collision
// groups.
struct SpreadCtx : CheckCtx {
    template <int N>
    __device__ __forceinline__ void env_gates(int, const float (&x)[N], const float (&y)[N], const float (&z)[N],
                                              const float (&r)[N], bool (&hit)[N]) const {
        env_hits_each<N, false>(obs, x, y, z, r, live(), hit);
    }
    __device__ __forceinline__ void fixed_gate(int, float, float, float) {}
    template <int NS>
    __device__ __forceinline__ void self_near(const uint32_t *) { self_groups_own<NS>(Share{}, near); }
    template <int N, bool EARLY>
    __device__ __forceinline__ bool env_any_bounded(const float (&x)[N], const float (&y)[N], const float (&z)[N],
                                                    const float (&r)[N], bool on, float gx, float gy, float gz,
                                                    float gr) const {
        return env_leaves_bounded<N, EARLY, false, true>(obs, Share{}, x, y, z, r, on, gx, gy, gz, gr);
    }
};

// ---------------------------------------------------------------------------
// robots

struct SphereRobot {     // Robots.hh:190-237; fkcc<Sphere>, utils.cuh:330-334
    static constexpr int DOF = 3;
    static constexpr int NSPHERES = 1;
    static constexpr float kSpread = 4.0f;   // its positions lie in a cube of side 10
    __host__ __device__ static constexpr float lower(int) { return -5.0f; }
    __host__ __device__ static constexpr float span(int) { return 10.0f; }
    template <class Ctx>
    __device__ __forceinline__ static void check(const float *q, Ctx &ctx) {
        const float x[1] = {q[0]}, y[1] = {q[1]}, z[1] = {q[2]}, r[1] = {1.0f};
        bool h[1];
        if (ctx.any(ctx.live())) {
            ctx.template env_gates<1>(0, x, y, z, r, h);
            if (ctx.live() && h[0]) ctx.hit();
        }
        ctx.stop();
    }
    __device__ __forceinline__ static void fk_spheres(const float *q, float *out) {
        out[0] = q[0]; out[1] = q[1]; out[2] = q[2];
    }
};

// kSpread (see launch_check): joint distance at which poses count as unrelated
#define PRRTC_GEN_ROBOT(NAME, NS, SPREAD)                                                      \
    struct NAME##Robot {                                                                       \
        static constexpr float kSpread = SPREAD;                                               \
        static constexpr int DOF = gen::NS::DOF;                                               \
        static constexpr int NSPHERES = gen::NS::NSPHERES;                                     \
        __host__ __device__ static constexpr float lower(int i) { return gen::NS::lower(i); } \
        __host__ __device__ static constexpr float span(int i) { return gen::NS::span(i); }   \
        template <class Ctx>                                                                   \
        __device__ __forceinline__ static void check(const float *q, Ctx &ctx) {               \
            gen::NS::check(q, ctx);                                                            \
        }                                                                                      \
        __device__ __forceinline__ static void fk_spheres(const float *q, float *out) {       \
            gen::NS::fk_spheres(q, out);                                                       \
        }                                                                                      \
    };
PRRTC_GEN_ROBOT(Panda, panda, 2.2f)
PRRTC_GEN_ROBOT(Fetch, fetch, 1.6f)
PRRTC_GEN_ROBOT(Baxter, baxter, 4.2f)
PRRTC_GEN_ROBOT(Ur5, ur5, 3.5f)
#undef PRRTC_GEN_ROBOT

// Every robot the library is built for, as X(id, struct): the one list the
// dispatch switches expand.  A robot from the model compiler is one more
// line here, its generated header above and its id in include/prrtc.h.
#define PRRTC_FOR_EACH_ROBOT(X)        \
    X(PRRTC_ROBOT_SPHERE, SphereRobot) \
    X(PRRTC_ROBOT_PANDA, PandaRobot)   \
    X(PRRTC_ROBOT_FETCH, FetchRobot)   \
    X(PRRTC_ROBOT_BAXTER, BaxterRobot) \
    X(PRRTC_ROBOT_UR5, Ur5Robot)
constexpr int kNumRobots = 5;   // ids 0 .. kNumRobots - 1
constexpr bool robot_ids_dense() {
    int n = 0, top = -1;
#define PRRTC_COUNT_ROBOT(ID, R) n++; top = ID > top ? ID : top;
    PRRTC_FOR_EACH_ROBOT(PRRTC_COUNT_ROBOT)
#undef PRRTC_COUNT_ROBOT
    return n == kNumRobots && top == kNumRobots - 1;
}
static_assert(robot_ids_dense(), "PRRTC_FOR_EACH_ROBOT lists ids 0 .. kNumRobots - 1");
// The type of a robot in a call expanded from PRRTC_FOR_EACH_ROBOT.
template <class R> struct RobotTag { using type = R; };

}  // namespace prrtc
