// Host build of the broad phase's arithmetic (device_common.h), for
// tests/test_reach.py.  Modes:
//   lds    a staged scene takes scene_lds_f4 float4, at most scene_lds_f4_most
//   reach  an obstacle whose ball is just out of a wave's reach hits none of
//          its positions; prints, for each kind of obstacle, how many were
//          tried and the least by which the gap between the surfaces exceeds
//          1 mm and half the relative pad (less the rounding of the coordinates)
//          args: log10 of the smallest and largest scale of the positions,
//          sign of the obstacles' radii
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

#include "../../prrtc_amd/csrc/host_common.h"

using namespace prrtc;

static int lds() {
    std::mt19937 rng(1);
    for (int t = 0; t < 2000; t++) {
        int n[5];
        for (int &c : n) c = rng() % 3 ? rng() % 200 : 0;
        const int f4 = scene_payload_f4(n[0], n[1], n[2], n[3], n[4]);
        const int balls = n[1] + n[2] + n[3] + n[4];   // what stage_scene appends
        const int asked = scene_lds_f4(n[0], n[1], n[2], n[3], n[4]);
        if (asked != f4 + balls || asked > scene_lds_f4_most(f4)) return 1;
    }
    return 0;
}

struct V {
    double x, y, z;
    V operator+(V o) const { return {x + o.x, y + o.y, z + o.z}; }
    V operator-(V o) const { return {x - o.x, y - o.y, z - o.z}; }
    V operator*(double s) const { return {x * s, y * s, z * s}; }
};
static double dot(V a, V b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
static double len(V a) { return std::sqrt(dot(a, a)); }
static V unit(V a) { return a * (1.0 / len(a)); }
static V cross(V a, V b) { return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x}; }
static float4 row(V a, double w) { return make_float4((float)a.x, (float)a.y, (float)a.z, (float)w); }

// One obstacle of the given kind, its bulk turned so that it comes closest
// along -u; kept as rows (as packed) and the ball the library gives it.
struct Obstacle {
    int kind;   // 0 sphere, 1 capsule, 2 z-capsule, 3 cuboid, 4 z-cuboid
    float4 r[4], ball;
    float test(float x, float y, float z, float rad) const {
        switch (kind) {
            case 0: return sphere_test(r[0], x, y, z, rad);
            case 1: return capsule_test(r[0], r[1], x, y, z, rad);
            case 2: return z_capsule_test(r[0], r[1], x, y, z, rad);
            case 3: return cuboid_test(r[0], r[1], r[2], r[3], x, y, z, rad);
            default: return z_cuboid_test(r[0], r[1], r[2], x, y, z, rad);
        }
    }
    // distance of a point to the obstacle's solid, in 64 bits
    double distance(V p) const {
        const V c{r[0].x, r[0].y, r[0].z};
        if (kind == 0) return len(p - c) - std::fabs(r[0].w);
        if (kind <= 2) {
            const V v{kind == 1 ? r[1].x : 0.0, kind == 1 ? r[1].y : 0.0, r[1].z};
            const double t = std::min(1.0, std::max(0.0, dot(p - c, v) / std::max(dot(v, v), 1e-300)));
            return len(p - (c + v * t)) - std::fabs(r[0].w);
        }
        const V d = p - c, a[3] = {{r[1].x, r[1].y, r[1].z}, {r[2].x, r[2].y, r[2].z},
                                   {kind == 3 ? r[3].x : 0.0, kind == 3 ? r[3].y : 0.0, kind == 3 ? r[3].z : 1.0}};
        const double h[3] = {r[0].w, r[1].w, r[2].w};
        double s = 0;
        for (int k = 0; k < 3; k++) {
            const double e = std::max(0.0, std::fabs(dot(a[k], d)) - h[k]);
            s += e * e;
        }
        return std::sqrt(s);
    }
};

// centre `at`, towards -u, size s (half-length, half-extents, radius)
static Obstacle make(int kind, V at, V u, double s, double radius, std::mt19937 &rng) {
    std::uniform_real_distribution<double> f(0.2, 1.0);
    Obstacle o;
    o.kind = kind;
    if (kind == 0) {
        o.r[0] = row(at, radius);
        o.ball = o.r[0];
        o.ball.w = sphere_ball_radius(o.r[0].w);
    } else if (kind <= 2) {
        const V half = kind == 1 ? u * s : V{0, 0, s};
        const V v = half * 2.0;
        o.r[0] = row(at - half, radius);
        o.r[1] = row(v, 0);
        o.r[1].w = 1.0f / sq3(o.r[1].x, o.r[1].y, o.r[1].z);
        o.ball = capsule_ball(o.r[0], o.r[1].x, o.r[1].y, o.r[1].z);
    } else {
        // a corner along -u: u = sum of axis_k * h_k / |h|
        const double h[3] = {s * f(rng), s * f(rng), s * f(rng)};
        V a[3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}};
        if (kind == 3) {   // turn (h / |h|) into u: reflect, then flip an axis to keep the hand
            const V w = unit(V{h[0], h[1], h[2]}) - u;
            if (len(w) > 1e-6) {
                const V n = unit(w);
                for (V &e : a) e = e - n * (2.0 * dot(n, e));
            }
        }
        o.r[0] = row(at, h[0]);
        o.r[1] = row(a[0], h[1]);
        o.r[2] = row(a[1], h[2]);
        // the cull radius as the library's pack makes it
        float scene[15] = {o.r[0].x, o.r[0].y, o.r[0].z, (float)a[0].x, (float)a[0].y, (float)a[0].z,
                           (float)a[1].x, (float)a[1].y, (float)a[1].z, (float)a[2].x, (float)a[2].y, (float)a[2].z,
                           (float)h[0], (float)h[1], (float)h[2]};
        const double R = std::sqrt((double)scene[12] * scene[12] + (double)scene[13] * scene[13] +
                                   (double)scene[14] * scene[14]);
        o.r[3] = row(a[2], (float)(R * (1.0 + 1.0 / 65536.0) + 1e-3));   // pinned by test_cuboid_cull_radius
        o.ball = o.r[0];
        o.ball.w = o.r[3].w;
    }
    return o;
}

static int reach(double lo, double hi, double sign) {
    std::mt19937 rng(7);
    std::normal_distribution<double> g(0, 1);
    std::uniform_real_distribution<double> f(0, 1);
    int used[5] = {};
    double worst[5] = {1e300, 1e300, 1e300, 1e300, 1e300};
    for (int t = 0; t < 20000; t++) {
        const int kind = t % 5;
        const double scale = std::pow(10.0, lo + (hi - lo) * f(rng));
        const V mid = V{g(rng), g(rng), g(rng)} * scale;
        const double spread = std::min(scale, 1.0) * std::pow(10.0, -4 * f(rng));
        float x[64], y[64], z[64];
        for (int l = 0; l < 64; l++) {
            x[l] = (float)(mid.x + spread * g(rng));
            y[l] = (float)(mid.y + spread * g(rng));
            z[l] = (float)(mid.z + spread * g(rng));
        }
        const float r = (float)std::pow(10.0, -2 + 1.5 * f(rng));
        // the ball as ball_centre and ball_radius form it
        WaveBall c{0.5f * (x[0] + x[63]), 0.5f * (y[0] + y[63]), 0.5f * (z[0] + z[63]), 0.0f};
        float d2 = 0.0f;
        int far = 0;
        for (int l = 0; l < 64; l++) {
            const float d = sq3(x[l] - c.x, y[l] - c.y, z[l] - c.z);
            if (d > d2) d2 = d, far = l;
        }
        c.r = padded_root(d2);
        const V centre{c.x, c.y, c.z};
        V u = V{x[far], y[far], z[far]} - centre;
        u = len(u) > 0 ? unit(u) : V{1, 0, 0};
        if (kind == 2) u = V{0, 0, u.z < 0 ? -1.0 : 1.0};
        const double size = std::pow(10.0, -2 + 2 * f(rng)), radius = sign * std::pow(10.0, -2 + 1.5 * f(rng));
        // the nearest place along u at which the library calls it out of reach
        double in = 0, out = 8.0 * (c.r + r + size + std::fabs(radius)) + 1e-5 * scale;
        std::mt19937 shape = rng;
        auto at = [&](double d) {
            std::mt19937 s = shape;
            return make(kind, centre + u * d, u, size, radius, s);
        };
        if (in_reach(at(out).ball, c, c.r + r)) continue;
        for (int k = 0; k < 60; k++) {
            const double d = 0.5 * (in + out);
            (in_reach(at(d).ball, c, c.r + r) ? in : out) = d;
        }
        const Obstacle o = at(out);
        used[kind]++;
        for (int l = 0; l < 64; l++) {
            if (o.test(x[l], y[l], z[l], r) < 0.0f) {
                std::printf("kind %d hits at scale %g, size %g, radius %g\n", kind, scale, size, radius);
                return 1;
            }
            const double gap = o.distance(V{x[l], y[l], z[l]}) - r;
            const double owed = 1e-3 + std::ldexp(c.r + o.ball.w, -17) - std::ldexp(len(V{o.r[0].x, o.r[0].y, o.r[0].z}), -22);
            worst[kind] = std::min(worst[kind], gap - owed);
        }
    }
    for (int k = 0; k < 5; k++) std::printf("%d %d %.6g\n", k, used[k], worst[k]);
    return 0;
}

int main(int argc, char **argv) {
    if (argc == 2 && !std::strcmp(argv[1], "lds")) return lds();
    if (argc == 5 && !std::strcmp(argv[1], "reach")) return reach(std::atof(argv[2]), std::atof(argv[3]), std::atof(argv[4]));
    return 2;
}
