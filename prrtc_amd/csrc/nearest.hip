// Nearest-node search over SoA trees on gfx950: the planner's scan
// (nearest<D>, planner_device.h) exposed for measurement and parity.
//
// Replaces the per-block tree scans of the reference planner
// (src/planning/pRRTC.cu:384-423 extend, 478-514 connect; distance at
// src/planning/utils.cuh:89-109): there each of the 128 threads of a block
// strides the AoS node array and a shared-memory reduction picks the minimum.
// Here one workgroup answers one query (k_nearest: its waves stride the
// tree's SoA columns in 1024-node chunks of float4 loads and reduce by lane
// shuffles and LDS), or several queries of one tree at once (k_nearest_tile:
// every node read serves all of them).  Ties go to the smaller index.
#include <hip/hip_runtime.h>

#include "host_common.h"
#include "planner_device.h"

namespace prrtc {

// Query k = t * qpt + j asks tree t (`trees + t * D * cap`) for the node
// nearest to queries[k]; idx[k] and dist2[k] receive the answer.
template <int D>
__global__ __launch_bounds__(kMaxTaskWaves * kWave) void k_nearest(const float *__restrict__ trees, int cap, int n,
                                                                    const float *__restrict__ queries, int qpt,
                                                                    int n_queries, int *__restrict__ idx,
                                                                    float *__restrict__ dist2) {
    __shared__ float red[2 * kMaxTaskWaves];
    const XcdRange range(n_queries);   // the queries of one tree are consecutive
    for (int k = range.first; k < range.end; k += range.stride) {
        const float *tree = trees + (size_t)(k / qpt) * D * cap;
        float q[D];
#pragma unroll
        for (int d = 0; d < D; d++) q[d] = queries[(size_t)k * D + d];
        float best;
        const int i = nearest<D>(tree, cap, n, q, best, red, team_workgroup());
        if (threadIdx.x == 0) {
            idx[k] = i;
            dist2[k] = best;
        }
    }
}

// Smallest value over the wave of non-negative floats (their bit patterns
// order alike); on every lane.  All 64 lanes must be active.
__device__ __forceinline__ float wave_min_nonneg(float v) {
    return __int_as_float((int)~wave_max(~(uint32_t)__float_as_int(v)));
}

// Q queries of one tree per workgroup.  Nodes lie 4 to a lane, 256 to a step
// (steps are dealt to the waves in turn), and each node's coordinates are
// read once for all Q queries, whose own coordinates sit in scalar registers.
// Against a query at a time, which streams the tree through L2 once per query
// (bound by L2: 64 trees of 50k nodes x 7, 64 queries each, 200 us), it is
// bound by the 2 D vector instructions per node and query.
//
// A wave keeps one best (distance, index) per query for all its lanes: a step
// costs a query the distances, the minimum of the lane's four and one
// compare; only a step that beats the wave's best (a handful of times per
// scan) finds the lane and the node.  Nodes are visited in increasing index
// order and a later equal distance does not replace, so the smaller index
// wins; a NaN distance never wins; the start is (+inf, 0) as in nearest<D>.
constexpr int kTileStep = 4 * kWave;
static_assert(kScanChunk % kTileStep == 0, "tree storage is whole steps");

template <int D, int Q>
__global__ __launch_bounds__(kMaxTaskWaves * kWave) void k_nearest_tile(const float *__restrict__ trees, int cap, int n,
                                                                         const float *__restrict__ queries, int qpt,
                                                                         int tiles, int n_tiles, int *__restrict__ idx,
                                                                         float *__restrict__ dist2) {
#pragma clang fp contract(off)
    __shared__ float red_d[kMaxTaskWaves][Q];
    __shared__ int red_i[kMaxTaskWaves][Q];
    const int lane = lane_id(), wave = wave_id(), waves = blockDim.x / kWave;
    const XcdRange range(n_tiles);
    for (int g = range.first; g < range.end; g += range.stride) {
        const int t = g / tiles, q0 = (g % tiles) * Q;   // tree, first query of the tile
        const int nq = min(Q, qpt - q0);
        const float *tree = trees + (size_t)t * D * cap;
        float q[Q][D];
#pragma unroll
        for (int j = 0; j < Q; j++) {
            // a short tile repeats its last query
            const float *src = queries + ((size_t)t * qpt + q0 + min(j, nq - 1)) * D;
#pragma unroll
            for (int d = 0; d < D; d++) q[j][d] = src[d];
        }
        float best[Q];
        int at[Q];
#pragma unroll
        for (int j = 0; j < Q; j++) { best[j] = __builtin_huge_valf(); at[j] = 0; }
        const int w0 = __builtin_amdgcn_readfirstlane(wave);
        for (int c = w0 * kTileStep; c < n; c += waves * kTileStep) {
            float4 v[D];
#pragma unroll
            for (int d = 0; d < D; d++)
                v[d] = reinterpret_cast<const float4 *>(tree + (size_t)d * cap + c)[lane];
            const int left = n - c - 4 * lane;   // the lane's nodes below n: min(4, left)
#pragma unroll
            for (int j = 0; j < Q; j++) {
                float a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int d = 0; d < D; d++) {
                    float diff = v[d].x - q[j][d];
                    a[0] = fmaf(diff, diff, a[0]);
                    diff = v[d].y - q[j][d];
                    a[1] = fmaf(diff, diff, a[1]);
                    diff = v[d].z - q[j][d];
                    a[2] = fmaf(diff, diff, a[2]);
                    diff = v[d].w - q[j][d];
                    a[3] = fmaf(diff, diff, a[3]);
                }
                if (c + kTileStep > n) {   // the last step: nodes from n on are not the tree's
#pragma unroll
                    for (int e = 0; e < 4; e++) a[e] = e < left ? a[e] : __builtin_huge_valf();
                }
                const float m = fminf(fminf(a[0], a[1]), fminf(a[2], a[3]));
                if (ballot(m < best[j]) == 0) continue;
                const float nb = wave_min_nonneg(m < best[j] ? m : best[j]);
                const int l = __builtin_ctzll(ballot(m == nb));   // the first lane that has it
                int e = 3;
#pragma unroll
                for (int k = 2; k >= 0; k--) e = lane_value(a[k], l) == nb ? k : e;
                best[j] = nb;
                at[j] = c + 4 * l + e;
            }
        }
        if (lane == 0) {
#pragma unroll
            for (int j = 0; j < Q; j++) { red_d[wave][j] = best[j]; red_i[wave][j] = at[j]; }
        }
        __syncthreads();
        if ((int)threadIdx.x < nq) {
            const int j = threadIdx.x;
            float b = red_d[0][j];
            int i = red_i[0][j];
            for (int w = 1; w < waves; w++) {
                const float ob = red_d[w][j];
                const int oi = red_i[w][j];
                if (ob < b || (ob == b && oi < i)) { b = ob; i = oi; }
            }
            idx[(size_t)t * qpt + q0 + j] = i;
            dist2[(size_t)t * qpt + q0 + j] = b;
        }
        __syncthreads();   // red is written again by the next tile
    }
}

template <int D, int Q>
static void launch_tile(const float *trees, int cap, int n, const float *queries, int qpt, int n_trees, int waves,
                        int *idx, float *dist2, hipStream_t s) {
    const int tiles = (qpt + Q - 1) / Q, n_tiles = n_trees * tiles;
    const int grid = std::max(1, std::min(n_tiles, num_cus() * 64));
    hipLaunchKernelGGL((k_nearest_tile<D, Q>), dim3(grid), dim3(waves * kWave), 0, s, trees, cap, n, queries, qpt,
                       tiles, n_tiles, idx, dist2);
    PRRTC_HIP(hipGetLastError());
}

template <int D>
static void launch_nearest(const float *trees, int cap, int n, const float *queries, int qpt, int n_trees,
                           int waves, int *idx, float *dist2, hipStream_t s) {
    const int n_queries = n_trees * qpt;
    // As many queries per workgroup as leave every CU two workgroups and a wave
    // for each SIMD, two where D is 3 and the shared reads save least: fewer
    // would idle part of the chip for longer than they save.  (64 trees of 50k
    // nodes, 64 queries each, one wave, D 7 and 8: 193 and 220 us a query at a
    // time; eight to a workgroup, half the SIMDs idle, 282 and 300; four, 174
    // and 184.  D 3: 90 us; four to a workgroup 147.)
    auto fills = [&](int q) {
        const long long tiles = (long long)n_trees * ((qpt + q - 1) / q);
        return qpt >= q && tiles >= 2ll * num_cus() && tiles * waves >= (D > 3 ? 4ll : 8ll) * num_cus();
    };
    // (a query's coordinates take D scalar registers: 8 of 14 do not fit)
    if constexpr (D <= 8) {
        if (fills(8)) return launch_tile<D, 8>(trees, cap, n, queries, qpt, n_trees, waves, idx, dist2, s);
    }
    if (fills(4)) return launch_tile<D, 4>(trees, cap, n, queries, qpt, n_trees, waves, idx, dist2, s);
    // A pair saves three of six reads a node where D is 3, which is no more
    // than a half-empty pair or a one-wave workgroup costs: 256 trees of 50k
    // nodes, 3 queries each, four waves, 32 us a query at a time, 36 in pairs;
    // 64 trees, 64 queries, one wave, 90 and 102; 8 trees, 128 queries, four
    // waves, 32 and 28.
    if (fills(2) && (D > 3 || (qpt % 2 == 0 && waves > 1)))
        return launch_tile<D, 2>(trees, cap, n, queries, qpt, n_trees, waves, idx, dist2, s);
    const int grid = std::max(1, std::min(n_queries, num_cus() * 64));
    hipLaunchKernelGGL(k_nearest<D>, dim3(grid), dim3(waves * kWave), 0, s, trees, cap, n, queries, qpt, n_queries,
                       idx, dist2);
    PRRTC_HIP(hipGetLastError());
}

}  // namespace prrtc

using namespace prrtc;

extern "C" int prrtc_nearest_async(int dof, const float *d_trees, int cap, int n_nodes, int n_trees,
                                   const float *d_queries, int queries_per_tree, int waves, int *d_idx,
                                   float *d_dist2, void *stream) {
    return guarded("prrtc_nearest_async", [&]() -> int {
        if ((dof != 3 && dof != 7 && dof != 8 && dof != 14) || n_trees < 0 || queries_per_tree < 0 ||
            n_nodes < 1 || cap < n_nodes || cap % kScanChunk != 0 || waves < 1 || waves > kMaxTaskWaves ||
            (n_trees > 0 && queries_per_tree > 0 && (!d_trees || !d_queries || !d_idx || !d_dist2))) {
            set_error("prrtc_nearest_async: invalid argument (dof 3/7/8/14, 1 <= n_nodes <= cap, cap a multiple "
                      "of %d, 1 <= waves <= %d)", kScanChunk, kMaxTaskWaves);
            return PRRTC_EINVAL;
        }
        const long long nq = (long long)n_trees * queries_per_tree;
        if (nq == 0) return PRRTC_OK;
        if (nq > INT32_MAX) {
            set_error("prrtc_nearest_async: too many queries");
            return PRRTC_EINVAL;
        }
        const hipStream_t s = static_cast<hipStream_t>(stream);
        switch (dof) {
            case 3: launch_nearest<3>(d_trees, cap, n_nodes, d_queries, queries_per_tree, n_trees, waves, d_idx,
                                      d_dist2, s); break;
            case 7: launch_nearest<7>(d_trees, cap, n_nodes, d_queries, queries_per_tree, n_trees, waves, d_idx,
                                      d_dist2, s); break;
            case 8: launch_nearest<8>(d_trees, cap, n_nodes, d_queries, queries_per_tree, n_trees, waves, d_idx,
                                      d_dist2, s); break;
            case 14: launch_nearest<14>(d_trees, cap, n_nodes, d_queries, queries_per_tree, n_trees, waves, d_idx,
                                        d_dist2, s); break;
        }
        return PRRTC_OK;
    });
}
