// Generated by prrtc_amd/robots/gen_headers.py from ur5.json -- do not edit.
#pragma once

namespace prrtc::gen::ur5 {
constexpr int DOF = 6;
constexpr int NSPHERES = 29;
constexpr int SELF_GROUPS = 33;
__device__ __host__ constexpr float lower(int i) { constexpr float v[] = {-3.1415927410125732f, -3.1415927410125732f, -3.1415927410125732f, -3.1415927410125732f, -3.1415927410125732f, -3.1415927410125732f}; return v[i]; }
__device__ __host__ constexpr float span(int i) { constexpr float v[] = {6.2831854820251465f, 3.1415927410125732f, 6.2831854820251465f, 6.2831854820251465f, 6.2831854820251465f, 6.2831854820251465f}; return v[i]; }

#define PRRTC_FK_BODY \
    /* joint 0 (revolute, parent -1) */ \
    float s0, c0; sincosf(q[0], &s0, &c0); \
    const float R0_00 = c0; \
    const float R0_01 = -s0; \
    const float R0_10 = s0; \
    const float R0_11 = c0; \
    /* joint 1 (revolute, parent 0) */ \
    const float M1_00 = 6.123234262925839e-17f * R0_00; \
    const float M1_01 = -R0_00; \
    const float M1_10 = 6.123234262925839e-17f * R0_10; \
    const float M1_11 = -R0_10; \
    float s1, c1; sincosf(q[1], &s1, &c1); \
    const float R1_00 = c1 * M1_00 + s1 * M1_01; \
    const float R1_01 = c1 * M1_01 - s1 * M1_00; \
    const float R1_10 = c1 * M1_10 + s1 * M1_11; \
    const float R1_11 = c1 * M1_11 - s1 * M1_10; \
    const float R1_20 = -c1 - 6.123234262925839e-17f * s1; \
    const float R1_21 = -6.123234262925839e-17f * c1 + s1; \
    const float t1_0 = 0.1358499974012375f * R0_01; \
    const float t1_1 = 0.1358499974012375f * R0_11; \
    /* joint 2 (revolute, parent 1) */ \
    float s2, c2; sincosf(q[2], &s2, &c2); \
    const float R2_00 = c2 * R1_00 + s2 * R1_01; \
    const float R2_01 = c2 * R1_01 - s2 * R1_00; \
    const float R2_10 = c2 * R1_10 + s2 * R1_11; \
    const float R2_11 = c2 * R1_11 - s2 * R1_10; \
    const float R2_20 = c2 * R1_20 + s2 * R1_21; \
    const float R2_21 = c2 * R1_21 - s2 * R1_20; \
    const float t2_0 = t1_0 + -0.42500001192092896f * R1_01 + -0.11969999969005585f * R0_01; \
    const float t2_1 = t1_1 + -0.42500001192092896f * R1_11 + -0.11969999969005585f * R0_11; \
    const float t2_2 = 0.08915899693965912f + -0.42500001192092896f * R1_21; \
    /* joint 3 (revolute, parent 2) */ \
    const float M3_00 = 6.123234262925839e-17f * R2_00 + R2_01; \
    const float M3_01 = -R2_00 + 6.123234262925839e-17f * R2_01; \
    const float M3_10 = 6.123234262925839e-17f * R2_10 + R2_11; \
    const float M3_11 = -R2_10 + 6.123234262925839e-17f * R2_11; \
    const float M3_20 = 6.123234262925839e-17f * R2_20 + R2_21; \
    const float M3_21 = -R2_20 + 6.123234262925839e-17f * R2_21; \
    float s3, c3; sincosf(q[3], &s3, &c3); \
    const float R3_00 = c3 * M3_00 + s3 * M3_01; \
    const float R3_01 = c3 * M3_01 - s3 * M3_00; \
    const float R3_10 = c3 * M3_10 + s3 * M3_11; \
    const float R3_11 = c3 * M3_11 - s3 * M3_10; \
    const float R3_20 = c3 * M3_20 + s3 * M3_21; \
    const float R3_21 = c3 * M3_21 - s3 * M3_20; \
    const float t3_0 = t2_0 + -0.3922500014305115f * R2_01; \
    const float t3_1 = t2_1 + -0.3922500014305115f * R2_11; \
    const float t3_2 = t2_2 + -0.3922500014305115f * R2_21; \
    /* joint 4 (revolute, parent 3) */ \
    const float M4_02 = -R3_01; \
    const float M4_12 = -R3_11; \
    const float M4_22 = -R3_21; \
    float s4, c4; sincosf(q[4], &s4, &c4); \
    const float R4_00 = c4 * R3_00 + s4 * R0_01; \
    const float R4_01 = c4 * R0_01 - s4 * R3_00; \
    const float R4_10 = c4 * R3_10 + s4 * R0_11; \
    const float R4_11 = c4 * R0_11 - s4 * R3_10; \
    const float R4_20 = c4 * R3_20; \
    const float R4_21 = -s4 * R3_20; \
    const float t4_0 = t3_0 + 0.09300000220537186f * R0_01; \
    const float t4_1 = t3_1 + 0.09300000220537186f * R0_11; \
    /* joint 5 (revolute, parent 4) */ \
    const float M5_01 = -M4_02; \
    const float M5_11 = -M4_12; \
    const float M5_21 = -M4_22; \
    float s5, c5; sincosf(q[5], &s5, &c5); \
    const float R5_00 = c5 * R4_00 + s5 * M5_01; \
    const float R5_01 = c5 * M5_01 - s5 * R4_00; \
    const float R5_10 = c5 * R4_10 + s5 * M5_11; \
    const float R5_11 = c5 * M5_11 - s5 * R4_10; \
    const float R5_20 = c5 * R4_20 + s5 * M5_21; \
    const float R5_21 = c5 * M5_21 - s5 * R4_20; \
    const float t5_0 = t4_0 + 0.09465000033378601f * M4_02; \
    const float t5_1 = t4_1 + 0.09465000033378601f * M4_12; \
    const float t5_2 = t3_2 + 0.09465000033378601f * M4_22; \
    /* end FK */

__device__ __forceinline__ void fk_spheres(const float *q, float *out) {
    PRRTC_FK_BODY
    out[0] = 0.0f; out[1] = 0.0f; out[2] = 0.04500000178813934f;
    out[3] = 0.0f; out[4] = 0.0f; out[5] = 0.08915899693965912f;
    out[6] = 0.07000000029802322f * R0_01; out[7] = 0.07000000029802322f * R0_11; out[8] = 0.08915899693965912f;
    out[9] = t1_0; out[10] = t1_1; out[11] = 0.08915899693965912f;
    out[12] = -0.08500000089406967f * R1_01 + t1_0; out[13] = -0.08500000089406967f * R1_11 + t1_1; out[14] = 0.08915899693965912f + -0.08500000089406967f * R1_21;
    out[15] = -0.17000000178813934f * R1_01 + t1_0; out[16] = -0.17000000178813934f * R1_11 + t1_1; out[17] = 0.08915899693965912f + -0.17000000178813934f * R1_21;
    out[18] = -0.2549999952316284f * R1_01 + t1_0; out[19] = -0.2549999952316284f * R1_11 + t1_1; out[20] = 0.08915899693965912f + -0.2549999952316284f * R1_21;
    out[21] = -0.3400000035762787f * R1_01 + t1_0; out[22] = -0.3400000035762787f * R1_11 + t1_1; out[23] = 0.08915899693965912f + -0.3400000035762787f * R1_21;
    out[24] = -0.42500001192092896f * R1_01 + t1_0; out[25] = -0.42500001192092896f * R1_11 + t1_1; out[26] = 0.08915899693965912f + -0.42500001192092896f * R1_21;
    out[27] = -0.42500001192092896f * R1_01 + -0.05999999865889549f * R0_01 + t1_0; out[28] = -0.42500001192092896f * R1_11 + -0.05999999865889549f * R0_11 + t1_1; out[29] = 0.08915899693965912f + -0.42500001192092896f * R1_21;
    out[30] = t2_0; out[31] = t2_1; out[32] = t2_2;
    out[33] = -0.07999999821186066f * R2_01 + t2_0; out[34] = -0.07999999821186066f * R2_11 + t2_1; out[35] = -0.07999999821186066f * R2_21 + t2_2;
    out[36] = -0.1599999964237213f * R2_01 + t2_0; out[37] = -0.1599999964237213f * R2_11 + t2_1; out[38] = -0.1599999964237213f * R2_21 + t2_2;
    out[39] = -0.23999999463558197f * R2_01 + t2_0; out[40] = -0.23999999463558197f * R2_11 + t2_1; out[41] = -0.23999999463558197f * R2_21 + t2_2;
    out[42] = -0.3199999928474426f * R2_01 + t2_0; out[43] = -0.3199999928474426f * R2_11 + t2_1; out[44] = -0.3199999928474426f * R2_21 + t2_2;
    out[45] = -0.3922500014305115f * R2_01 + t2_0; out[46] = -0.3922500014305115f * R2_11 + t2_1; out[47] = -0.3922500014305115f * R2_21 + t2_2;
    out[48] = t3_0; out[49] = t3_1; out[50] = t3_2;
    out[51] = 0.05000000074505806f * R0_01 + t3_0; out[52] = 0.05000000074505806f * R0_11 + t3_1; out[53] = t3_2;
    out[54] = t4_0; out[55] = t4_1; out[56] = t3_2;
    out[57] = 0.05000000074505806f * M4_02 + t4_0; out[58] = 0.05000000074505806f * M4_12 + t4_1; out[59] = 0.05000000074505806f * M4_22 + t3_2;
    out[60] = t5_0; out[61] = t5_1; out[62] = t5_2;
    out[63] = 0.05000000074505806f * R4_01 + t5_0; out[64] = 0.05000000074505806f * R4_11 + t5_1; out[65] = 0.05000000074505806f * R4_21 + t5_2;
    out[66] = 2.449293581093244e-18f * R5_00 + 0.12229999899864197f * R4_01 + t5_0; out[67] = 2.449293581093244e-18f * R5_10 + 0.12229999899864197f * R4_11 + t5_1; out[68] = 2.449293581093244e-18f * R5_20 + 0.12229999899864197f * R4_21 + t5_2;
    out[69] = 0.03500000014901161f * R0_01; out[70] = 0.03500000014901161f * R0_11; out[71] = 0.08915899693965912f;
    out[72] = -0.24285714328289032f * R1_01 + -0.008571428246796131f * R0_01 + t1_0; out[73] = -0.24285714328289032f * R1_11 + -0.008571428246796131f * R0_11 + t1_1; out[74] = 0.08915899693965912f + -0.24285714328289032f * R1_21;
    out[75] = -0.19870834052562714f * R2_01 + t2_0; out[76] = -0.19870834052562714f * R2_11 + t2_1; out[77] = -0.19870834052562714f * R2_21 + t2_2;
    out[78] = 0.02500000037252903f * R0_01 + t3_0; out[79] = 0.02500000037252903f * R0_11 + t3_1; out[80] = t3_2;
    out[81] = 0.02500000037252903f * M4_02 + t4_0; out[82] = 0.02500000037252903f * M4_12 + t4_1; out[83] = 0.02500000037252903f * M4_22 + t3_2;
    out[84] = 0.02500000037252903f * R4_01 + t5_0; out[85] = 0.02500000037252903f * R4_11 + t5_1; out[86] = 0.02500000037252903f * R4_21 + t5_2;
}
__host__ __device__ constexpr float radius(int i) { constexpr float v[] = {0.09000000357627869f, 0.07500000298023224f, 0.07000000029802322f, 0.06499999761581421f, 0.054999999701976776f, 0.054999999701976776f, 0.054999999701976776f, 0.054999999701976776f, 0.06499999761581421f, 0.05999999865889549f, 0.05000000074505806f, 0.05000000074505806f, 0.05000000074505806f, 0.05000000074505806f, 0.05000000074505806f, 0.05000000074505806f, 0.04500000178813934f, 0.04500000178813934f, 0.04500000178813934f, 0.04500000178813934f, 0.03999999910593033f, 0.03999999910593033f, 0.03999999910593033f, 0.10999999940395355f, 0.3080083429813385f, 0.2487083375453949f, 0.07000000029802322f, 0.07000000029802322f, 0.06499999761581421f}; return v[i]; }

template <class Ctx>
__device__ __forceinline__ void check(const float *q, Ctx &ctx) {
    PRRTC_FK_BODY
    uint64_t gate = 0;  /* bit k: env check k's gate sphere hit */
    if (ctx.any(ctx.live())) {
        {
            const float ex[7] = {0.03500000014901161f * R0_01, -0.24285714328289032f * R1_01 + -0.008571428246796131f * R0_01 + t1_0, -0.19870834052562714f * R2_01 + t2_0, 0.02500000037252903f * R0_01 + t3_0, 0.02500000037252903f * M4_02 + t4_0, 0.02500000037252903f * R4_01 + t5_0, 2.449293581093244e-18f * R5_00 + 0.12229999899864197f * R4_01 + t5_0};
            const float ey[7] = {0.03500000014901161f * R0_11, -0.24285714328289032f * R1_11 + -0.008571428246796131f * R0_11 + t1_1, -0.19870834052562714f * R2_11 + t2_1, 0.02500000037252903f * R0_11 + t3_1, 0.02500000037252903f * M4_12 + t4_1, 0.02500000037252903f * R4_11 + t5_1, 2.449293581093244e-18f * R5_10 + 0.12229999899864197f * R4_11 + t5_1};
            const float ez[7] = {0.08915899693965912f, 0.08915899693965912f + -0.24285714328289032f * R1_21, -0.19870834052562714f * R2_21 + t2_2, t3_2, 0.02500000037252903f * M4_22 + t3_2, 0.02500000037252903f * R4_21 + t5_2, 2.449293581093244e-18f * R5_20 + 0.12229999899864197f * R4_21 + t5_2};
            const float er[7] = {0.10999999940395355f, 0.3080083429813385f, 0.2487083375453949f, 0.07000000029802322f, 0.07000000029802322f, 0.06499999761581421f, 0.03999999910593033f};
            bool eh[7];
            ctx.template env_gates<7>(0, ex, ey, ez, er, eh);
            gate |= ((uint64_t)eh[0] << 0) | ((uint64_t)eh[1] << 1) | ((uint64_t)eh[2] << 2) | ((uint64_t)eh[3] << 3) | ((uint64_t)eh[4] << 4) | ((uint64_t)eh[5] << 5) | ((uint64_t)eh[6] << 6);
        }
    }
    ctx.share_gates(gate);
    if (ctx.live() && (gate & 64ull)) ctx.hit();
    if (ctx.stop()) return;
    /* env leaves: shoulder_link */
    if (ctx.any(ctx.live() && (gate >> 0 & 1))) {
        const bool on = ctx.live() && (gate >> 0 & 1);
        {
            const float ex[2] = {0.0f, 0.07000000029802322f * R0_01};
            const float ey[2] = {0.0f, 0.07000000029802322f * R0_11};
            const float ez[2] = {0.08915899693965912f, 0.08915899693965912f};
            const float er[2] = {0.07500000298023224f, 0.07000000029802322f};
            const bool eh = ctx.template env_any<2, true>(ex, ey, ez, er, on);
            if (on && eh) ctx.hit();
        }
        if (ctx.stop()) return;
    }
    /* env leaves: upper_arm_link */
    if (ctx.any(ctx.live() && (gate >> 1 & 1))) {
        const bool on = ctx.live() && (gate >> 1 & 1);
        {
            const float ex[7] = {t1_0, -0.08500000089406967f * R1_01 + t1_0, -0.17000000178813934f * R1_01 + t1_0, -0.2549999952316284f * R1_01 + t1_0, -0.3400000035762787f * R1_01 + t1_0, -0.42500001192092896f * R1_01 + t1_0, -0.42500001192092896f * R1_01 + -0.05999999865889549f * R0_01 + t1_0};
            const float ey[7] = {t1_1, -0.08500000089406967f * R1_11 + t1_1, -0.17000000178813934f * R1_11 + t1_1, -0.2549999952316284f * R1_11 + t1_1, -0.3400000035762787f * R1_11 + t1_1, -0.42500001192092896f * R1_11 + t1_1, -0.42500001192092896f * R1_11 + -0.05999999865889549f * R0_11 + t1_1};
            const float ez[7] = {0.08915899693965912f, 0.08915899693965912f + -0.08500000089406967f * R1_21, 0.08915899693965912f + -0.17000000178813934f * R1_21, 0.08915899693965912f + -0.2549999952316284f * R1_21, 0.08915899693965912f + -0.3400000035762787f * R1_21, 0.08915899693965912f + -0.42500001192092896f * R1_21, 0.08915899693965912f + -0.42500001192092896f * R1_21};
            const float er[7] = {0.06499999761581421f, 0.054999999701976776f, 0.054999999701976776f, 0.054999999701976776f, 0.054999999701976776f, 0.06499999761581421f, 0.05999999865889549f};
            const bool eh = ctx.template env_any_bounded<7, true>(ex, ey, ez, er, on, -0.24285714328289032f * R1_01 + -0.008571428246796131f * R0_01 + t1_0, -0.24285714328289032f * R1_11 + -0.008571428246796131f * R0_11 + t1_1, 0.08915899693965912f + -0.24285714328289032f * R1_21, 0.30901309847831726f);
            if (on && eh) ctx.hit();
        }
        if (ctx.stop()) return;
    }
    /* env leaves: forearm_link */
    if (ctx.any(ctx.live() && (gate >> 2 & 1))) {
        const bool on = ctx.live() && (gate >> 2 & 1);
        {
            const float ex[6] = {t2_0, -0.07999999821186066f * R2_01 + t2_0, -0.1599999964237213f * R2_01 + t2_0, -0.23999999463558197f * R2_01 + t2_0, -0.3199999928474426f * R2_01 + t2_0, -0.3922500014305115f * R2_01 + t2_0};
            const float ey[6] = {t2_1, -0.07999999821186066f * R2_11 + t2_1, -0.1599999964237213f * R2_11 + t2_1, -0.23999999463558197f * R2_11 + t2_1, -0.3199999928474426f * R2_11 + t2_1, -0.3922500014305115f * R2_11 + t2_1};
            const float ez[6] = {t2_2, -0.07999999821186066f * R2_21 + t2_2, -0.1599999964237213f * R2_21 + t2_2, -0.23999999463558197f * R2_21 + t2_2, -0.3199999928474426f * R2_21 + t2_2, -0.3922500014305115f * R2_21 + t2_2};
            const float er[6] = {0.05000000074505806f, 0.05000000074505806f, 0.05000000074505806f, 0.05000000074505806f, 0.05000000074505806f, 0.05000000074505806f};
            const bool eh = ctx.template env_any_bounded<6, true>(ex, ey, ez, er, on, -0.19870834052562714f * R2_01 + t2_0, -0.19870834052562714f * R2_11 + t2_1, -0.19870834052562714f * R2_21 + t2_2, 0.24971213936805725f);
            if (on && eh) ctx.hit();
        }
        if (ctx.stop()) return;
    }
    /* env leaves: wrist_1_link */
    if (ctx.any(ctx.live() && (gate >> 3 & 1))) {
        const bool on = ctx.live() && (gate >> 3 & 1);
        {
            const float ex[2] = {t3_0, 0.05000000074505806f * R0_01 + t3_0};
            const float ey[2] = {t3_1, 0.05000000074505806f * R0_11 + t3_1};
            const float ez[2] = {t3_2, t3_2};
            const float er[2] = {0.04500000178813934f, 0.04500000178813934f};
            const bool eh = ctx.template env_any<2, true>(ex, ey, ez, er, on);
            if (on && eh) ctx.hit();
        }
        if (ctx.stop()) return;
    }
    /* env leaves: wrist_2_link */
    if (ctx.any(ctx.live() && (gate >> 4 & 1))) {
        const bool on = ctx.live() && (gate >> 4 & 1);
        {
            const float ex[2] = {t4_0, 0.05000000074505806f * M4_02 + t4_0};
            const float ey[2] = {t4_1, 0.05000000074505806f * M4_12 + t4_1};
            const float ez[2] = {t3_2, 0.05000000074505806f * M4_22 + t3_2};
            const float er[2] = {0.04500000178813934f, 0.04500000178813934f};
            const bool eh = ctx.template env_any<2, true>(ex, ey, ez, er, on);
            if (on && eh) ctx.hit();
        }
        if (ctx.stop()) return;
    }
    /* env leaves: wrist_3_link */
    if (ctx.any(ctx.live() && (gate >> 5 & 1))) {
        const bool on = ctx.live() && (gate >> 5 & 1);
        {
            const float ex[2] = {t5_0, 0.05000000074505806f * R4_01 + t5_0};
            const float ey[2] = {t5_1, 0.05000000074505806f * R4_11 + t5_1};
            const float ez[2] = {t5_2, 0.05000000074505806f * R4_21 + t5_2};
            const float er[2] = {0.03999999910593033f, 0.03999999910593033f};
            const bool eh = ctx.template env_any<2, true>(ex, ey, ez, er, on);
            if (on && eh) ctx.hit();
        }
        if (ctx.stop()) return;
    }
    ctx.template self_own<33>();
    /* self: wrist_2_link vs. base_link */
    if (ctx.mine(0)) {
        const bool g = ctx.live() && ctx.self(t4_0, t4_1, t3_2, 0.0f, 0.0f, 0.04500000178813934f, 0.13500000536441803f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_2_link vs. base_link */
    if (ctx.mine(1)) {
        const bool g = ctx.live() && ctx.self(0.05000000074505806f * M4_02 + t4_0, 0.05000000074505806f * M4_12 + t4_1, 0.05000000074505806f * M4_22 + t3_2, 0.0f, 0.0f, 0.04500000178813934f, 0.13500000536441803f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_2_link vs. shoulder_link */
    if (ctx.mine(2)) {
        const bool g = ctx.live() && ctx.self(t4_0, t4_1, t3_2, 0.0f, 0.0f, 0.08915899693965912f, 0.12000000476837158f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_2_link vs. shoulder_link */
    if (ctx.mine(3)) {
        const bool g = ctx.live() && ctx.self(t4_0, t4_1, t3_2, 0.07000000029802322f * R0_01, 0.07000000029802322f * R0_11, 0.08915899693965912f, 0.11500000208616257f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_2_link vs. shoulder_link */
    if (ctx.mine(4)) {
        const bool g = ctx.live() && ctx.self(0.05000000074505806f * M4_02 + t4_0, 0.05000000074505806f * M4_12 + t4_1, 0.05000000074505806f * M4_22 + t3_2, 0.0f, 0.0f, 0.08915899693965912f, 0.12000000476837158f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_2_link vs. shoulder_link */
    if (ctx.mine(5)) {
        const bool g = ctx.live() && ctx.self(0.05000000074505806f * M4_02 + t4_0, 0.05000000074505806f * M4_12 + t4_1, 0.05000000074505806f * M4_22 + t3_2, 0.07000000029802322f * R0_01, 0.07000000029802322f * R0_11, 0.08915899693965912f, 0.11500000208616257f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_2_link vs. upper_arm_link */
    if (ctx.mine(6)) {
        const bool g = ctx.live() && ctx.self(t4_0, t4_1, t3_2, t1_0, t1_1, 0.08915899693965912f, 0.10999999940395355f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_2_link vs. upper_arm_link */
    if (ctx.mine(7)) {
        const bool g = ctx.live() && ctx.self(t4_0, t4_1, t3_2, -0.08500000089406967f * R1_01 + t1_0, -0.08500000089406967f * R1_11 + t1_1, 0.08915899693965912f + -0.08500000089406967f * R1_21, 0.10000000149011612f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_2_link vs. upper_arm_link */
    if (ctx.mine(8)) {
        const bool g = ctx.live() && ctx.self(t4_0, t4_1, t3_2, -0.17000000178813934f * R1_01 + t1_0, -0.17000000178813934f * R1_11 + t1_1, 0.08915899693965912f + -0.17000000178813934f * R1_21, 0.10000000149011612f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_2_link vs. upper_arm_link */
    if (ctx.mine(9)) {
        const bool g = ctx.live() && ctx.self(0.05000000074505806f * M4_02 + t4_0, 0.05000000074505806f * M4_12 + t4_1, 0.05000000074505806f * M4_22 + t3_2, t1_0, t1_1, 0.08915899693965912f, 0.10999999940395355f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_2_link vs. upper_arm_link */
    if (ctx.mine(10)) {
        const bool g = ctx.live() && ctx.self(0.05000000074505806f * M4_02 + t4_0, 0.05000000074505806f * M4_12 + t4_1, 0.05000000074505806f * M4_22 + t3_2, -0.08500000089406967f * R1_01 + t1_0, -0.08500000089406967f * R1_11 + t1_1, 0.08915899693965912f + -0.08500000089406967f * R1_21, 0.10000000149011612f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_2_link vs. upper_arm_link */
    if (ctx.mine(11)) {
        const bool g = ctx.live() && ctx.self(0.05000000074505806f * M4_02 + t4_0, 0.05000000074505806f * M4_12 + t4_1, 0.05000000074505806f * M4_22 + t3_2, -0.17000000178813934f * R1_01 + t1_0, -0.17000000178813934f * R1_11 + t1_1, 0.08915899693965912f + -0.17000000178813934f * R1_21, 0.10000000149011612f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_3_link vs. base_link */
    if (ctx.mine(12)) {
        const bool g = ctx.live() && ctx.self(t5_0, t5_1, t5_2, 0.0f, 0.0f, 0.04500000178813934f, 0.12999999523162842f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_3_link vs. base_link */
    if (ctx.mine(13)) {
        const bool g = ctx.live() && ctx.self(0.05000000074505806f * R4_01 + t5_0, 0.05000000074505806f * R4_11 + t5_1, 0.05000000074505806f * R4_21 + t5_2, 0.0f, 0.0f, 0.04500000178813934f, 0.12999999523162842f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_3_link vs. shoulder_link */
    if (ctx.mine(14)) {
        const bool g = ctx.live() && ctx.self(t5_0, t5_1, t5_2, 0.0f, 0.0f, 0.08915899693965912f, 0.11500000208616257f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_3_link vs. shoulder_link */
    if (ctx.mine(15)) {
        const bool g = ctx.live() && ctx.self(t5_0, t5_1, t5_2, 0.07000000029802322f * R0_01, 0.07000000029802322f * R0_11, 0.08915899693965912f, 0.10999999940395355f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_3_link vs. shoulder_link */
    if (ctx.mine(16)) {
        const bool g = ctx.live() && ctx.self(0.05000000074505806f * R4_01 + t5_0, 0.05000000074505806f * R4_11 + t5_1, 0.05000000074505806f * R4_21 + t5_2, 0.0f, 0.0f, 0.08915899693965912f, 0.11500000208616257f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_3_link vs. shoulder_link */
    if (ctx.mine(17)) {
        const bool g = ctx.live() && ctx.self(0.05000000074505806f * R4_01 + t5_0, 0.05000000074505806f * R4_11 + t5_1, 0.05000000074505806f * R4_21 + t5_2, 0.07000000029802322f * R0_01, 0.07000000029802322f * R0_11, 0.08915899693965912f, 0.10999999940395355f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_3_link vs. upper_arm_link */
    if (ctx.mine(18)) {
        const bool g = ctx.live() && ctx.self(t5_0, t5_1, t5_2, t1_0, t1_1, 0.08915899693965912f, 0.10499999672174454f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_3_link vs. upper_arm_link */
    if (ctx.mine(19)) {
        const bool g = ctx.live() && ctx.self(t5_0, t5_1, t5_2, -0.08500000089406967f * R1_01 + t1_0, -0.08500000089406967f * R1_11 + t1_1, 0.08915899693965912f + -0.08500000089406967f * R1_21, 0.0949999988079071f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_3_link vs. upper_arm_link */
    if (ctx.mine(20)) {
        const bool g = ctx.live() && ctx.self(t5_0, t5_1, t5_2, -0.17000000178813934f * R1_01 + t1_0, -0.17000000178813934f * R1_11 + t1_1, 0.08915899693965912f + -0.17000000178813934f * R1_21, 0.0949999988079071f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_3_link vs. upper_arm_link */
    if (ctx.mine(21)) {
        const bool g = ctx.live() && ctx.self(0.05000000074505806f * R4_01 + t5_0, 0.05000000074505806f * R4_11 + t5_1, 0.05000000074505806f * R4_21 + t5_2, t1_0, t1_1, 0.08915899693965912f, 0.10499999672174454f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_3_link vs. upper_arm_link */
    if (ctx.mine(22)) {
        const bool g = ctx.live() && ctx.self(0.05000000074505806f * R4_01 + t5_0, 0.05000000074505806f * R4_11 + t5_1, 0.05000000074505806f * R4_21 + t5_2, -0.08500000089406967f * R1_01 + t1_0, -0.08500000089406967f * R1_11 + t1_1, 0.08915899693965912f + -0.08500000089406967f * R1_21, 0.0949999988079071f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: wrist_3_link vs. upper_arm_link */
    if (ctx.mine(23)) {
        const bool g = ctx.live() && ctx.self(0.05000000074505806f * R4_01 + t5_0, 0.05000000074505806f * R4_11 + t5_1, 0.05000000074505806f * R4_21 + t5_2, -0.17000000178813934f * R1_01 + t1_0, -0.17000000178813934f * R1_11 + t1_1, 0.08915899693965912f + -0.17000000178813934f * R1_21, 0.0949999988079071f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: ee_link vs. base_link */
    if (ctx.mine(24)) {
        const bool g = ctx.live() && ctx.self(2.449293581093244e-18f * R5_00 + 0.12229999899864197f * R4_01 + t5_0, 2.449293581093244e-18f * R5_10 + 0.12229999899864197f * R4_11 + t5_1, 2.449293581093244e-18f * R5_20 + 0.12229999899864197f * R4_21 + t5_2, 0.0f, 0.0f, 0.04500000178813934f, 0.12999999523162842f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: ee_link vs. shoulder_link */
    if (ctx.mine(25)) {
        const bool g = ctx.live() && ctx.self(2.449293581093244e-18f * R5_00 + 0.12229999899864197f * R4_01 + t5_0, 2.449293581093244e-18f * R5_10 + 0.12229999899864197f * R4_11 + t5_1, 2.449293581093244e-18f * R5_20 + 0.12229999899864197f * R4_21 + t5_2, 0.0f, 0.0f, 0.08915899693965912f, 0.11500000208616257f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: ee_link vs. shoulder_link */
    if (ctx.mine(26)) {
        const bool g = ctx.live() && ctx.self(2.449293581093244e-18f * R5_00 + 0.12229999899864197f * R4_01 + t5_0, 2.449293581093244e-18f * R5_10 + 0.12229999899864197f * R4_11 + t5_1, 2.449293581093244e-18f * R5_20 + 0.12229999899864197f * R4_21 + t5_2, 0.07000000029802322f * R0_01, 0.07000000029802322f * R0_11, 0.08915899693965912f, 0.10999999940395355f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: ee_link vs. upper_arm_link */
    if (ctx.mine(27)) {
        const bool g = ctx.live() && ctx.self(2.449293581093244e-18f * R5_00 + 0.12229999899864197f * R4_01 + t5_0, 2.449293581093244e-18f * R5_10 + 0.12229999899864197f * R4_11 + t5_1, 2.449293581093244e-18f * R5_20 + 0.12229999899864197f * R4_21 + t5_2, t1_0, t1_1, 0.08915899693965912f, 0.10499999672174454f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: ee_link vs. upper_arm_link */
    if (ctx.mine(28)) {
        const bool g = ctx.live() && ctx.self(2.449293581093244e-18f * R5_00 + 0.12229999899864197f * R4_01 + t5_0, 2.449293581093244e-18f * R5_10 + 0.12229999899864197f * R4_11 + t5_1, 2.449293581093244e-18f * R5_20 + 0.12229999899864197f * R4_21 + t5_2, -0.08500000089406967f * R1_01 + t1_0, -0.08500000089406967f * R1_11 + t1_1, 0.08915899693965912f + -0.08500000089406967f * R1_21, 0.0949999988079071f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: ee_link vs. upper_arm_link */
    if (ctx.mine(29)) {
        const bool g = ctx.live() && ctx.self(2.449293581093244e-18f * R5_00 + 0.12229999899864197f * R4_01 + t5_0, 2.449293581093244e-18f * R5_10 + 0.12229999899864197f * R4_11 + t5_1, 2.449293581093244e-18f * R5_20 + 0.12229999899864197f * R4_21 + t5_2, -0.17000000178813934f * R1_01 + t1_0, -0.17000000178813934f * R1_11 + t1_1, 0.08915899693965912f + -0.17000000178813934f * R1_21, 0.0949999988079071f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: forearm_link vs. base_link */
    if (ctx.mine(30)) {
        const bool g = ctx.live() && ctx.self(-0.23999999463558197f * R2_01 + t2_0, -0.23999999463558197f * R2_11 + t2_1, -0.23999999463558197f * R2_21 + t2_2, 0.0f, 0.0f, 0.04500000178813934f, 0.14000000059604645f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: forearm_link vs. base_link */
    if (ctx.mine(31)) {
        const bool g = ctx.live() && ctx.self(-0.3199999928474426f * R2_01 + t2_0, -0.3199999928474426f * R2_11 + t2_1, -0.3199999928474426f * R2_21 + t2_2, 0.0f, 0.0f, 0.04500000178813934f, 0.14000000059604645f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
    /* self: forearm_link vs. base_link */
    if (ctx.mine(32)) {
        const bool g = ctx.live() && ctx.self(-0.3922500014305115f * R2_01 + t2_0, -0.3922500014305115f * R2_11 + t2_1, -0.3922500014305115f * R2_21 + t2_2, 0.0f, 0.0f, 0.04500000178813934f, 0.14000000059604645f);
        if (ctx.any(g)) {
            if (g) ctx.hit();
            if (ctx.stop()) return;
        }
    }
}
#undef PRRTC_FK_BODY

}  // namespace prrtc::gen::ur5
