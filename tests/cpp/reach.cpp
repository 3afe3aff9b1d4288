// Host build of the broad phase's arithmetic (device_common.h), for
// tests/test_reach.py.  Modes:
//   lds    a staged scene takes scene_lds_f4 float4, at most scene_lds_f4_most
#include <cstdio>
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

int main(int argc, char **argv) {
    if (argc == 2 && !std::strcmp(argv[1], "lds")) return lds();
    return 2;
}
