// A store, stores_done, a store: compiled (never run) by tests/test_stores.py.
#include "../../prrtc_amd/csrc/host_common.h"
#include "../../prrtc_amd/csrc/planner_device.h"

extern "C" __global__ void two_stores(int *a, int *b) {
    a[threadIdx.x] = 1;
    prrtc::stores_done();
    b[threadIdx.x] = 2;
}
