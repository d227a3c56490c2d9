// State and records of the HIP runtime of fake_hip.cpp.
#pragma once

#include <hip/hip_runtime_api.h>

#include <map>
#include <string>
#include <vector>

namespace fake {

struct Launch {
    std::string name;          // mangled kernel name
    dim3 grid, block;
    void *pointer = nullptr;   // what k_fill_zero clears
};

struct State {
    int n_devices = 1, device = 0;
    int occupancy = 2;                     // resident workgroups per compute unit; 0: the runtime cannot tell
    size_t malloc_limit = ~size_t(0);      // device allocations of this size and more fail
    bool host_malloc_fails = false;
    hipError_t last_error = hipSuccess;
    std::vector<Launch> launches;
    std::vector<size_t> allocated;         // device allocations
    std::vector<unsigned> host_flags;      // flags of the pinned allocations
};

State &state();

}  // namespace fake
