// fake_hip.h -- controls of the host-only HIP stand-in (fake_hip.cpp).
#pragma once
#include <cstddef>
#include <cstdint>
#include <string>
#include <vector>

namespace fake {

struct Launch {
  std::string name;  // row pair rowpair wave solo solo_flow lane lane_flow ...
  int size = 0;      // geometry, positions or quads of a chain
  int grid = 0;
  int lanes = 0;
  bool plain = false, row2 = false;
};

extern std::vector<Launch> launches;  // the jump kernels, in order
extern int nulls;                     // launches that were given a null pointer they use
extern int64_t allocs;                // hipMalloc calls so far
extern int64_t fail_from, fail_to;    // the calls (counted from 1) in this range fail
extern int64_t live_bytes, live_count;
extern int64_t pinned;                // hipHostMalloc calls so far
extern size_t capacity;               // device memory; a call beyond it fails
inline void fail_next(int64_t k, int64_t n = 1) { fail_from = allocs + k; fail_to = fail_from + n - 1; }
inline void fail_none() { fail_from = fail_to = 0; }

}  // namespace fake
