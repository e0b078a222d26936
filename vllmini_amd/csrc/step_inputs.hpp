// What the launches of a decode step read, from pinned host memory to where they read it, and the tokens' ids to theirs: one launch.
//
// Bound by a trip over the bus (about 2 us) and a launch.  Two copies of the runtime, one off the host and one between device tensors, each go to another queue and back:
// 12 layers x 32 sequences with 64 blocks of room each (98 KB) 31 us between two replays of a step's graph, so 7: of the block tables only the columns that the sequences use are read.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace vmi_step {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct Inputs {
  const char* host;   // pinned: head bytes, then a table of rows x ld whole numbers, of which the first `used` of a row count
  char* dev;          // the same, in device memory
  int64_t head;       // a multiple of 16
  int rows, ld, used, n;
  const int64_t* ids;
  int64_t* ids_out;   // n of them
};

__global__ __launch_bounds__(256) void inputs_kernel(const Inputs p) {
  const int64_t units = p.head >> 4, cells = (int64_t)p.rows * p.used;
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < units) {
    reinterpret_cast<u32x4*>(p.dev)[i] = reinterpret_cast<const u32x4*>(p.host)[i];
    return;
  }
  i -= units;
  if (i < cells) {
    const int64_t r = i / p.used, at = p.head + (r * p.ld + (i - r * p.used)) * 4;
    *reinterpret_cast<int32_t*>(p.dev + at) = *reinterpret_cast<const int32_t*>(p.host + at);
    return;
  }
  i -= cells;
  if (i < p.n) p.ids_out[i] = p.ids[i];
}

inline bool inputs_fit(const Inputs& p) {
  return p.host && p.dev && p.head >= 0 && (p.head & 15) == 0 && !((uintptr_t)p.host & 15) && !((uintptr_t)p.dev & 15) && p.rows >= 0 && p.used >= 0 && p.used <= p.ld &&
         p.n >= 0 && (p.n == 0 || (p.ids && p.ids_out)) && (p.head >> 4) + (int64_t)p.rows * p.used + p.n < (int64_t)1 << 31;
}
inline void launch_inputs(const Inputs& p, hipStream_t st) {
  const int64_t all = (p.head >> 4) + (int64_t)p.rows * p.used + p.n;
  if (all > 0) hipLaunchKernelGGL(inputs_kernel, dim3((unsigned)((all + 255) / 256)), dim3(256), 0, st, p);
}

}  // namespace vmi_step
