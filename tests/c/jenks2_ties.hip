// The mask of a two-class split at any position, for the tests: fb_jenks2_gpu takes the split it
// finds, which is practically never inside a run of equal values.
#include <hip/hip_runtime.h>

#include "../../if_i_could_turn_back_time_amd/csrc/fourbit_jenks2_mask.h"

// Scratch bytes of ties_mask for n values.
extern "C" int64_t ties_scratch_bytes(int64_t n) { return 256 + 4 * tie_segments(n); }

// keep [n] (uint8) for w [n], its sort and *split, device pointers; scratch 256-byte aligned.
extern "C" int ties_mask(const float* w, int64_t n, const float* sorted, const int64_t* split,
                         uint8_t* keep, void* scratch, void* stream) {
  if (!w || !sorted || !split || !keep || !scratch || n < 1 || n > INT32_MAX) return -1;
  launch_mask(w, (int)n, sorted, split, static_cast<J2Ties*>(scratch),
              reinterpret_cast<int*>(static_cast<uint8_t*>(scratch) + 256), keep,
              static_cast<hipStream_t>(stream));
  return hipGetLastError() == hipSuccess ? 0 : -2;
}
