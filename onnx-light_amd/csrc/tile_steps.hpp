// The split of a tile GEMM's K steps (tile_gemm.hpp) into those read with plain
// loads and the guarded rest.  No HIP header, so that a CPU compiler takes it
// too: which bytes a plain step reads is checked over small shapes on the host.
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define OLA_HOST_DEVICE __host__ __device__
#else
#define OLA_HOST_DEVICE
#endif

namespace onnxl_amd {
namespace tg {

// Steps of `step` k values, ceil(K / step) in all, that plain 16-byte loads may
// read: no k of theirs lies past K, and every piece ends inside its matrix (one
// of a row-major B, `rows`, of pitch `pitch` bytes may cross into the next
// rows).  The others, at most two, come after them.
OLA_HOST_DEVICE inline int PlainSteps(int64_t K, int step, bool rows, int64_t pitch) {
  int plain = (int)((K + step - 1) / step);
  if (plain > 0 && (K % step != 0 || (rows && pitch % 16 != 0))) {  // K = 0: no step of either kind
    --plain;
    if (rows && plain > 0 && (K - (int64_t)plain * step + 1) * pitch < 16) --plain;
  }
  return plain;
}

}  // namespace tg
}  // namespace onnxl_amd
