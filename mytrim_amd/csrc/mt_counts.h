// The count of a history's outstanding flights (queued or running), which serves
// the cascade budget alone.  A wave counts until it has seen every primary
// started; from then on it neither adds the recoils it pushes nor takes off the
// flights it ends, while another wave, which read the primaries' counter earlier,
// may still count.  So before every primary has started a push finds a count of at
// least 1 (the pushing flight is outstanding), and afterwards a count says nothing.
#pragma once
#include <hip/hip_runtime.h>

namespace mt {

// whether a push may have found `before` outstanding flights, with `started`
// primaries started (read after it) of n_hist
__host__ __device__ __forceinline__ bool count_possible(int before, unsigned long long started, long long n_hist) {
  return before >= 1 || started >= (unsigned long long)n_hist;
}

}  // namespace mt
