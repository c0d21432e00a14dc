// sep_split32.hip -- the two-kernel H.psi of sep_split.h in float.
#include <hip/hip_runtime.h>

#include "sep_split.h"

namespace sep {
template struct SplitOps<float>;
}  // namespace sep
