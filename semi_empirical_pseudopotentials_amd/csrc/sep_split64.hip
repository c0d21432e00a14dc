// sep_split64.hip -- the two-kernel H.psi of sep_split.h in double.
#include <hip/hip_runtime.h>

#include "sep_split.h"

namespace sep {
template struct SplitOps<double>;
}  // namespace sep
