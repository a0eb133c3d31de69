// Anchored line kernels instantiated for float (see lines_anchored.h).
#include <algorithm>

#include "lines_anchored.h"

namespace x3d {
template int launch_anchored<float>(const LineCall<float> &, const LineTriple<float> *, bool *, hipStream_t);
}  // namespace x3d
