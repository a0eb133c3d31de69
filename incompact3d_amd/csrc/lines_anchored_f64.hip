// Anchored line kernels instantiated for double (see lines_anchored.h).
#include <algorithm>

#include "lines_anchored.h"

namespace x3d {
template int launch_anchored<double>(const LineCall<double> &, const LineTriple<double> *, bool *, hipStream_t);
}  // namespace x3d
