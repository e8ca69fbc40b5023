// Row-wise assembly, FP64 values (direct_rows.h).
#include "direct_rows.h"

namespace slx {

hipError_t launch_direct_f64(const DirectDev& d, const DirectLaunch& q) { return launch_direct_k<double>(d, q); }

}  // namespace slx
