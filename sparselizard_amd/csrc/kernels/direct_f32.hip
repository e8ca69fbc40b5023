// Row-wise assembly, FP32 values (direct_rows.h).
#include "direct_rows.h"

namespace slx {

hipError_t launch_direct_f32(const DirectDev& d, const DirectLaunch& q) { return launch_direct_k<float>(d, q); }

}  // namespace slx
