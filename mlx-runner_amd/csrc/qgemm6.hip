// The MLX-layout GEMM (qgemmx.h) at 6-bit codes: a file per width, so they build side by side.
#include "qgemmx.h"

namespace mlxr {
hipError_t qgemmx_launch6(const QGemmXDev& d, int gs, int cut, hipStream_t s) { return qgemmx_width<6>(d, gs, cut, s); }
}  // namespace mlxr
