// The MLX-layout GEMM (qgemmx.h) at 5-bit codes: a file per width, so they build side by side.
#include "qgemmx.h"

namespace mlxr {
hipError_t qgemmx_launch5(const QGemmXDev& d, int gs, int cut, hipStream_t s) { return qgemmx_width<5>(d, gs, cut, s); }
}  // namespace mlxr
