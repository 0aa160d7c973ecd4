// Shared by the MLX-layout GEMM (qgemmx.h, gemm.hip) and the small batch (qmm.hip): operand types and constants.
#pragma once
#include "kernels.h"

namespace mlxr {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef __bf16 gx_bf8 __attribute__((ext_vector_type(8)));
typedef uint32_t gx_u4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* gx_lptr;

constexpr int GX_K = 64, GX_NST = 3;
constexpr int GX_RSRC_W3 = 0x00020000;   // raw buffer, 32-bit data format
// s_waitcnt vmcnt(n) (n < 64), expcnt and lgkmcnt not waited for
constexpr int gx_wait_vm(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }
// groups padded to a multiple of 4 (one chunk)
__host__ __device__ constexpr int gx_gpad(int G) { return (G + 3) / 4 * 4; }

constexpr int GX_GSUM = 24;   // bytes of a token's group sums of a chunk: hi, mid, lo bf16 parts of 4 groups

struct QGemmXDev;
// The GEMM of one code width over a cut (tile shape 0 .. 2).
hipError_t qgemmx_launch2(const QGemmXDev& d, int gs, int cut, hipStream_t s);
hipError_t qgemmx_launch3(const QGemmXDev& d, int gs, int cut, hipStream_t s);
hipError_t qgemmx_launch4(const QGemmXDev& d, int gs, int cut, hipStream_t s);
hipError_t qgemmx_launch5(const QGemmXDev& d, int gs, int cut, hipStream_t s);
hipError_t qgemmx_launch6(const QGemmXDev& d, int gs, int cut, hipStream_t s);
hipError_t qgemmx_launch8(const QGemmXDev& d, int gs, int cut, hipStream_t s);

}  // namespace mlxr
