// Host side and pre-passes of the MLX-layout GEMM (kernel: qgemmx.h, one file per code width).
#include "qgemmx.h"

namespace mlxr {

// Pre-pass: row t of x -> hi / lo (f16, [T][K]); gsum[g][t] (each group's sum of the scaled x,
// summed in k order per 8-chunk and chunks in order; zero past G) as three bf16 parts (truncations: hi + mid +
// lo exact), [Gp / 4][T][part][4]; inv[t] = 2^-e, nz[t] = any
// lo != 0.
__global__ __launch_bounds__(256) void x_split_kernel(const float* __restrict__ x, int xs, int K, int gs, int T, uint16_t* __restrict__ hi,
                                                      uint16_t* __restrict__ lo, void* __restrict__ gsum, float* __restrict__ inv,
                                                      int* __restrict__ nz) {
    extern __shared__ float xsp_part[];   // K / 8 chunk sums
    __shared__ float red[4];
    __shared__ int anyl;
    const int t = blockIdx.x, tid = threadIdx.x;
    const float* row = x + (int64_t)t * xs;
    if (tid == 0) anyl = 0;
    float mx = 0.0f;
    for (int c = tid; c < K / 8; c += 256) {
        const float4 a = reinterpret_cast<const float4*>(row)[2 * c], b = reinterpret_cast<const float4*>(row)[2 * c + 1];
        mx = fmaxf(mx, fmaxf(fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))),
                             fmaxf(fmaxf(fabsf(b.x), fabsf(b.y)), fmaxf(fabsf(b.z), fabsf(b.w)))));
    }
    mx = wave_max(mx);
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    int e = 0;
    if (mx > 0.0f && mx <= 3.0e38f) { frexpf(mx, &e); e = 14 - e; e = e < -126 ? -126 : (e > 126 ? 126 : e); }
    const float sc = ldexpf(1.0f, e);
    if (tid == 0) inv[t] = ldexpf(1.0f, -e);
    int any = 0;
    for (int c = tid; c < K / 8; c += 256) {
        const float4 a = reinterpret_cast<const float4*>(row)[2 * c], b = reinterpret_cast<const float4*>(row)[2 * c + 1];
        const float v[8] = {a.x * sc, a.y * sc, a.z * sc, a.w * sc, b.x * sc, b.y * sc, b.z * sc, b.w * sc};
        uint32_t h[4], l[4];
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint16_t h0 = f32_to_f16(v[2 * i]), h1 = f32_to_f16(v[2 * i + 1]);
            const uint16_t l0 = f32_to_f16(v[2 * i] - f16_to_f32(h0)), l1 = f32_to_f16(v[2 * i + 1] - f16_to_f32(h1));
            h[i] = (uint32_t)h0 | ((uint32_t)h1 << 16);
            l[i] = (uint32_t)l0 | ((uint32_t)l1 << 16);
            any |= (l[i] & 0x7FFF7FFFu) != 0;
        }
#pragma unroll
        for (int i = 0; i < 8; i++) sum += v[i];
        reinterpret_cast<uint4*>(hi + (int64_t)t * K)[c] = uint4{h[0], h[1], h[2], h[3]};
        reinterpret_cast<uint4*>(lo + (int64_t)t * K)[c] = uint4{l[0], l[1], l[2], l[3]};
        xsp_part[c] = sum;
    }
    if (any) anyl = 1;
    __syncthreads();
    const int cpg = gs >> 3, G = K / gs, Gp = gx_gpad(G);
    for (int g = tid; g < Gp; g += 256) {
        float s = 0.0f;
        if (g < G)
            for (int c = 0; c < cpg; c++) s += xsp_part[g * cpg + c];
        auto tr = [](float v) { return __uint_as_float(__float_as_uint(v) & 0xFFFF0000u); };
        const float vh = tr(s), r1 = s - vh, vm = tr(r1), vl = r1 - vm;
        uint16_t* o = static_cast<uint16_t*>(gsum) + ((int64_t)(g >> 2) * T + t) * 12 + (g & 3);
        o[0] = (uint16_t)(__float_as_uint(vh) >> 16); o[4] = (uint16_t)(__float_as_uint(vm) >> 16); o[8] = (uint16_t)(__float_as_uint(vl) >> 16);
    }
    if (tid == 0) nz[t] = anyl;
}

// Pre-pass: the scales and biases repacked to [Gp / 4][O][4] (s, then b; their stored 16-bit words,
// zero past G), so that 4 groups of 256 consecutive rows are 2 KB of consecutive bytes. A workgroup
// moves 64 rows x 64 groups through LDS: row-contiguous reads, chunk-contiguous writes.
__global__ __launch_bounds__(256) void scale_repack_kernel(const uint16_t* __restrict__ s, const uint16_t* __restrict__ b, int O, int G,
                                                            uint16_t* __restrict__ out) {
    __shared__ uint16_t tile[2][64][66];
    const int Gp = gx_gpad(G), nc = Gp / 4, tid = threadIdx.x;
    const int n0 = blockIdx.x * 64, g0 = blockIdx.y * 64;
#pragma unroll 4
    for (int i = 0; i < 16; i++) {
        const int idx = i * 256 + tid, r = idx >> 6, gl = idx & 63, n = n0 + r, g = g0 + gl;
        const bool in = n < O && g < G;
        tile[0][r][gl] = in ? s[(int64_t)n * G + g] : 0;
        tile[1][r][gl] = in ? b[(int64_t)n * G + g] : 0;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int idx = i * 256 + tid, cl = idx >> 6, r = idx & 63, c = g0 / 4 + cl, n = n0 + r;
        if (c >= nc || n >= O) continue;
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const uint16_t* t = &tile[p][r][4 * cl];
            reinterpret_cast<uint2*>(out)[(int64_t)p * nc * O + (int64_t)c * O + n] =
                uint2{(uint32_t)t[0] | ((uint32_t)t[1] << 16), (uint32_t)t[2] | ((uint32_t)t[3] << 16)};
        }
    }
}

// ---------------------------------------------------------------------------------------------
// The tile GEMM's operand pre-pass (f16, per-row power-of-two scale; used by ptile.hip's launcher).
__global__ __launch_bounds__(256) void x_to_f16_kernel(const float* x, int xs, int K, uint16_t* out, float* inv) {
    __shared__ float red[4];
    const int t = blockIdx.x, tid = threadIdx.x;
    const float* row = x + (int64_t)t * xs;
    float mx = 0.0f;
    for (int g = tid; g < K / 8; g += 256) {
        const float4 a = reinterpret_cast<const float4*>(row)[2 * g], b = reinterpret_cast<const float4*>(row)[2 * g + 1];
        mx = fmaxf(mx, fmaxf(fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))),
                             fmaxf(fmaxf(fabsf(b.x), fabsf(b.y)), fmaxf(fabsf(b.z), fabsf(b.w)))));
    }
    mx = wave_max(mx);
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    int e = 0;
    if (mx > 0.0f && mx <= 3.0e38f) { frexpf(mx, &e); e = 14 - e; e = e < -126 ? -126 : (e > 126 ? 126 : e); }
    const float sc = ldexpf(1.0f, e);
    if (tid == 0) inv[t] = ldexpf(1.0f, -e);
    for (int g = tid; g < K / 8; g += 256) {
        const float4 a = reinterpret_cast<const float4*>(row)[2 * g], b = reinterpret_cast<const float4*>(row)[2 * g + 1];
        uint4 o;
        o.x = (uint32_t)f32_to_f16(a.x * sc) | ((uint32_t)f32_to_f16(b.x * sc) << 16);
        o.y = (uint32_t)f32_to_f16(a.y * sc) | ((uint32_t)f32_to_f16(b.y * sc) << 16);
        o.z = (uint32_t)f32_to_f16(a.z * sc) | ((uint32_t)f32_to_f16(b.z * sc) << 16);
        o.w = (uint32_t)f32_to_f16(a.w * sc) | ((uint32_t)f32_to_f16(b.w * sc) << 16);
        reinterpret_cast<uint4*>(out + (int64_t)t * K)[g] = o;
    }
}

hipError_t launch_x_to_f16(const float* x, int xs, int K, int T, uint16_t* out, float* inv, hipStream_t s) {
    if (K % 8 || xs % 4 || T < 1) return hipErrorInvalidValue;
    if (launch_row_f16(x, xs, K, T, out, inv, s)) return hipGetLastError();
    hipLaunchKernelGGL(x_to_f16_kernel, dim3(T), dim3(256), 0, s, x, xs, K, out, inv);
    return hipGetLastError();
}


bool qgemm_supported(int K, int gs) { return K % GX_K == 0 && (gs == 32 || gs == 64 || gs == 128) && K % gs == 0; }

// Fixed K slices of a matrix: a function of its sizes alone, so a token's result never depends on T or on
// the launch's cut. As many as give a launch of few tokens a workgroup per CU (32 tokens x 128 rows), of at
// least 1024 inputs: a launch that walks them itself parks its running sum in y (3 us a slice and 8 bytes
// per output at 8 TB/s), so wide matrices, which need none for that, get none. No five or seven: a launch of
// middling T spreads them evenly over two, three or four workgroups a tile. From 8192 inputs on four or eight,
// unless wide: 27648 -> 16384 at 96 tokens takes 271 us in four slices, 427 in two; 27648 -> 7168 at 256 252 and, in
// five, 357; 27648 -> 4800 at 384 258 and, in six, 316 (4 bits).
static int qgemm_slices(int K, int O) {
    const int want = (33000 + O / 2) / O;
    if (K >= 8192) return want >= 8 ? 8 : want >= 2 ? 4 : 1;
    const int n = want < K / 1024 ? want : K / 1024;
    return n < 1 ? 1 : n == 5 || n == 7 ? n - 1 : n;
}

// The launch's tile shape and the workgroups per tile its slices are spread over, by expected time.
// Measured (us a 64-k block, one or more workgroups a CU): 128 x 256 tiles 2.05, one per CU; 64 x 128 1.3 alone,
// 1.05 each when a CU has several; 32 x 128 0.8 and 0.88; groups of 32 15% more. Over 13 matrices (3 .. 8 bits,
// 1664 .. 14336 inputs, 722 .. 28000 rows) at 16 .. 512 tokens its choice takes 1% more than the best of
// all cuts. 8 bits, 4096 -> 14336, 512 tokens: 128 x 256 unsplit 145 us (64 x 128: 216); 16 tokens: 32 x 128 in two
// slices 41 us (128 x 256 unsplit 142); 3 bits, 14336 -> 4096, 48 tokens: 64 x 128 in eight 58 us (616).
struct QGemmCut { int cut, S; };
struct QGemmKind { int tok, rows; double a, alone, shared; };
static const QGemmKind qgemm_kinds[] = {{GxBig::TOK, GxBig::NR, 14.0, 2.05, 0.0}, {GxMid::TOK, GxMid::NR, 12.0, 1.3, 1.05},
                                        {GxSmall::TOK, GxSmall::NR, 9.0, 0.8, 0.88}};
static size_t qgemm_tiles(const QGemmKind& k, int T, int O) { return (size_t)((T + k.tok - 1) / k.tok) * ((O + k.rows - 1) / k.rows); }
static bool qgemm_cut_fits(const QGemmKind& k, int T, int O, int SF, int S, bool split) {
    const size_t tiles = qgemm_tiles(k, T, O);
    return S == 1 || (S > 1 && S <= SF && split && tiles <= QGEMM_SPLIT_TILES && tiles * SF * k.tok * k.rows <= QGEMM_SPLIT_PART);
}
static QGemmCut qgemm_cut(int T, int K, int O, int gs, int SF, int cus, bool split) {
    QGemmCut best{0, 1};
    double bt = 1e30;
    for (int c = 0; c < 3; c++)
        for (int S = 1; S <= SF; S++) {
            const QGemmKind& k = qgemm_kinds[c];
            const size_t tiles = qgemm_tiles(k, T, O);
            if (!qgemm_cut_fits(k, T, O, SF, S, split)) continue;
            const double n = (double)(tiles * S) / cus, blocks = (double)K / GX_K * ((SF + S - 1) / S) / SF * (gs == 32 ? 1.15 : 1.0);
            double t = k.a + blocks * (c == 0 ? (double)((tiles * S + cus - 1) / cus) * k.alone : n * k.shared > k.alone ? n * k.shared : k.alone);
            if (S > 1) t += 6.0 + (double)(tiles * SF * k.tok * k.rows) * 8 / 4e6;
            else t += (SF - 1) * (3.0 + (double)T * O * 8 / 8e6);
            if (t < bt) { bt = t; best = QGemmCut{c, S}; }
        }
    return best;
}

hipError_t launch_qgemm(const QGemmArgs& a, hipStream_t s) {
    if (!qgemm_supported(a.K, a.gs) || a.T < 1 || !a.xbf || !a.xlo || !a.xgs || !a.xsc || !a.xnz || !a.wsb) return hipErrorInvalidValue;
    const int G = a.K / a.gs, Gp = gx_gpad(G);
    if (!a.x_ready) {
        hipLaunchKernelGGL(x_split_kernel, dim3(a.T), dim3(256), (size_t)(a.K / 8) * 4, s, a.x, a.x_stride, a.K, a.gs, a.T, a.xbf,
                           a.xlo, (void*)a.xgs, a.xsc, a.xnz);
        if (hipError_t e = hipGetLastError()) return e;
    }
    // scales and biases straight from the matrix where pairs of groups are whole dwords (repacking them
    // first cost 10 .. 12 us a call), else repacked
    const bool direct = G % 2 == 0 && ((reinterpret_cast<uintptr_t>(a.m.s) | reinterpret_cast<uintptr_t>(a.m.b)) & 3) == 0;
    if (!direct) {
        hipLaunchKernelGGL(scale_repack_kernel, dim3((unsigned)((a.m.O + 63) / 64), (unsigned)((Gp + 63) / 64)), dim3(256), 0, s, a.m.s, a.m.b,
                           a.m.O, G, a.wsb);
        if (hipError_t e = hipGetLastError()) return e;
    }
    QGemmXDev d{};
    d.w = a.m.w; d.s = direct ? a.m.s : a.wsb; d.b = a.m.b; d.bias = a.m.bias; d.st = a.st; d.direct = direct;
    d.K = a.K; d.O = a.O; d.T = a.T; d.ys = a.y_stride; d.SF = qgemm_slices(a.K, a.O);
    d.xh = a.xbf; d.xl = a.xlo; d.gsum = reinterpret_cast<const uint16_t*>(a.xgs); d.inv = a.xsc; d.nz = a.xnz; d.y = a.y;
    const int cus = device_cus();
    const bool split = a.split && a.split_floats >= QGEMM_SPLIT_FLOATS;
    QGemmCut q{a.cut, a.slices};
    if (a.cut < 0) q = qgemm_cut(a.T, a.K, a.O, a.gs, d.SF, cus, split);
    else if (a.cut > 2 || !qgemm_cut_fits(qgemm_kinds[a.cut], a.T, a.O, d.SF, a.slices, split)) return hipErrorInvalidValue;
    d.S = q.S;
    if (q.S > 1) { d.cnt = reinterpret_cast<unsigned*>(a.split); d.part = a.split + QGEMM_SPLIT_TILES; }
    switch (a.bits) {
        case 2: return qgemmx_launch2(d, a.gs, q.cut, s);
        case 3: return qgemmx_launch3(d, a.gs, q.cut, s);
        case 4: return qgemmx_launch4(d, a.gs, q.cut, s);
        case 5: return qgemmx_launch5(d, a.gs, q.cut, s);
        case 6: return qgemmx_launch6(d, a.gs, q.cut, s);
        case 8: return qgemmx_launch8(d, a.gs, q.cut, s);
    }
    return hipErrorInvalidValue;
}

// Scratch of the MLX-layout GEMM (per call): the x pre-pass' group sums (floats) and the repacked
// scales and biases (16-bit words).
size_t qgemm_gsum_floats(int T, int K, int gs) { return (size_t)T * gx_gpad(K / gs) / 4 * (GX_GSUM / 4); }
size_t qgemm_scale_halves(int O, int K, int gs) { return (size_t)2 * gx_gpad(K / gs) * O; }

}  // namespace mlxr
