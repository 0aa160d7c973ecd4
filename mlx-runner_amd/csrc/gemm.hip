// Host side and pre-passes of the MLX-layout GEMM (kernel: qgemmx.h, one file per code width), and the
// small batch (T <= 8) over the same layout.
#include "qgemmx.h"

namespace mlxr {

// Pre-pass: row t of x -> hi / lo (f16, [T][K]); gsum[g][t] (each group's sum of the scaled x,
// summed in k order per 8-chunk and chunks in order; zero past G); inv[t] = 2^-e, nz[t] = any
// lo != 0.
// BF3: the sums as three bf16 parts (truncations: hi + mid + lo exact) instead, [Gp / 4][T][part][4].
template <bool BF3>
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
        if constexpr (BF3) {
            auto tr = [](float v) { return __uint_as_float(__float_as_uint(v) & 0xFFFF0000u); };
            const float vh = tr(s), r1 = s - vh, vm = tr(r1), vl = r1 - vm;
            uint16_t* o = static_cast<uint16_t*>(gsum) + ((int64_t)(g >> 2) * T + t) * 12 + (g & 3);
            o[0] = (uint16_t)(__float_as_uint(vh) >> 16); o[4] = (uint16_t)(__float_as_uint(vm) >> 16); o[8] = (uint16_t)(__float_as_uint(vl) >> 16);
        } else {
            static_cast<float*>(gsum)[(int64_t)g * T + t] = s;
        }
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
// per output at 8 TB/s), so wide matrices, which need none for that, get none.
static int qgemm_slices(int K, int O) {
    const int want = (33000 + O / 2) / O, most = K / 1024 < 8 ? K / 1024 : 8;
    return want < 1 || most < 1 ? 1 : want < most ? want : most;
}

// The launch's tile shape and the workgroups per tile its slices are spread over, by expected time.
// Measured (us a 64-k block, one or more workgroups a CU): 128 x 256 tiles 2.05, one per CU; 64 x 128 1.3 alone,
// 1.05 each when a CU has several; 32 x 128 0.8 and 0.88; groups of 32 15% more. Over 13 matrices (3 .. 8 bits,
// 1664 .. 14336 inputs, 722 .. 28000 rows) at 16 .. 512 tokens its choice takes 1% more than the best of
// all cuts. 8 bits, 4096 -> 14336, 512 tokens: 128 x 256 unsplit 145 us (64 x 128: 216); 16 tokens: 32 x 128 in two
// slices 41 us (128 x 256 unsplit 142); 3 bits, 14336 -> 4096, 48 tokens: 64 x 128 in eight 58 us (616).
struct QGemmCut { int cut, S; };
static QGemmCut qgemm_cut(int T, int K, int O, int gs, int SF, int cus, bool split) {
    struct Kind { int tok, rows; double a, alone, shared; };
    static const Kind kinds[] = {{GxBig::TOK, GxBig::NR, 14.0, 2.05, 0.0}, {GxMid::TOK, GxMid::NR, 12.0, 1.3, 1.05},
                                 {GxSmall::TOK, GxSmall::NR, 9.0, 0.8, 0.88}};
    QGemmCut best{0, 1};
    double bt = 1e30;
    for (int c = 0; c < 3; c++)
        for (int S = 1; S <= SF; S++) {
            const Kind& k = kinds[c];
            const size_t tiles = (size_t)((T + k.tok - 1) / k.tok) * ((O + k.rows - 1) / k.rows);
            if (S > 1 && (!split || tiles > QGEMM_SPLIT_TILES || tiles * SF * k.tok * k.rows > QGEMM_SPLIT_PART)) continue;
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
        hipLaunchKernelGGL((x_split_kernel<true>), dim3(a.T), dim3(256), (size_t)(a.K / 8) * 4, s, a.x, a.x_stride, a.K, a.gs, a.T, a.xbf,
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
    static int cus = 0;
    if (!cus) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return hipErrorInvalidDevice;
    }
    const bool split = a.split && a.split_floats >= QGEMM_SPLIT_FLOATS;
    const QGemmCut q = qgemm_cut(a.T, a.K, a.O, a.gs, d.SF, cus, split);
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


// ---------------------------------------------------------------------------------------------
// Small batch (T <= 8) on the matrix cores, code widths 4 and 8: the same arithmetic as the GEMM
// above (exact codes, x as f16 hi + lo with a per-token power of two, scale and bias per group in
// fp32), shaped for a few tokens. v_mfma_f32_16x16x32_f16 with the tokens as the 16 A rows (rows
// past T zero) and 16 weight rows as the B columns, so each lane's accumulator holds its own
// weight row (its scale and bias load with its codes) for tokens 4 (lane / 16) .. + 3.
// A 1024-thread workgroup owns 16 rows; its 16 waves take a sixteenth of the groups each and add
// their partial sums in wave order. Lane quarter q takes codes GS/4 q .. + GS/4 - 1 of every
// group (the k order inside a group is free: the same for codes and x), so its codes are one
// contiguous load per group.
struct QmmXDev {
    const uint8_t* w[3]; const uint16_t* s[3]; const uint16_t* b[3]; const uint16_t* bias[3];
    int o1, o2, K, O, T, ys;
    const uint16_t* xh; const uint16_t* xl; const float* gsum; const float* inv; const int* nz; float* y;
};
constexpr int QX_WAVES = 4;

template <int BITS, int GS, int ST>
__global__ __launch_bounds__(256) void qmmx_kernel(QmmXDev a) {
    __shared__ f32x4_t red[QX_WAVES][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, q = lane >> 4, T = a.T;
    const int K = a.K, G = K / GS, g0 = G * wave / QX_WAVES, g1 = G * (wave + 1) / QX_WAVES;
    const int n = blockIdx.x * 16 + l16;   // the lane's weight row
    int row = min(n, a.O - 1), part = 0;
    if (row >= a.o1) {
        if (row < a.o1 + a.o2) { part = 1; row -= a.o1; }
        else { part = 2; row -= a.o1 + a.o2; }
    }
    const uint8_t* wp = a.w[part] + (int64_t)row * (K / 8 * BITS);
    const uint16_t* sp = a.s[part] + (int64_t)row * G;
    const uint16_t* bp = a.b[part] + (int64_t)row * G;
    const bool tok = l16 < T;                                   // A row l16: a token
    const int64_t xo = (int64_t)(tok ? l16 : 0) * K;
    // any token with lo parts (the loads issued together, not one round trip per token)
    int nzv[8];
#pragma unroll
    for (int t = 0; t < 8; t++) nzv[t] = a.nz[min(t, T - 1)];
    int lo = 0;
#pragma unroll
    for (int t = 0; t < 8; t++) lo |= nzv[t];
    constexpr int CPL = GS / 4, NS = GS / 32, DW = CPL * BITS / 32;
    constexpr int QX_NB = GS == 128 ? 2 : 4;   // groups per batch of loads
    f32x4_t tot = {0.0f, 0.0f, 0.0f, 0.0f};
    // groups in batches of QX_NB: every load of a batch is issued before any is used, so a wave
    // pays one memory round trip per batch
    for (int gb = g0; gb < g1; gb += QX_NB) {
        uint32_t cw[QX_NB][DW];
        float sv[QX_NB], bv[QX_NB], xs[QX_NB][4];
        half8_t ah[QX_NB][NS];
#pragma unroll
        for (int u = 0; u < QX_NB; u++) {
            const int g = min(gb + u, g1 - 1), k0 = g * GS + CPL * q;
            const uint32_t* cp = reinterpret_cast<const uint32_t*>(wp + k0 / 8 * BITS);
            if constexpr (DW % 4 == 0) {
#pragma unroll
                for (int i = 0; i < DW / 4; i++) {
                    const uint4 v = gload_u4(cp + 4 * i);
                    cw[u][4 * i] = v.x; cw[u][4 * i + 1] = v.y; cw[u][4 * i + 2] = v.z; cw[u][4 * i + 3] = v.w;
                }
            } else if constexpr (DW == 2) {
                const uint2 v = *reinterpret_cast<const uint2*>(cp);
                cw[u][0] = v.x; cw[u][1] = v.y;
            } else {
                cw[u][0] = cp[0];
            }
            sv[u] = ld_scale<ST>(sp + g) * 16777216.0f;
            bv[u] = ld_scale<ST>(bp + g);
#pragma unroll
            for (int i = 0; i < 4; i++) xs[u][i] = 4 * q + i < T ? a.gsum[(int64_t)g * T + 4 * q + i] : 0.0f;
#pragma unroll
            for (int st = 0; st < NS; st++)
                ah[u][st] = tok ? __builtin_bit_cast(half8_t, gload_u4(a.xh + xo + k0 + 8 * st)) : (half8_t)0;
        }
#pragma unroll
        for (int u = 0; u < QX_NB; u++) {
            if (gb + u >= g1) break;
            const int k0 = (gb + u) * GS + CPL * q;
            f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int st = 0; st < NS; st++) {
                half8_t bw;
                if constexpr (BITS == 4) {
                    const uint32_t ev = cw[u][st] & 0x0F0F0F0Fu, od = (cw[u][st] >> 4) & 0x0F0F0F0Fu;
                    bw = __builtin_bit_cast(half8_t, gx_u4{__builtin_amdgcn_perm(od, ev, 0x0C040C00u), __builtin_amdgcn_perm(od, ev, 0x0C050C01u),
                                                           __builtin_amdgcn_perm(od, ev, 0x0C060C02u), __builtin_amdgcn_perm(od, ev, 0x0C070C03u)});
                } else {
                    const uint32_t c0 = cw[u][2 * st], c1 = cw[u][2 * st + 1];
                    bw = __builtin_bit_cast(half8_t, gx_u4{__builtin_amdgcn_perm(0u, c0, 0x0C010C00u), __builtin_amdgcn_perm(0u, c0, 0x0C030C02u),
                                                           __builtin_amdgcn_perm(0u, c1, 0x0C010C00u), __builtin_amdgcn_perm(0u, c1, 0x0C030C02u)});
                }
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[u][st], bw, acc, 0, 0, 0);
                if (lo) {
                    const half8_t al = tok ? __builtin_bit_cast(half8_t, gload_u4(a.xl + xo + k0 + 8 * st)) : (half8_t)0;
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, bw, acc, 0, 0, 0);
                }
            }
#pragma unroll
            for (int i = 0; i < 4; i++) tot[i] = fmaf(sv[u], acc[i], fmaf(bv[u], xs[u][i], tot[i]));
        }
    }
    red[wave][lane] = tot;
    __syncthreads();
    if (wave != 0 || n >= a.O) return;
    f32x4_t sum = red[0][lane];
#pragma unroll
    for (int w = 1; w < QX_WAVES; w++) sum += red[w][lane];
    const float bias = a.bias[part] ? ld_scale<ST>(a.bias[part] + row) : 0.0f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int t = 4 * q + i;
        if (t < T) a.y[(int64_t)t * a.ys + n] = sum[i] * a.inv[t] + bias;
    }
}

// Small batch over the MLX layout with wide code loads (widths 4 and 8, groups of 8 * gs | K):
// the same operands and arithmetic as qmmx_kernel, laid out so that each lane's code load is 16
// bytes. A "span" is 64 bytes of one weight row (4 lanes x 16 bytes, 128 / BITS codes per lane);
// lane quarter q holds span bytes 16 q .. 16 q + 15, and MFMA step j takes its codes 8 j .. 8 j + 7,
// matched in the A operand by the same tokens' x at the same k. A span may hold several
// quantization groups (4-bit gs 32 / 64: lanes of one group are q, or q / 2); each group then runs
// its own MFMAs with the x of the other groups' lanes zeroed, so every accumulator holds one
// group and is folded with that group's scale and bias in fp32 (y += s 2^24 acc + b sum x).
// A batch is QY_NG groups of a row: its spans' codes, the 16-byte runs of scales and biases and
// every span's x are loaded before any is used (one memory round trip per batch); the token
// group sums sit in LDS. The x of a batch reaches LDS by buffer -> LDS copies (1 KB of 4 tokens'
// chunks per copy at 32 codes per lane, of 8 tokens' at 16; no lane loading what another lane
// loads) and the A operands are read from there. 16 rows per workgroup, the four waves on a quarter of the batches each,
// partial sums added in wave order.
template <int BITS, int GS> struct QyShape {
    static constexpr int C = BITS == 8 ? 16 : 32;        // codes per lane per span
    static constexpr int NDW = C * BITS / 32;            // their dwords (2, 3, 4 or 6)
    static constexpr int SPAN = 4 * C;                   // codes of a row per span
    static constexpr int NG = GS == 128 ? 4 : 8;         // groups per batch
    static constexpr int SPB = NG * GS / SPAN;           // spans per batch
    static constexpr int NGS = SPAN / GS;                // groups per span
    static constexpr int LPG = GS / C;                   // lane quarters per group
    static constexpr int STEPS = C / 8;                  // MFMA steps per span
};

template <int BITS, int GS, int ST, int NW, bool PF>
__global__ __launch_bounds__(64 * NW) void qmmy_kernel(QmmXDev a) {
    using S = QyShape<BITS, GS>;
    static_assert(S::SPAN >= GS && S::SPB >= 1, "span shape");
    // dynamic LDS: [G][8] token group sums (zero past T), then (32 codes per lane) each wave's x
    // buffers: per span, TT = T rounded up to 4 token rows of 256 bytes, 16-byte chunk c of token t
    // at slot c ^ t (a B-operand read of 16 tokens' same chunk hits distinct banks)
    extern __shared__ __attribute__((aligned(16))) float qy_gsum[];
    __shared__ f32x4_t red[NW][64];
    constexpr bool XL = true;                                  // x through LDS
    constexpr int NBUF = PF ? 2 : 1;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, q = lane >> 4, T = a.T;
    const int K = a.K, G = K / GS, NB = G / S::NG;
    // (a span's x per token: CPS chunks of 16 bytes, RB bytes; one copy carries TPI tokens)
    constexpr int CPS = S::SPAN / 8, TPI = 64 / CPS, RB = S::SPAN * 2;
    const int TT = (T + 3) & ~3, TTX = (T + TPI - 1) / TPI * TPI, XWB = S::SPB * TTX * RB;
    uint8_t* xlds = reinterpret_cast<uint8_t*>(qy_gsum) + (size_t)(K / GS) * 32;
    for (int i = tid; i < G * 8; i += 64 * NW) {
        const int g = i >> 3, t = i & 7;
        qy_gsum[i] = t < T ? a.gsum[(int64_t)g * T + t] : 0.0f;
    }
    const int n = blockIdx.x * 16 + l16;   // the lane's weight row
    int row = min(n, a.O - 1), part = 0;
    if (row >= a.o1) {
        if (row < a.o1 + a.o2) { part = 1; row -= a.o1; }
        else { part = 2; row -= a.o1 + a.o2; }
    }
    const uint8_t* wp = a.w[part] + (int64_t)row * (K / 8 * BITS) + 4 * S::NDW * q;
    const uint16_t* sp = a.s[part] + (int64_t)row * G;
    const uint16_t* bp = a.b[part] + (int64_t)row * G;
    const int TT0 = (T + 3) & ~3;
    const int64_t xo = (int64_t)min(S::NGS == 4 ? (int)(l16 % TT0) : l16, T - 1) * K + S::C * q;   // the token of A row l16
    int nzv[8];
#pragma unroll
    for (int t = 0; t < 8; t++) nzv[t] = a.nz[min(t, T - 1)];
    int lo = 0;
#pragma unroll
    for (int t = 0; t < 8; t++) lo |= nzv[t];
    const int gq = q / S::LPG;                                  // the lane's group within a span
    __syncthreads();
    const int b0 = NB * wave / NW, b1 = NB * (wave + 1) / NW;
    f32x4_t tot = {0.0f, 0.0f, 0.0f, 0.0f};
    // codes and scales of batch bt (every load unconditional, indices clamped: a load issued in a
    // branch would make the compiler's later waits count from zero)
    uint32_t cw[S::SPB][S::NDW];
    uint32_t sw[S::NG / 2], bw[S::NG / 2];
    auto load_w = [&](int bt) {
        bt = max(0, min(bt, NB - 1));
        const int k0 = bt * S::NG * GS;
#pragma unroll
        for (int u = 0; u < S::SPB; u++) {
            const uint8_t* p = wp + (int64_t)(k0 + u * S::SPAN) / 8 * BITS;
            if constexpr (S::NDW == 4) {
                const uint4 v = gload_u4(p);
                cw[u][0] = v.x; cw[u][1] = v.y; cw[u][2] = v.z; cw[u][3] = v.w;
            } else {
                typedef const __attribute__((address_space(1))) uint32_t* gp32;
#pragma unroll
                for (int i = 0; i < S::NDW; i++) cw[u][i] = *((gp32)p + i);
            }
        }
        if constexpr (S::NG == 8) {
            const uint4 s4 = gload_u4(sp + S::NG * bt), b4 = gload_u4(bp + S::NG * bt);
            sw[0] = s4.x; sw[1] = s4.y; sw[2] = s4.z; sw[3] = s4.w;
            bw[0] = b4.x; bw[1] = b4.y; bw[2] = b4.z; bw[3] = b4.w;
        } else {
            const uint2 s2 = *reinterpret_cast<const uint2*>(sp + S::NG * bt), b2 = *reinterpret_cast<const uint2*>(bp + S::NG * bt);
            sw[0] = s2.x; sw[1] = s2.y; bw[0] = b2.x; bw[1] = b2.y;
        }
    };
    // x of batch bt into LDS buffer buf by buffer -> LDS copies: per span and 4 tokens one 1 KB copy,
    // lane i: token 4 tq + i / 16, chunk (i & 15) ^ token (rows past T repeat row T - 1, unread)
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.xh), 0, T * K * 2, 0x00020000);
    auto dma_x = [&](int bt, int buf) {
        bt = max(0, min(bt, NB - 1));
        const int k0 = bt * S::NG * GS;
        uint8_t* rb = xlds + (size_t)(wave * NBUF + buf) * XWB;
#pragma unroll
        for (int u = 0; u < S::SPB; u++)
            for (int tq = 0; tq < TTX / TPI; tq++) {
                const int t = TPI * tq + lane / CPS, c = (lane % CPS) ^ (t & (CPS - 1));
                const uint32_t off = (uint32_t)(min(t, T - 1) * K + k0 + u * S::SPAN + 8 * c) * 2u;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (__attribute__((address_space(3))) void*)(rb + (u * TTX + TPI * tq) * RB), 16, off, 0, 0, 0);
            }
    };
    // A rows: NGP = 16 / TT group slots of TT token rows; row l16 is token ta of slot pa. D rows
    // 4 q .. 4 q + 3: tokens td0 .. td0 + 3 of slot pd. One MFMA set covers NGP groups of a span.
    // (PACK: spans of four groups; otherwise one slot: row l16 is token l16, D rows tokens 4 q ..)
    constexpr bool PACK = S::NGS == 4;
    const int NGP = PACK ? 16 / TT : 1, pa = PACK ? l16 / TT : 0, ta = PACK ? l16 % TT : l16;
    const int pd = PACK ? (4 * q) / TT : 0, td0 = PACK ? (4 * q) % TT : 4 * q;
    const bool tva = ta < T;
    const int mr = min(ta, TTX - 1);
    if constexpr (PF) {
        load_w(b0);
        if constexpr (XL) dma_x(b0, 0);
    }
    for (int bt = b0; bt < b1; bt++) {
        const int k0 = bt * S::NG * GS;
        if constexpr (!PF) {
            load_w(bt);
            if constexpr (XL) dma_x(bt, 0);
        }
        half8_t xv[S::SPB][S::STEPS];
        if constexpr (XL) {
            // this batch's copies (and codes) have landed
            __builtin_amdgcn_s_waitcnt(0x0F70);
            asm volatile("" ::: "memory");
            const uint8_t* rb = xlds + (size_t)(wave * NBUF + (PF ? (bt - b0) & 1 : 0)) * XWB;
#pragma unroll
            for (int u = 0; u < S::SPB; u++)
#pragma unroll
                for (int j = 0; j < S::STEPS; j++) {
                    const half8_t v = *reinterpret_cast<const half8_t*>(rb + (u * TTX + mr) * RB + (((S::C / 8) * q + j) ^ (mr & (CPS - 1))) * 16);
                    xv[u][j] = tva ? v : (half8_t)0;
                }
        } else {
#pragma unroll
            for (int u = 0; u < S::SPB; u++)
#pragma unroll
                for (int j = 0; j < S::STEPS; j++) {
                    const half8_t v = __builtin_bit_cast(half8_t, gload_u4(a.xh + xo + k0 + u * S::SPAN + 8 * j));
                    xv[u][j] = tva ? v : (half8_t)0;
                }
        }
        // this batch's codes and scales into their own registers; with PF (waves of three or more
        // batches) the next batch's stream in behind
        uint32_t cur[S::SPB][S::NDW];
        uint32_t scur[S::NG / 2], bcur[S::NG / 2];
#pragma unroll
        for (int u = 0; u < S::SPB; u++)
#pragma unroll
            for (int i = 0; i < S::NDW; i++) cur[u][i] = cw[u][i];
#pragma unroll
        for (int i = 0; i < S::NG / 2; i++) { scur[i] = sw[i]; bcur[i] = bw[i]; }
        if constexpr (PF) {
            load_w(bt + 1);
            if constexpr (XL) dma_x(bt + 1, (bt + 1 - b0) & 1);
        }
#pragma unroll
        for (int u = 0; u < S::SPB; u++) {
#define cd cur[u]
            half8_t wv[S::STEPS], xl[S::STEPS];
#pragma unroll
            for (int j = 0; j < S::STEPS; j++) {
                if constexpr (BITS == 4) {
                    const uint32_t ev = cd[j] & 0x0F0F0F0Fu, od = (cd[j] >> 4) & 0x0F0F0F0Fu;
                    wv[j] = __builtin_bit_cast(half8_t, gx_u4{__builtin_amdgcn_perm(od, ev, 0x0C040C00u), __builtin_amdgcn_perm(od, ev, 0x0C050C01u),
                                                              __builtin_amdgcn_perm(od, ev, 0x0C060C02u), __builtin_amdgcn_perm(od, ev, 0x0C070C03u)});
                } else if constexpr (BITS == 8) {
                    const uint32_t c0 = cd[2 * j], c1 = cd[2 * j + 1];
                    wv[j] = __builtin_bit_cast(half8_t, gx_u4{__builtin_amdgcn_perm(0u, c0, 0x0C010C00u), __builtin_amdgcn_perm(0u, c0, 0x0C030C02u),
                                                              __builtin_amdgcn_perm(0u, c1, 0x0C010C00u), __builtin_amdgcn_perm(0u, c1, 0x0C030C02u)});
                } else {
                    // codes 8 j .. 8 j + 7: bits 8 BITS j .. + 8 BITS of the lane's little-endian stream
                    const int b = 8 * BITS * j, i0 = b >> 5, sh = b & 31;
                    const uint64_t w = ((uint64_t)(i0 + 1 < S::NDW ? cd[i0 + 1] : 0u) << 32 | cd[i0]) >> sh;
                    constexpr uint32_t m = (1u << BITS) - 1;
                    uint32_t h[4];
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        h[e] = ((uint32_t)(w >> (2 * e * BITS)) & m) | (((uint32_t)(w >> ((2 * e + 1) * BITS)) & m) << 16);
                    wv[j] = __builtin_bit_cast(half8_t, gx_u4{h[0], h[1], h[2], h[3]});
                }
                xl[j] = (half8_t)0;
                if (lo && tva) xl[j] = __builtin_bit_cast(half8_t, gload_u4(a.xl + xo + k0 + u * S::SPAN + 8 * j));
            }
#undef cd
#pragma unroll
            for (int set = 0; set < S::NGS; set++) {
                if (PACK && set * NGP >= S::NGS) break;
                // A row l16 carries group set * NGP + pa: the x of the lanes holding that group's codes
                const bool mine = S::NGS == 1 || set * NGP + pa == gq;
                f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int j = 0; j < S::STEPS; j++) {
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(mine ? xv[u][j] : (half8_t)0, wv[j], acc, 0, 0, 0);
                    if (lo) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(mine ? xl[j] : (half8_t)0, wv[j], acc, 0, 0, 0);
                }
                // this lane's D rows: group set * NGP + pd of the span, tokens td0 ..
                const int gs_ = set * NGP + pd;
                const bool live = !PACK || gs_ < S::NGS;
                const int gb = u * S::NGS + min(gs_, S::NGS - 1);   // group within the batch
                uint32_t sd = scur[0], bd = bcur[0];
                if constexpr (PACK) {
#pragma unroll
                    for (int i = 1; i < S::NG / 2; i++)
                        if ((gb >> 1) == i) { sd = scur[i]; bd = bcur[i]; }
                } else {
                    sd = scur[gb >> 1]; bd = bcur[gb >> 1];
                }
                const uint32_t sr = (sd >> (16 * (gb & 1))) & 0xFFFFu, br = (bd >> (16 * (gb & 1))) & 0xFFFFu;
                const float sv = live ? (ST == 0 ? __uint_as_float(sr << 16) : f16_to_f32((uint16_t)sr)) * 16777216.0f : 0.0f;
                const float bv = live ? (ST == 0 ? __uint_as_float(br << 16) : f16_to_f32((uint16_t)br)) : 0.0f;
                const f32x4_t xs = *reinterpret_cast<const f32x4_t*>(qy_gsum + (bt * S::NG + gb) * 8 + td0);
#pragma unroll
                for (int i = 0; i < 4; i++) tot[i] = fmaf(sv, acc[i], fmaf(bv, xs[i], tot[i]));
            }
        }
    }
    red[wave][lane] = tot;
    __syncthreads();
    // the lanes of slot 0 add every wave's and every slot's partial sums of their tokens, in order
    if (wave != 0 || pd != 0 || n >= a.O) return;
    f32x4_t sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < NW; w++)
        for (int p = 0; p < NGP; p++) sum += red[w][lane + 16 * p * (TT / 4)];
    const float bias = a.bias[part] ? ld_scale<ST>(a.bias[part] + row) : 0.0f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int t = td0 + i;
        if (t < T) a.y[(int64_t)t * a.ys + n] = sum[i] * a.inv[t] + bias;
    }
}

// qmmy_kernel's shapes: widths 2 / 3 / 4 / 6 at gs 32 / 64 / 128, 8-bit at gs 32 / 64; K a multiple of
// a batch; the group sums' LDS within 64 KiB
static bool qmmy_supported(int K, int bits, int gs) {
    const bool b32 = bits == 2 || bits == 3 || bits == 4 || bits == 6;   // 32 codes per lane
    if (!((b32 && (gs == 32 || gs == 64 || gs == 128)) || (bits == 8 && (gs == 32 || gs == 64)))) return false;
    const int ng = gs == 128 ? 4 : 8;
    return K % (ng * gs) == 0 && (size_t)(K / gs) * 32 <= 65536;
}

bool qmmx_supported(int K, int bits, int gs) {
    if (qmmy_supported(K, bits, gs)) return true;
    return (bits == 4 || bits == 8) && (gs == 32 || gs == 64 || gs == 128) && K % gs == 0 && K % 32 == 0;
}

hipError_t launch_qmmx(const QmmSmallArgs& a, hipStream_t s) {
    if (!qmmx_supported(a.K, a.bits, a.gs) || a.T < 1 || a.T > 8 || !a.xbf || !a.xlo || !a.xgs || !a.xsc || !a.xnz)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL((x_split_kernel<false>), dim3(a.T), dim3(256), (size_t)(a.K / 8) * 4, s, a.x, a.x_stride, a.K, a.gs, a.T, a.xbf, a.xlo,
                       a.xgs, a.xsc, a.xnz);
    if (hipError_t e = hipGetLastError()) return e;
    QmmXDev d{};
    for (int i = 0; i < 3; i++) {
        const QMat& m = a.part[i < a.nparts ? i : a.nparts - 1];
        d.w[i] = m.w; d.s[i] = m.s; d.b[i] = m.b; d.bias[i] = m.bias;
    }
    d.o1 = a.part[0].O; d.o2 = a.nparts > 1 ? a.part[1].O : 0;
    d.K = a.K; d.O = a.O; d.T = a.T; d.ys = a.y_stride;
    d.xh = a.xbf; d.xl = a.xlo; d.gsum = a.xgs; d.inv = a.xsc; d.nz = a.xnz; d.y = a.y;
    const dim3 grid((unsigned)((a.O + 15) / 16));
    if (qmmy_supported(a.K, a.bits, a.gs)) {
        // eight waves (an eighth of the batches each) where a quarter of the batches would be a
        // long chain per wave; the next batch's loads in flight behind each batch where a wave has
        // three or more; LDS: group sums, then (32 codes per lane) every wave's x buffers
        const int ng = a.gs == 128 ? 4 : 8, nb = a.K / a.gs / ng;
        bool w8 = nb >= 16, pf = nb / (w8 ? 8 : 4) >= 3;
        const int C = a.bits == 8 ? 16 : 32, spb = ng * a.gs / (4 * C), tpi = 64 / (C / 2), tt = (a.T + tpi - 1) / tpi * tpi;
        auto lds_of = [&](bool w, bool p) {
            return (size_t)(a.K / a.gs) * 32 + (size_t)(w ? 8 : 4) * (p ? 2 : 1) * spb * tt * (8 * C);
        };
        // (160 KiB of LDS less the 8 KiB of the waves' partial sums)
        constexpr size_t QY_LDS_MAX = 152 * 1024;
        if (lds_of(w8, pf) > QY_LDS_MAX) w8 = pf = false;
        const size_t lds = lds_of(w8, pf);
        if (lds > QY_LDS_MAX) return hipErrorInvalidValue;
        static bool attr = false;
        if (!attr) {
#define QMMY_ATTR1(B, GS, ST) \
            for (const void* f : {(const void*)qmmy_kernel<B, GS, ST, 8, true>, (const void*)qmmy_kernel<B, GS, ST, 8, false>, \
                                  (const void*)qmmy_kernel<B, GS, ST, 4, false>}) \
                if (hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)QY_LDS_MAX)) return e;
#define QMMY_ATTR(B) QMMY_ATTR1(B, 32, 0) QMMY_ATTR1(B, 64, 0) QMMY_ATTR1(B, 128, 0) QMMY_ATTR1(B, 32, 1) QMMY_ATTR1(B, 64, 1) QMMY_ATTR1(B, 128, 1)
            QMMY_ATTR(2) QMMY_ATTR(3) QMMY_ATTR(4) QMMY_ATTR(6)
            QMMY_ATTR1(8, 32, 0) QMMY_ATTR1(8, 64, 0) QMMY_ATTR1(8, 32, 1) QMMY_ATTR1(8, 64, 1)
#undef QMMY_ATTR
#undef QMMY_ATTR1
            attr = true;
        }
#define QMMY_GO(B, GS) if (a.bits == B && a.gs == GS) { \
        if (w8 && pf) { \
            if (a.st == 0) hipLaunchKernelGGL((qmmy_kernel<B, GS, 0, 8, true>), grid, dim3(512), lds, s, d); \
            else hipLaunchKernelGGL((qmmy_kernel<B, GS, 1, 8, true>), grid, dim3(512), lds, s, d); \
        } else if (w8) { \
            if (a.st == 0) hipLaunchKernelGGL((qmmy_kernel<B, GS, 0, 8, false>), grid, dim3(512), lds, s, d); \
            else hipLaunchKernelGGL((qmmy_kernel<B, GS, 1, 8, false>), grid, dim3(512), lds, s, d); \
        } else { \
            if (a.st == 0) hipLaunchKernelGGL((qmmy_kernel<B, GS, 0, 4, false>), grid, dim3(256), lds, s, d); \
            else hipLaunchKernelGGL((qmmy_kernel<B, GS, 1, 4, false>), grid, dim3(256), lds, s, d); \
        } \
        return hipGetLastError(); }
        QMMY_GO(2, 32) QMMY_GO(2, 64) QMMY_GO(2, 128) QMMY_GO(3, 32) QMMY_GO(3, 64) QMMY_GO(3, 128)
        QMMY_GO(4, 32) QMMY_GO(4, 64) QMMY_GO(4, 128) QMMY_GO(6, 32) QMMY_GO(6, 64) QMMY_GO(6, 128)
        QMMY_GO(8, 32) QMMY_GO(8, 64)
#undef QMMY_GO
    }
#define QMMX_GO(B, GS) if (a.bits == B && a.gs == GS) { \
        if (a.st == 0) hipLaunchKernelGGL((qmmx_kernel<B, GS, 0>), grid, dim3(64 * QX_WAVES), 0, s, d); \
        else hipLaunchKernelGGL((qmmx_kernel<B, GS, 1>), grid, dim3(64 * QX_WAVES), 0, s, d); \
        return hipGetLastError(); }
    QMMX_GO(4, 32) QMMX_GO(4, 64) QMMX_GO(4, 128) QMMX_GO(8, 32) QMMX_GO(8, 64) QMMX_GO(8, 128)
#undef QMMX_GO
    return hipErrorInvalidValue;
}

}  // namespace mlxr
