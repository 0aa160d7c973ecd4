// Small batch (T <= 8) over MLX affine-quantized weights on the matrix cores.
//
// Semantics: the reference's generic `qmm` (Kernels.swift:60-113): y[t][o] = sum over groups of
// s * (sum_j q_j x_tj) + b * (sum_j x_tj), rows of up to three matrices [A | B | C], optional row bias.
//
// MI355X layout: v_mfma_f32_16x16x32_f16 with the tokens as A rows, x as f16 hi parts in rows 0-7 and lo
// parts in rows 8-15 (x = hi + lo to ~2^-22 after a power-of-two scaling of the token's slice), and 16 weight
// rows as B columns, so one instruction does both parts and each lane folds its own weight row's scale and
// bias, once per group, in fp32. Codes enter as exact f16 integers (a code OR-ed into the mantissa of 1024,
// then 1024 subtracted, 2 codes an instruction).
// A workgroup of four waves takes 64 RT rows and a range of the K chunks (256 codes); each wave RT tiles of
// 16 rows. The range's x is converted once per workgroup, slices of four chunks at a time, into LDS in the
// A operand's own order ([step of 32 codes][16-byte slot per lane]), together with the groups' sums; the
// waves then stream their codes straight to registers, DEPTH chunks ahead, without barriers in a slice.
// Lane quarter q reads 64 consecutive codes of its row per chunk (8 BITS bytes: whole cache lines for a row's
// four lanes) and the quarters exchange them by lane swaps, so that an instruction's four quarters hold one
// group (reading each group's quarters in place, 2 BITS bytes per lane, ran at the same 117 us for 5120 -> 17000
// at gs 32 whatever the width: the cache's lines per instruction bound it).
// Ranges of K (where the rows alone leave the chip idle) meet in the scratch: the last workgroup of a row block
// adds them in order.
// What bounds it now: the vector work per chunk (code conversion, exchange, folds: ~250 instructions per wave
// and 4 KB of 16 x 256 codes) and, at few rows, the chain x load -> conversion -> first chunk (~6 us).
// Against a pre-pass launch and a kernel of 16 rows per workgroup with x through LDS per wave (us, T = 4):
// 4096 -> 14336 at 8 bits 32.7 -> 22.0, 14336 -> 4096 at 6 bits 41.5 -> 20.1, 14336 -> 512 at 4 bits 27.7 -> 10.6,
// 1024 -> 512 at 4 bits 9.3 -> 7.6; without the exchange 4096 -> 30000 at 3 bits took 33.9, with it 31.
#include "qgemm.h"

namespace mlxr {

constexpr int QB_CH = 256;     // codes per chunk
constexpr int QB_SL = 4;       // chunks per slice of x in LDS
constexpr int QB_RT = 4;       // 16-row tiles per wave (max)

struct QbDev {
    const uint8_t* w[3]; const uint16_t* s[3]; const uint16_t* b[3]; const uint16_t* bias[3];
    int o1, o2, K, O, T, xs, ys, nb, S, RT;
    const float* x; float* y;
    unsigned* cnt; float* part;     // S > 1: row-block counters (zero between launches), partial sums [S][T][O]
};

typedef _Float16 qb_h2 __attribute__((ext_vector_type(2)));
typedef float qb_f2 __attribute__((ext_vector_type(2)));

template <int BITS, int GS> struct QbShape {
    static constexpr int GC = QB_CH / GS;                  // groups per chunk
    static constexpr int NDW = 2 * BITS;                   // dwords of a lane's 64 codes of a chunk
    static constexpr int NSC = GS == 32 ? 2 : 1;           // their scales
    static constexpr int DEPTH = BITS == 8 ? 2 : 3;        // chunks of codes in flight
};

// N consecutive dwords (4-byte aligned)
template <int N>
__device__ __forceinline__ void qb_load(const uint8_t* p, uint32_t* d) {
    typedef uint32_t v2 __attribute__((ext_vector_type(2), aligned(4)));
    typedef uint32_t v3 __attribute__((ext_vector_type(3), aligned(4)));
    typedef uint32_t v4 __attribute__((ext_vector_type(4), aligned(4)));
    if constexpr (N >= 4) {
        const v4 v = *(const __attribute__((address_space(1))) v4*)p;
        d[0] = v.x; d[1] = v.y; d[2] = v.z; d[3] = v.w;
        if constexpr (N > 4) qb_load<N - 4>(p + 16, d + 4);
    } else if constexpr (N == 3) {
        const v3 v = *(const __attribute__((address_space(1))) v3*)p;
        d[0] = v.x; d[1] = v.y; d[2] = v.z;
    } else if constexpr (N == 2) {
        const v2 v = *(const __attribute__((address_space(1))) v2*)p;
        d[0] = v.x; d[1] = v.y;
    } else {
        d[0] = *(const __attribute__((address_space(1))) uint32_t*)p;
    }
}

// Two codes at bit P of each half of e (P + BITS <= 10) as f16 integers.
template <int BITS, int P>
__device__ __forceinline__ uint32_t qb_pair(uint32_t e) {
    constexpr uint32_t m = ((1u << BITS) - 1) << P;
    const qb_h2 r = __builtin_bit_cast(qb_h2, (e & (m | m << 16)) | 0x64006400u);
    constexpr float f = 1.0f / (1 << P);
    const qb_h2 o = {(_Float16)(-1024.0f * f), (_Float16)(-1024.0f * f)};
    if constexpr (P == 0) return __builtin_bit_cast(uint32_t, r + o);
    const qb_h2 k = {(_Float16)f, (_Float16)f};
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(r, k, o));
}

// Codes 8 j .. 8 j + 7 of a lane's piece (d: its dwords from bit 0) as a B operand, in the order 0 4 1 5 2 6 3 7
// (8 bits: in order).
template <int BITS, int N>
__device__ __forceinline__ half8_t qb_codes(const uint32_t* d, int j) {
    const int i = BITS * j >> 2, sh = 8 * (BITS * j & 3);
    auto at = [&](int n) { return n < N ? d[n] : 0u; };
    const uint32_t w0 = sh ? __builtin_amdgcn_alignbit(at(i + 1), at(i), sh) : at(i);
    const uint32_t w1 = BITS > 4 ? (sh ? __builtin_amdgcn_alignbit(at(i + 2), at(i + 1), sh) : at(i + 1)) : 0u;
    gx_u4 v;
    if constexpr (BITS == 2) {
        const uint32_t e = __builtin_amdgcn_perm(0u, w0, 0x0C010C00u);
        v = gx_u4{qb_pair<2, 0>(e), qb_pair<2, 2>(e), qb_pair<2, 4>(e), qb_pair<2, 6>(e)};
    } else if constexpr (BITS == 3) {
        const uint32_t e = __builtin_amdgcn_perm(w0 >> 12, w0, 0x05040100u);
        v = gx_u4{qb_pair<3, 0>(e), qb_pair<3, 3>(e), qb_pair<3, 6>(e), qb_pair<3, 0>(e >> 9)};
    } else if constexpr (BITS == 4) {
        v = gx_u4{qb_pair<4, 0>(w0), qb_pair<4, 4>(w0), qb_pair<4, 0>(w0 >> 8), qb_pair<4, 4>(w0 >> 8)};
    } else if constexpr (BITS == 6) {
        const uint32_t e0 = __builtin_amdgcn_perm(w1, w0, 0x04030100u), e1 = __builtin_amdgcn_perm(w1, w0, 0x05040201u);
        v = gx_u4{qb_pair<6, 0>(e0), qb_pair<6, 0>(e0 >> 6), qb_pair<6, 4>(e1), qb_pair<6, 0>(e1 >> 10)};
    } else {
        const qb_h2 o = {(_Float16)-1024.0f, (_Float16)-1024.0f};
        auto two = [&](uint32_t w, uint32_t sel) {
            return __builtin_bit_cast(uint32_t, __builtin_bit_cast(qb_h2, __builtin_amdgcn_perm(0x64646464u, w, sel)) + o);
        };
        v = gx_u4{two(w0, 0x04010400u), two(w0, 0x04030402u), two(w1, 0x04010400u), two(w1, 0x04030402u)};
    }
    return __builtin_bit_cast(half8_t, v);
}

// m[r] of quarter q to m[q] of quarter r (a quarter: 16 lanes).
__device__ __forceinline__ void qb_transpose(uint32_t (&m)[4]) {
    const auto a = __builtin_amdgcn_permlane32_swap(m[0], m[2], false, false), b = __builtin_amdgcn_permlane32_swap(m[1], m[3], false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false), d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    m[0] = c[0]; m[1] = c[1]; m[2] = d[0]; m[3] = d[1];
}

template <int BITS, int GS, int ST>
__global__ __launch_bounds__(256, 3) void qmb_kernel(QbDev a) {
    using H = QbShape<BITS, GS>;
    constexpr int DEPTH = H::DEPTH;
    __shared__ __attribute__((aligned(1024))) uint8_t xl[QB_SL * 8192];      // [step][quarter][16 rows] x 16 bytes, rows ^ (4 step + quarter)
    __shared__ __attribute__((aligned(16))) float gsum[QB_SL * H::GC][16];    // the scaled x's group sums (rows 8-15: 0)
    __shared__ __attribute__((aligned(16))) float inv[16];
    extern __shared__ __attribute__((aligned(16))) f32x4_t qb_tot[];         // [RT][256]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, q = lane >> 4, T = a.T, K = a.K, G = K / GS, RT = a.RT;
    const int blk = (int)blockIdx.x % a.nb, z = (int)blockIdx.x / a.nb;
    const int C = (K + QB_CH - 1) / QB_CH, c0 = C * z / a.S, c1 = C * (z + 1) / a.S;
    const int row0 = blk * 64 * RT + 16 * wave + l16;                        // this lane's weight row of tile 0

    // x of chunks [cs, cs + QB_SL): token t = wave, wave + 4; lane: 8 values at 8 (lane + 64 u)
    float4 xv[2][QB_SL / 2][2];
    auto load_x = [&](int cs) {
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int u = 0; u < QB_SL / 2; u++) {
                if (4 * h >= T) continue;
                const int t = wave + 4 * h, k = cs * QB_CH + 8 * (lane + 64 * u);
                const float* p = a.x + (int64_t)min(t, T - 1) * a.xs + min(k, K - 8);   // (zeroed in convert_x)
                xv[h][u][0] = gload4(p); xv[h][u][1] = gload4(p + 4);
            }
    };
    auto convert_x = [&](int cs) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int t = wave + 4 * h;
            if (t >= T && cs != c0) continue;     // rows past T: zeros, written once
            float mx = 0.0f;
#pragma unroll
            for (int u = 0; u < QB_SL / 2; u++)
                if (t >= T || cs * QB_CH + 8 * (lane + 64 * u) >= K) xv[h][u][0] = xv[h][u][1] = float4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int u = 0; u < QB_SL / 2; u++)
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const float4 v = xv[h][u][e];
                    mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
                }
            mx = wave_max(mx);
            int e = 0;
            if (mx > 0.0f && mx <= 3.0e38f) { frexpf(mx, &e); e = 14 - e; e = e < -126 ? -126 : (e > 126 ? 126 : e); }
            const float sc = ldexpf(1.0f, e);
            if (lane < 2) inv[t + 8 * lane] = ldexpf(1.0f, -e);
#pragma unroll
            for (int u = 0; u < QB_SL / 2; u++) {
                const int kk = 8 * (lane + 64 * u);
                const int step = GS == 32 ? kk / 32 : 2 * (kk / 64) + kk / 8 % 2, sq = GS == 32 ? kk / 8 % 4 : kk / 16 % 4;
                const float4 va = xv[h][u][0], vb = xv[h][u][1];
                const float v[8] = {va.x * sc, va.y * sc, va.z * sc, va.w * sc, vb.x * sc, vb.y * sc, vb.z * sc, vb.w * sc};
                uint32_t hw[4], lw[4];
                float sum = 0.0f;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float x0 = BITS == 8 ? v[2 * i] : v[i], x1 = BITS == 8 ? v[2 * i + 1] : v[i + 4];
                    const qb_h2 h = __builtin_convertvector((qb_f2{x0, x1}), qb_h2);
                    const qb_h2 l = {(_Float16)(x0 - (float)h[0]), (_Float16)(x1 - (float)h[1])};
                    hw[i] = __builtin_bit_cast(uint32_t, h);
                    lw[i] = __builtin_bit_cast(uint32_t, l);
                }
#pragma unroll
                for (int i = 0; i < 8; i++) sum += v[i];
                uint8_t* p = xl + step * 1024 + sq * 256;
                const int f = (4 * step + sq) & 15;
                *reinterpret_cast<uint4*>(p + 16 * (t ^ f)) = uint4{hw[0], hw[1], hw[2], hw[3]};
                *reinterpret_cast<uint4*>(p + 16 * ((t + 8) ^ f)) = uint4{lw[0], lw[1], lw[2], lw[3]};
                sum = quad_sum(sum);
                if constexpr (GS >= 64) sum += dpp<0x141>(sum);
                if constexpr (GS >= 128) sum += dpp<0x140>(sum);
                if (lane % (GS / 8) == 0) { gsum[kk / GS][t] = sum; gsum[kk / GS][t + 8] = 0.0f; }
            }
        }
    };

    // load cursor: slice [lcs, lcs + ln), tile lrt, chunk lc of the slice
    int lcs = c0, ln = min(QB_SL, c1 - c0), lrt = 0, lc = 0;
    const uint8_t* wp; const uint16_t* sp; const uint16_t* bp;
    // (distances added under a mask: an index by the part would be a load, and its wait one for all in flight)
    const uint64_t w0 = (uint64_t)a.w[0], w1 = (uint64_t)a.w[1] - w0, w2 = (uint64_t)a.w[2] - (uint64_t)a.w[1];
    const uint64_t sc0 = (uint64_t)a.s[0], sc1 = (uint64_t)a.s[1] - sc0, sc2 = (uint64_t)a.s[2] - (uint64_t)a.s[1];
    const uint64_t bi0 = (uint64_t)a.b[0], bi1 = (uint64_t)a.b[1] - bi0, bi2 = (uint64_t)a.b[2] - (uint64_t)a.b[1];
    const int o1 = a.o1, o2 = a.o2, O1 = a.O - 1;
    auto row_ptrs = [&](int rt) {
        int row = min(row0 + 64 * rt, O1);
        const uint64_t p1 = row >= o1 ? ~0ull : 0ull, p2 = row >= o1 + o2 ? ~0ull : 0ull;
        row -= (int)(p1 & (uint64_t)o1) + (int)(p2 & (uint64_t)o2);
        wp = (const uint8_t*)(w0 + (p1 & w1) + (p2 & w2)) + (int64_t)row * (K / 8 * BITS);
        sp = (const uint16_t*)(sc0 + (p1 & sc1) + (p2 & sc2)) + (int64_t)row * G;
        bp = (const uint16_t*)(bi0 + (p1 & bi1) + (p2 & bi2)) + (int64_t)row * G;
    };
    uint32_t cw[DEPTH][H::NDW];
    uint16_t sw[DEPTH][H::NSC], bw[DEPTH][H::NSC];
    auto load_w = [&](int d) {
        const int piece = min(4 * (lcs + lc) + q, K / 64 - 1);
#pragma unroll
        for (int i = 0; i < H::NSC; i++) {
            const int g = GS == 128 ? piece / 2 : H::NSC * piece + i;
            sw[d][i] = gload(sp + g); bw[d][i] = gload(bp + g);
        }
        qb_load<H::NDW>(wp + (int64_t)piece * (8 * BITS), cw[d]);
        // (the last chunk's loads repeat past the end, unread)
        if (++lc == ln) {
            lc = 0;
            if (++lrt == RT) {
                lrt = 0;
                if (lcs + QB_SL < c1) { lcs += QB_SL; ln = min(QB_SL, c1 - lcs); }
            }
            if (RT > 1) row_ptrs(lrt);
        }
    };

    load_x(c0);
    row_ptrs(0);
#pragma unroll
    for (int d = 0; d < DEPTH; d++) load_w(d);
    convert_x(c0);
    lds_barrier();
    if (c0 + QB_SL < c1) load_x(c0 + QB_SL);   // a slice ahead

    f32x4_t tot = {0.0f, 0.0f, 0.0f, 0.0f};
    int cs = c0, n = min(QB_SL, c1 - c0), rt = 0, c = 0;
    const int units = RT * (c1 - c0);
    const uint32_t xa = lane * 16 ^ 16 * q;      // ^ 64 (step & 3), + 1024 step
    for (int u0 = 0; u0 < units; u0 += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; d++) {
            if (u0 + d < units) {
                f32x4_t acc[4];       // of a quarter's 64 codes (gs 32: of one of its two groups)
#pragma unroll
                for (int jj = 0; jj < 2; jj++) {
                    // every LDS read before the first product, every product before the first fold
                    half8_t xf[4];
#pragma unroll
                    for (int g = 0; g < 4; g++) xf[g] = *reinterpret_cast<const half8_t*>(xl + c * 8192 + (2 * g + jj) * 1024 + (xa ^ (64u * ((2 * g + jj) & 3))));
                    // this quarter's codes 16 r + 8 jj .. (gs 32: 32 jj + 8 r ..), r = 0 .. 3, to quarter r
                    gx_u4 v[4];
#pragma unroll
                    for (int r = 0; r < 4; r++) v[r] = __builtin_bit_cast(gx_u4, qb_codes<BITS, H::NDW>(cw[d], GS == 32 ? 4 * jj + r : 2 * r + jj));
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        uint32_t m[4] = {v[0][k], v[1][k], v[2][k], v[3][k]};
                        qb_transpose(m);
                        v[0][k] = m[0]; v[1][k] = m[1]; v[2][k] = m[2]; v[3][k] = m[3];
                    }
#pragma unroll
                    for (int g = 0; g < 4; g++) {
                        const bool first = GS == 32 || (jj == 0 && (GS == 64 || g % 2 == 0));
                        const int o = GS == 128 ? g & 2 : g;     // gs 128: two quarters' codes are one group
                        acc[o] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[g], __builtin_bit_cast(half8_t, v[g]), first ? f32x4_t{0.0f, 0.0f, 0.0f, 0.0f} : acc[o], 0, 0, 0);
                    }
                    if (GS != 32 && jj == 0) continue;
                    uint32_t sb[4];
                    {
                        const int i = GS == 32 ? jj : 0;
                        const uint32_t w = (uint32_t)sw[d][i] | (uint32_t)bw[d][i] << 16;
                        sb[0] = sb[1] = sb[2] = sb[3] = w;
                        qb_transpose(sb);
                    }
#pragma unroll
                    for (int g = 0; g < 4; g += GS == 128 ? 2 : 1) {
                        const int gi = GS == 32 ? 2 * g + jj : GS == 64 ? g : g / 2;
                        const uint32_t w = (cs + c) * H::GC + gi < G ? sb[g] : 0u;
                        const float sv = ST == 0 ? __uint_as_float(w << 16) : f16_to_f32((uint16_t)w);
                        const float bv = ST == 0 ? __uint_as_float(w & 0xFFFF0000u) : f16_to_f32((uint16_t)(w >> 16));
                        const f32x4_t gx = *reinterpret_cast<const f32x4_t*>(&gsum[c * H::GC + gi][4 * q]);
#pragma unroll
                        for (int k = 0; k < 4; k++) tot[k] = fmaf(sv, acc[g][k], fmaf(bv, gx[k], tot[k]));
                    }
                }
                if (++c == n) {      // the tile's part of this slice is done
                    c = 0;
                    const f32x4_t iv = *reinterpret_cast<const f32x4_t*>(&inv[4 * q]);
                    f32x4_t v = {tot[0] * iv[0], tot[1] * iv[1], tot[2] * iv[2], tot[3] * iv[3]};
                    if (cs > c0) v += qb_tot[rt * 256 + tid];
                    qb_tot[rt * 256 + tid] = v;
                    tot = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
                    if (++rt == RT) {
                        rt = 0;
                        if (cs + QB_SL < c1) {
                            cs += QB_SL;
                            n = min(QB_SL, c1 - cs);
                            lds_barrier();
                            convert_x(cs);
                            lds_barrier();
                            if (cs + QB_SL < c1) load_x(cs + QB_SL);
                        }
                    }
                }
            }
            load_w(d);
        }
    }

    auto finish = [&](int t, int n, float v) {
        int row = n, part = 0;
        if (row >= a.o1) {
            if (row < a.o1 + a.o2) { part = 1; row -= a.o1; }
            else { part = 2; row -= a.o1 + a.o2; }
        }
        a.y[(int64_t)t * a.ys + n] = v + (a.bias[part] ? ld_scale<ST>(a.bias[part] + row) : 0.0f);
    };
    for (int r = 0; r < RT; r++) {
        const f32x4_t v = qb_tot[r * 256 + tid];
        const int n = row0 + 64 * r;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float sum = xor32_sum(v[i]);            // hi and lo parts
            const int t = 4 * q + i;
            if (q >= 2 || t >= T || n >= a.O) continue;
            if (a.S == 1) finish(t, n, sum);
            else part_store(a.part + ((int64_t)z * T + t) * a.O + n, sum);
        }
    }
    if (a.S == 1) return;
    parts_stored();
    __shared__ int last;
    if (tid == 0) last = part_last(a.cnt + blk, a.S);
    __syncthreads();
    if (!last) return;
    if (tid == 0) part_rearm(a.cnt + blk);
    for (int i = tid; i < 64 * RT * T; i += 256) {
        const int n = blk * 64 * RT + i % (64 * RT), t = i / (64 * RT);
        if (n >= a.O) continue;
        float sum = 0.0f;
        for (int y = 0; y < a.S; y += 8) {   // in order, eight loads together
            float v[8];
#pragma unroll
            for (int k = 0; k < 8; k++)
                v[k] = part_load(a.part + ((int64_t)min(y + k, a.S - 1) * T + t) * a.O + n);
#pragma unroll
            for (int k = 0; k < 8; k++)
                if (y + k < a.S) sum += v[k];
        }
        finish(t, n, sum);
    }
}

// The shapes whose x goes to the matrix cores as f16 hi + lo: a value keeps 22 bits beside the largest of its
// 1024 inputs, fewer the smaller it is beside that, and an infinity comes out as NaN. 5-bit codes, and 2, 3 and
// 6 bits where K is no whole number of eight groups (four of 128 codes), hold x in fp32 and stay on the vector
// path (4096 -> 14336 at 5 bits, T = 4: 43 us there, 23 here; 8320 -> 4096 at 3 bits: 31 and 17).
bool qmb_supported(int K, int bits, int gs) {
    if ((gs != 32 && gs != 64 && gs != 128) || K % gs) return false;
    if (bits == 4 || bits == 8) return true;
    return bits != 5 && K % ((gs == 128 ? 4 : 8) * gs) == 0 && K / gs <= 2048;
}

hipError_t launch_qmb(const QmmSmallArgs& a, hipStream_t s) {
    if (!qmb_supported(a.K, a.bits, a.gs) || a.T < 1 || a.T > 8) return hipErrorInvalidValue;
    QbDev d{};
    for (int i = 0; i < 3; i++) {
        const QMat& m = a.part[i < a.nparts ? i : a.nparts - 1];
        d.w[i] = m.w; d.s[i] = m.s; d.b[i] = m.b; d.bias[i] = m.bias;
    }
    d.o1 = a.part[0].O; d.o2 = a.nparts > 1 ? a.part[1].O : 0;
    d.K = a.K; d.O = a.O; d.T = a.T; d.xs = a.x_stride; d.ys = a.y_stride; d.x = a.x; d.y = a.y;
    const int C = (a.K + QB_CH - 1) / QB_CH, cus = device_cus();
    // Tiles per wave and K ranges by expected time: a round of a workgroup per CU takes 2 us to start, 0.3 us a
    // chunk to convert x and 0.7 us a chunk and tile (a CU holds three or four workgroups, so later rounds
    // overlap a little); ranges add the hand-over, more with more partial sums. Over 120 shapes (512 .. 151936 rows,
    // 1024 .. 28672 inputs, widths and group sizes, T = 2 .. 8) it takes 0.37 .. 1.0 of the former kernels'
    // time: 5120 -> 17000 with four tiles and seven ranges 22 us, with two tiles and one range 36.
    const bool split = a.split && a.split_floats >= QGEMM_SPLIT_FLOATS;
    int RT = 1, S = 1;
    float best = 0.0f;
    for (int rt = 1; rt <= QB_RT; rt *= 2)
        for (int sl = 1; sl <= 16 && (sl == 1 || 2 * sl <= C); sl++) {
            const int nb = (a.O + 64 * rt - 1) / (64 * rt);
            if (sl > 1 && (!split || nb > (int)QGEMM_SPLIT_TILES || (size_t)sl * a.T * a.O > QGEMM_SPLIT_PART)) break;
            const int rounds = (nb * sl + cus - 1) / cus, chunks = (C + sl - 1) / sl;
            const float us = (0.2f + 0.8f * rounds) * (2.0f + chunks * (0.3f + 0.7f * rt)) + (sl > 1 ? 1.5f + sl * (0.2f + 0.02f * a.T * rt) : 0.0f);
            if (best == 0.0f || us < best) { best = us; RT = rt; S = sl; }
        }
    d.RT = RT; d.nb = (a.O + 64 * RT - 1) / (64 * RT);
    d.S = S < C ? S : C;
    if (d.S > 1) { d.cnt = reinterpret_cast<unsigned*>(a.split); d.part = a.split + QGEMM_SPLIT_TILES; }
    const dim3 grid(d.nb * d.S);
    const size_t lds = (size_t)RT * 4096;
#define QB_GO(B, GS) if (a.bits == B && a.gs == GS) { \
        if (a.st == 0) hipLaunchKernelGGL((qmb_kernel<B, GS, 0>), grid, dim3(256), lds, s, d); \
        else hipLaunchKernelGGL((qmb_kernel<B, GS, 1>), grid, dim3(256), lds, s, d); \
        return hipGetLastError(); }
#define QB_BITS(B) QB_GO(B, 32) QB_GO(B, 64) QB_GO(B, 128)
    QB_BITS(2) QB_BITS(3) QB_BITS(4) QB_BITS(6) QB_BITS(8)
#undef QB_BITS
#undef QB_GO
    return hipErrorInvalidValue;
}

}  // namespace mlxr
