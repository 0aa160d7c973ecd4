// Prefill quantized GEMM over the MLX affine layout, every code width: Y[T][O] = X[T][K] W[O][K]^T
// (+ bias), the reference's `qgemm` tiles (Kernels.swift:785-851) with fp32-level results.
//
// Arithmetic (w = s q + b per group of gs inputs):
//   y[m][n] = sum_g ( s[n][g] * sum_{k in g} q[n][k] x[m][k]  +  b[n][g] * sum_{k in g} x[m][k] )
// - The codes enter the matrix cores exactly: code q as the f16 subnormal with bit pattern q, i.e.
//   q * 2^-24 (q < 256 for every width), so no dequantization rounds anything.
// - x: each token row is multiplied by the power of two 2^e that puts max|x| in [2^13, 2^14)
//   (exact) and split into f16 hi + lo (x 2^e = hi + lo to ~2^-22 relative). Both enter the same
//   accumulator (v_mfma_f32_32x32x16_f16). A tile whose rows all have lo == 0 (inputs that are
//   bf16 values, e.g.) skips the lo products: they would add exact zeros.
// - A quantization group's products accumulate from zero and are folded in fp32 at its end (gs 128:
//   at its middle too): tot = fma(s 2^24, acc, tot).
// - The bias terms sum_g b[n][g] xsum[m][g] (xsum: the group's sum of scaled x, from the pre-pass)
//   go through the matrix cores too, 4 groups at a time, straight into tot: xsum as three bf16
//   parts and b as one (bf16 biases) or two (f16) bf16 parts, every product exact in fp32.
// - K is summed in fixed slices (qgemm_slices: a function of K and O alone), added in order, so a token's
//   result depends neither on T nor on how the launch is cut.
// - The row is multiplied back by 2^-e at the end.
//
// Tiling: a workgroup of WM x WN waves owns 32 I WM tokens x 32 J WN rows, each wave I x J tiles of
// 32 x 32 (128 x 256 by 8 waves; 64 x 128 and 32 x 128 by 4 for launches that those leave short of
// workgroups). K advances 64 at a time through three LDS stages filled by buffer -> LDS copies two
// blocks ahead (no registers hold the prefetch): X hi and lo (16-byte chunks XOR-swizzled by row, so
// 32 lanes reading 16 bytes of consecutive rows spread over the banks) and the raw code bytes of the
// rows; the scales, biases and token group sums of 4 groups at a time into two more buffers. Tiles are
// ordered so the token tiles of one weight tile run on the same XCD (its L2).
//
// What bounds it: a 128 x 256 tile's block takes ~2 us against 0.85 us of matrix-core time (4096 -> 14336 rows,
// 512 tokens, 8 bits: 64 blocks, 145 us, 415 TFLOP/s useful, twice that on the matrix cores with both parts of
// x); the rest is the barrier between the blocks, the folds and the copies' issue (a 1 KB copy holds its
// wave ~30 cycles), with two waves per SIMD in step. Before the swizzled pieces, the wide code reads and the
// copies spread over the steps: 193 us. Few tokens: the blocks' latency, hence the smaller tiles and slices.
#pragma once
#include "qgemm.h"

namespace mlxr {

struct QGemmXDev {
    const uint8_t* w; const uint16_t* s; const uint16_t* b; const uint16_t* bias; int st;
    int direct;               // s, b: the matrix's own [O][G] (G even); 0: s = the repacked [Gp / 4][O][4] of both
    int K, O, T, ys, nT, ntiles, SF, S;   // SF fixed K slices, over S workgroups per tile
    const uint16_t* xh; const uint16_t* xl; const uint16_t* gsum; const float* inv; const int* nz;
    float* y;
    unsigned* cnt; float* part;           // S > 1: tile counters (zero between launches), the slices' partial tiles
};

// A block's 64 codes of a row lie in LDS as 16-byte pieces. Rows of 24 and 40 bytes (3 and 5 bits) are not
// whole pieces: their last one is the row's last 16 bytes again, 8 bytes past where it would follow on.
template <int BITS> constexpr int gx_lrow() { return (8 * BITS + 15) / 16 * 16; }
// Rows 64 bytes apart (8 bits) start in one of four groups of banks, 32 apart (3, 4 bits) in eight: 32
// lanes reading the same codes of 32 rows met in 8 and 4 lanes a bank (8 bits: conflicts were 73% of the
// LDS' busy cycles). Their pieces are stored XORed with this; the reads are up to 16 bytes wide.
template <int BITS>
__device__ __forceinline__ int gx_swz(int r) { return BITS == 8 ? (r >> 2) & 3 : BITS == 4 || BITS == 3 ? (r >> 3) & 1 : 0; }

// The k order inside a group is free (the same for codes and x): lane half h of an MFMA takes NC
// consecutive codes of a row's group part, 8 per k-step: codes 32 h .. of a block (gs 64, 128: NC 32), or
// 32 part + 16 h .. (gs 32: NC 16). Their raw bytes in registers: NW dwords, read at lane address `row`
// (gx_code_base).
template <int BITS, int NC> struct GxRaw { static constexpr int NW = (NC * BITS + 31) / 32; uint32_t w[NW]; };
template <int BITS, int NC>
__device__ __forceinline__ int gx_code_base(int r, int h) {
    const int row = r * gx_lrow<BITS>();
    if constexpr (BITS == 8) return row + 16 * ((NC == 32 ? 2 * h : h) ^ gx_swz<8>(r));
    if constexpr (BITS == 4) return row + (NC == 32 ? 16 * (h ^ gx_swz<4>(r)) : 16 * gx_swz<4>(r) + 8 * h);
    if constexpr (BITS == 3) return row + (NC == 32 ? 16 * (h ^ gx_swz<3>(r)) : 16 * gx_swz<3>(r)) + 4 * h;
    return row + (h * NC * BITS / 8 & ~3);   // 5 bits at 16 codes: gx_read shifts the upper half's words
}
template <int BITS, int NC>
__device__ __forceinline__ GxRaw<BITS, NC> gx_read(const uint8_t* lds, uint32_t row, int h, int part) {
    GxRaw<BITS, NC> o;
    constexpr int NW = GxRaw<BITS, NC>::NW;
    if constexpr (BITS == 8 || BITS == 4) {
        // 16-byte pieces (4 bits at 16 codes: the lane's half of one)
        const uint32_t at = row ^ (uint32_t)(16 * part * (BITS == 8 ? 2 : 1));
        if constexpr (NC * BITS < 128) {
            const uint2 v = *reinterpret_cast<const uint2*>(lds + at);
            o.w[0] = v.x; o.w[1] = v.y;
        } else {
#pragma unroll
            for (int p = 0; p < NC * BITS / 128; p++) {
                const uint4 v = *reinterpret_cast<const uint4*>(lds + (at ^ (16u * p)));
                o.w[4 * p] = v.x; o.w[4 * p + 1] = v.y; o.w[4 * p + 2] = v.z; o.w[4 * p + 3] = v.w;
            }
        }
    } else if constexpr (BITS == 3) {
        // codes 0 .. 31 (12 bytes) in the first piece, 32 .. 63 four bytes into the second
        const uint32_t* p = reinterpret_cast<const uint32_t*>(lds + (row ^ (16u * part)) + 4 * part);
#pragma unroll
        for (int i = 0; i < NW; i++) o.w[i] = p[i];
    } else if constexpr (BITS == 5) {
        // the row's bytes 32 .. 39 lie 8 further on
        const uint8_t* p = lds + row + part * 20;
        const int at = part * 20 + (NC == 32 ? 20 : 8) * h;
#pragma unroll
        for (int i = 0; i < NW; i++) o.w[i] = *reinterpret_cast<const uint32_t*>(p + 4 * i + (at + 4 * i >= 32 ? 8 : 0));
    } else if constexpr (BITS * NC % 64 == 0) {   // whole 8-byte words
        const uint2* p = reinterpret_cast<const uint2*>(lds + row + part * 4 * BITS);
#pragma unroll
        for (int i = 0; i < NW / 2; i++) {
            const uint2 v = p[i];
            o.w[2 * i] = v.x; o.w[2 * i + 1] = v.y;
        }
    } else {
        const uint32_t* p = reinterpret_cast<const uint32_t*>(lds + row) + part * BITS;
#pragma unroll
        for (int i = 0; i < NW; i++) o.w[i] = p[i];
    }
    if constexpr ((NC * BITS) % 32 != 0) {   // 16 codes of an odd width: 16 h bits into the words
#pragma unroll
        for (int i = 0; i < NW; i++) {
            const uint32_t up = i + 1 < NW ? o.w[i + 1] : 0u;
            o.w[i] = h ? (o.w[i] >> 16) | (up << 16) : o.w[i];
        }
    }
    return o;
}
// The 8 codes of k-step ks as f16 subnormals, i.e. q * 2^-24 exactly.
template <int BITS, int NC>
__device__ __forceinline__ half8_t gx_codes(const GxRaw<BITS, NC>& o, int ks) {
    if constexpr (BITS == 4) {
        // even codes' bytes and odd codes' bytes, then byte permutes into (even, odd) 16-bit pairs
        const uint32_t v = o.w[ks], ev = v & 0x0F0F0F0Fu, od = (v >> 4) & 0x0F0F0F0Fu;
        return __builtin_bit_cast(half8_t, gx_u4{__builtin_amdgcn_perm(od, ev, 0x0C040C00u), __builtin_amdgcn_perm(od, ev, 0x0C050C01u),
                                                 __builtin_amdgcn_perm(od, ev, 0x0C060C02u), __builtin_amdgcn_perm(od, ev, 0x0C070C03u)});
    } else if constexpr (BITS == 8) {
        const uint32_t v = o.w[2 * ks], u = o.w[2 * ks + 1];
        return __builtin_bit_cast(half8_t, gx_u4{__builtin_amdgcn_perm(0u, v, 0x0C010C00u), __builtin_amdgcn_perm(0u, v, 0x0C030C02u),
                                                 __builtin_amdgcn_perm(0u, u, 0x0C010C00u), __builtin_amdgcn_perm(0u, u, 0x0C030C02u)});
    } else {
        constexpr uint32_t M = (1u << BITS) - 1u;
        auto code = [&](int c) {   // c is a constant: a bit field of one dword, or of two joined
            const int bit = c * BITS, wi = bit >> 5, off = bit & 31;
            if (off + BITS <= 32) return (o.w[wi] >> off) & M;
            return __builtin_amdgcn_alignbit(o.w[wi + 1], o.w[wi], (uint32_t)off) & M;
        };
        uint32_t q[4];
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] = code(8 * ks + 2 * i) | (code(8 * ks + 2 * i + 1) << 16);
        return __builtin_bit_cast(half8_t, gx_u4{q[0], q[1], q[2], q[3]});
    }
}

// A launch's tile shape.
template <int WM_, int WN_, int I_, int J_> struct GxCfg {
    static constexpr int WM = WM_, WN = WN_, I = I_, J = J_, NW = WM * WN, TOK = 32 * I * WM, NR = 32 * J * WN;
};
using GxBig = GxCfg<2, 4, 2, 2>;     // 128 tokens x 256 rows
using GxMid = GxCfg<1, 4, 2, 1>;     // 64 x 128
using GxSmall = GxCfg<1, 4, 1, 1>;   // 32 x 128
// bytes of a stage (X hi, X lo, codes), of a chunk buffer (scales [rows][4], biases [rows][4], the tokens'
// group sums as bf16 parts [tokens][hi, mid, lo][4]), of the workgroup's LDS
template <int BITS, class C> constexpr int gx_stage() { return 2 * C::TOK * GX_K * 2 + C::NR * gx_lrow<BITS>(); }
template <class C> constexpr int gx_chunk() { return C::NR * 16 + C::TOK * GX_GSUM; }
template <int BITS, class C> constexpr int gx_lds() { return GX_NST * gx_stage<BITS, C>() + 2 * gx_chunk<C>(); }

template <int BITS, int GS, class C, bool LO>
__device__ __forceinline__ void qgemmx_body(const QGemmXDev& a, uint8_t* lds, int tile, int z) {
    constexpr int I = C::I, J = C::J, NW = C::NW, TOK = C::TOK, NR = C::NR;
    constexpr int XB = TOK * GX_K * 2, STG = gx_stage<BITS, C>(), CB = gx_chunk<C>();
    constexpr int XCP = TOK / (8 * NW);                          // X copies per wave, part and block (1 KB = 8 rows)
    constexpr int PPR = gx_lrow<BITS>() / 16;                    // 16-byte pieces per row of codes
    constexpr int WCT = NR * PPR / 64;                           // code copies per block (1 KB),
    constexpr int WCP = (WCT + NW - 1) / NW;                     // per wave and block (some waves repeat another's)
    static_assert(XCP >= 1 && TOK % (8 * NW) == 0, "copies");
    constexpr int NCP = (LO ? 2 : 1) * XCP + WCP;                // copies a wave issues per block (a chunk adds some)
    constexpr int BPC = 4 * GS / GX_K;                           // blocks per chunk of 4 groups (2, 4 or 8)
    static_assert(NCP < 64 && BPC >= 2, "pipeline");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % C::WM, wn = wave / C::WM;
    const int ot = tile / a.nT, tt = tile - ot * a.nT;
    const int n0 = ot * NR, m0 = tt * TOK;
    const int K = a.K, G = K / GS, Gp = gx_gpad(G);
    const uint32_t rowb = (uint32_t)(K / 8 * BITS);     // code bytes per row
    const __amdgpu_buffer_rsrc_t xhr = __builtin_amdgcn_make_buffer_rsrc((void*)a.xh, 0, a.T * K * 2, GX_RSRC_W3);
    const __amdgpu_buffer_rsrc_t xlr = __builtin_amdgcn_make_buffer_rsrc((void*)a.xl, 0, a.T * K * 2, GX_RSRC_W3);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void*)a.w, 0, (int)((uint32_t)a.O * rowb), GX_RSRC_W3);
    const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc((void*)a.s, 0, a.direct ? a.O * G * 2 : Gp * a.O * 4, GX_RSRC_W3);
    const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc((void*)a.b, 0, a.direct ? a.O * G * 2 : 0, GX_RSRC_W3);
    const __amdgpu_buffer_rsrc_t gr = __builtin_amdgcn_make_buffer_rsrc((void*)a.gsum, 0, Gp / 4 * a.T * GX_GSUM, GX_RSRC_W3);
    uint8_t* cbuf = lds + GX_NST * STG;

    // Per-lane parts of the copies' offsets (the rest is uniform): X row lane / 8 of a copy's 8 and its
    // 16-byte chunk, XORed with (row / 2) % 8 (16 rows read together fill the banks); codes (copies of whole
    // rows): row lane / PPR and the piece that lies at the lane's place. Rows past T or O read past the
    // buffer's end: zeros.
    const uint32_t xl_off = (uint32_t)(lane >> 3) * (uint32_t)K * 2u + 16u * (uint32_t)((lane & 7) ^ (lane >> 4));
    constexpr bool WROWS = 64 % PPR == 0;
    auto piece = [](int c) { return BITS % 2 && c == PPR - 1 ? (uint32_t)(8 * BITS - 16) : 16u * c; };   // its bytes in the row's
    const uint32_t wl_off = WROWS ? (uint32_t)(lane / PPR) * rowb + piece((lane % PPR) ^ gx_swz<BITS>(lane / PPR)) : 0u;
    // copy p (< NCP) of this wave's copies of block blk into its stage: X hi, X lo, codes
    auto issue1 = [&](int blk, int p) {
        uint8_t* st = lds + (blk % GX_NST) * STG;
        // opaque copies: each offset is one add per copy here, not a register kept across the loop
        uint32_t xo = xl_off, wo = wl_off;
        int ln = lane;
        asm volatile("" : "+v"(xo), "+v"(wo), "+v"(ln));
        constexpr int NX = (LO ? 2 : 1) * XCP;
        if (p < NX) {
            const int h = p / XCP, q = XCP * wave + p % XCP;
            const uint32_t off = (xo ^ (64u * (q & 1))) + (((uint32_t)(m0 + 8 * q) * (uint32_t)K + (uint32_t)blk * GX_K) * 2u);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(h ? xlr : xhr, (gx_lptr)(st + h * XB + q * 1024), 16, off, 0, 0, 0);
            return;
        }
        const int c = p - NX, q = WCT % NW == 0 ? wave * WCP + c : (wave * WCP + c) % WCT;
        uint32_t off;
        if constexpr (WROWS) off = wo + (uint32_t)(n0 + q * (64 / PPR)) * rowb;   // a multiple of the swizzle's period
        else off = (uint32_t)(n0 + (q * 64 + ln) / PPR) * rowb + piece((q * 64 + ln) % PPR);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (gx_lptr)(st + 2 * XB + q * 1024), 16, off + (uint32_t)blk * (8u * BITS), 0, 0, 0);
    };
    auto issue = [&](int blk) {
#pragma unroll
        for (int p = 0; p < NCP; p++) issue1(blk, p);
    };
    // chunk ch (groups 4 ch .. 4 ch + 3) into buffer ch & 1: the rows' scales and biases (from the matrix:
    // 4-byte pieces, one copy of each per wave; words past a row's last group belong to the next row and
    // are not used; or repacked: 1 KB copies) and the token group sums
    auto issue_chunk = [&](int ch) {
        uint8_t* cb = cbuf + (ch & 1) * CB;
        constexpr int PD = NR / 32, PA = NR / 128, NG = (TOK * GX_GSUM + 1023) / 1024;
        // pieces: scales, biases, group sums; waves take them in turn
        const int np = a.direct ? PD : PA;
        for (int p = wave; p < 2 * np + NG; p += NW) {
            if (p < 2 * np) {
                const int part = p >= np, q = p - part * np;
                if (a.direct) {
                    const uint32_t off = ((uint32_t)(n0 + 32 * q + (lane >> 1)) * (uint32_t)G + 4u * (uint32_t)ch + 2u * (lane & 1)) * 2u;
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(part ? br : sr, (gx_lptr)(cb + part * NR * 8 + q * 256), 4, off, 0, 0, 0);
                } else {
                    const uint32_t off = (uint32_t)part * (uint32_t)Gp * (uint32_t)a.O * 2u + ((uint32_t)ch * (uint32_t)a.O + (uint32_t)n0 + 128u * q) * 8u + 16u * lane;
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(sr, (gx_lptr)(cb + part * NR * 8 + q * 1024), 16, off, 0, 0, 0);
                }
            } else {
                // the tokens' group sums are consecutive bytes (tokens past T: out of range or the next
                // chunk's, never used)
                const int o = (p - 2 * np) * 1024 + 16 * lane;
                if (o < TOK * GX_GSUM)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(gr, (gx_lptr)(cb + NR * 16 + (p - 2 * np) * 1024), 16,
                                                             ((uint32_t)ch * (uint32_t)a.T + (uint32_t)m0) * (uint32_t)GX_GSUM + (uint32_t)o, 0, 0, 0);
            }
        }
    };

    f32x16_t acc[J], tot[I][J];
#pragma unroll
    for (int i = 0; i < I; i++)
#pragma unroll
        for (int j = 0; j < J; j++) tot[i][j] = (f32x16_t)0.0f;

    // the bias terms of chunk ch's groups in [g0, g1) on the matrix cores: sum_g b[n][g] xsum[m][g]
    // with xsum as bf16 hi + mid + lo (truncations; exact) and b as bf16 bhi + blo (blo = 0 for bf16
    // biases; 3 bits for f16 ones), every product exact and summed in fp32.
    // 32x32x16 bf16: k 0-3 hi * bhi, 4-7 mid * bhi, 8-11 lo * bhi, 12-15 hi * blo (4 groups each);
    // f16 biases add mid * blo and lo * blo in a second product.
    auto bias_terms = [&](int ch, int g0, int g1) {
        const uint8_t* cb = cbuf + (ch & 1) * CB;
        const int h = lane >> 5, l31 = lane & 31;
        auto bw = [](float v) { return (uint32_t)(__float_as_uint(v) >> 16); };
        // groups outside the slice (or past the row: another row's words) count as zero
        uint32_t m0_ = 0, m1_ = 0;
        if (4 * ch >= g0 && 4 * ch < g1) m0_ |= 0xFFFFu;
        if (4 * ch + 1 >= g0 && 4 * ch + 1 < g1) m0_ |= 0xFFFF0000u;
        if (4 * ch + 2 >= g0 && 4 * ch + 2 < g1) m1_ |= 0xFFFFu;
        if (4 * ch + 3 >= g0 && 4 * ch + 3 < g1) m1_ |= 0xFFFF0000u;
        const bool f16b = a.st != 0;
        gx_u4 A1[I], A2[I];
#pragma unroll
        for (int i = 0; i < I; i++) {
            const uint8_t* xs = cb + NR * 16 + (wm * 32 * I + i * 32 + l31) * GX_GSUM;
            const uint2 lo16 = *reinterpret_cast<const uint2*>(xs + 16 * h), hi16 = *reinterpret_cast<const uint2*>(xs + 8 - 8 * h);
            A1[i] = gx_u4{lo16.x, lo16.y, hi16.x, hi16.y};              // h 0: hi, mid; h 1: lo, hi
            if (f16b) {
                const uint2 md = *reinterpret_cast<const uint2*>(xs + 8), lo = *reinterpret_cast<const uint2*>(xs + 16);
                A2[i] = h == 0 ? gx_u4{md.x, md.y, lo.x, lo.y} : gx_u4{0u, 0u, 0u, 0u};
            }
        }
#pragma unroll
        for (int j = 0; j < J; j++) {
            const int rr = wn * 32 * J + j * 32 + l31;
            uint2 b4 = *reinterpret_cast<const uint2*>(cb + NR * 8 + rr * 8);
            b4.x &= m0_; b4.y &= m1_;
            uint32_t ph0 = b4.x, ph1 = b4.y, pl0 = 0, pl1 = 0;
            if (f16b) {
                const uint16_t bb[4] = {(uint16_t)b4.x, (uint16_t)(b4.x >> 16), (uint16_t)b4.y, (uint16_t)(b4.y >> 16)};
                uint32_t bh[4], bl[4];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float f = f16_to_f32(bb[q]), fh = __uint_as_float(__float_as_uint(f) & 0xFFFF0000u);
                    bh[q] = bw(fh); bl[q] = bw(f - fh);
                }
                ph0 = bh[0] | (bh[1] << 16); ph1 = bh[2] | (bh[3] << 16);
                pl0 = bl[0] | (bl[1] << 16); pl1 = bl[2] | (bl[3] << 16);
            }
            const gx_u4 B1 = h == 0 ? gx_u4{ph0, ph1, ph0, ph1} : gx_u4{ph0, ph1, pl0, pl1};
#pragma unroll
            for (int i = 0; i < I; i++)
                tot[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(gx_bf8, A1[i]), __builtin_bit_cast(gx_bf8, B1), tot[i][j], 0, 0, 0);
            if (f16b) {
                const gx_u4 B2 = h == 0 ? gx_u4{pl0, pl1, pl0, pl1} : gx_u4{0u, 0u, 0u, 0u};
#pragma unroll
                for (int i = 0; i < I; i++)
                    tot[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(gx_bf8, A2[i]), __builtin_bit_cast(gx_bf8, B2), tot[i][j], 0, 0, 0);
            }
        }
    };

    const int nblk = K / GX_K;
    constexpr int unit = GS > GX_K ? GS / GX_K : 1;      // slice boundaries fall on group boundaries
    const int nunits = nblk / unit, SF = a.SF;
    auto bound = [&](int sl) { return nunits * sl / SF * unit; };
    const int sl0 = z * SF / a.S, sl1 = (z + 1) * SF / a.S, kbe = bound(sl1);
    int kb = bound(sl0), g0 = 0, g1 = 0, kbs = 0;

    // A block is NT steps of one 16-k step of one of the wave's I token tiles (gs 32: two groups, one after
    // the other). The token tiles take a group's codes in turn through one set of accumulators (32 J rows x
    // 32 tokens), each folded at its end, tot = fma(s 2^24, acc, tot), which leaves registers for the fragments. While a step's products issue, the next one's X
    // fragments are read, its codes unpacked (in the first tile's pass) and a few of the copies of the
    // block two ahead issued (all at once at the block's start they held the waves up for ~1400 of its 5600
    // cycles); the last step does the same for the next block, behind the barrier that its copies need.
    constexpr int NKS = GS == 32 ? 2 : 4, NC = 8 * NKS, NPART = 4 / NKS, NT = 4 * I;
    constexpr int PPS = (NCP + NT - 2) / (NT - 1);       // copies per step
    half8_t x[2][LO ? 2 : 1];
    GxRaw<BITS, NC> raw[NPART][J];
    uint16_t s16[NPART][J];
    // step s's X fragments (into set s & 1), the codes and scales of a block
    auto lane_now = [&] { int l = threadIdx.x & 63; asm volatile("" : "+v"(l)); return l; };
    auto xread = [&](int blk, int s) {
        const int ln = lane_now(), h = ln >> 5, l31 = ln & 31;
        const int part = s / (NKS * I), i = s / NKS % I, ks = 2 * NKS * part + s % NKS;   // X chunk NKS (2 part + h) + k
        const uint32_t xb = (uint32_t)(blk % GX_NST) * STG + (uint32_t)(wm * 32 * I + l31) * 128u + 16u * (uint32_t)((NKS * h) ^ ((l31 >> 1) & 7));
#pragma unroll
        for (int p = 0; p < (LO ? 2 : 1); p++)
            x[s & 1][p] = *reinterpret_cast<const half8_t*>(lds + (xb ^ (16u * ks)) + p * XB + i * 4096);
    };
    auto wread = [&](int blk) {
        const int ln = lane_now(), h = ln >> 5, l31 = ln & 31;
#pragma unroll
        for (int j = 0; j < J; j++) {
            const int r = wn * 32 * J + j * 32 + l31;
            const uint32_t wb = (uint32_t)(blk % GX_NST) * STG + 2 * XB + (uint32_t)gx_code_base<BITS, NC>(r, h);
#pragma unroll
            for (int part = 0; part < NPART; part++) {
                raw[part][j] = gx_read<BITS, NC>(lds, wb, h, part);
                const int g = (blk * GX_K + 16 * NKS * part) / GS;
                s16[part][j] = *reinterpret_cast<const uint16_t*>(cbuf + ((g >> 2) & 1) * CB + r * 8 + (g & 3) * 2);
            }
        }
    };
    // before block blk: this wave's copies of it have landed (those of the block after it, `more`, may still
    // be in flight), its LDS reads of the block before are done, and so are every wave's: that block's stage
    // may be overwritten, and so may the chunk buffer of the chunk before last.
    auto ready = [&](bool more) {
        if (more) __builtin_amdgcn_s_waitcnt(gx_wait_vm(NCP) & ~0x0F00);
        else __builtin_amdgcn_s_waitcnt(gx_wait_vm(0) & ~0x0F00);
        __builtin_amdgcn_s_barrier();
    };
    issue_chunk(kb / BPC);
    issue(kb);
    if (kb + 1 < kbe) issue(kb + 1);
    ready(kb + 1 < kbe);
    wread(kb);
    xread(kb, 0);
    auto step = [&] {
        if (kb + 1 < kbe && (kb + 1) % BPC == 0) issue_chunk((kb + 1) / BPC);
        half8_t bw[NKS][J];
#pragma unroll
        for (int j = 0; j < J; j++) bw[0][j] = gx_codes(raw[0][j], 0);
#pragma unroll
        for (int s = 0; s < NT; s++) {
            const int part = s / (NKS * I), i = s / NKS % I, k = s % NKS;
            float sv[J];
            __builtin_amdgcn_sched_barrier(0);
            if (s + 1 < NT) {
                xread(kb, s + 1);
                if (kb + 2 < kbe) {
#pragma unroll
                    for (int p = PPS * s; p < PPS * (s + 1) && p < NCP; p++) issue1(kb + 2, p);
                }
            } else {
                // the block's scales are needed once more, by this step's fold
#pragma unroll
                for (int j = 0; j < J; j++) sv[j] = (a.st == 0 ? bf16_to_f32(s16[part][j]) : f16_to_f32(s16[part][j])) * 16777216.0f;
                if (kb + 1 < kbe) {
                    ready(kb + 2 < kbe);
                    wread(kb + 1);
                    xread(kb + 1, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int p = 0; p < (LO ? 2 : 1); p++)
#pragma unroll
                for (int j = 0; j < J; j++)
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[s & 1][p], bw[k][j], k == 0 && p == 0 ? (f32x16_t)0.0f : acc[j], 0, 0, 0);
            const int s1 = s + 1, part1 = s1 / (NKS * I), k1 = s1 % NKS;
            if (s1 < NT && s1 / NKS % I == 0) {
#pragma unroll
                for (int j = 0; j < J; j++) bw[k1][j] = gx_codes(raw[part1][j], k1);
#pragma unroll
                for (int q = 0; q < (LO ? 2 : 1) * J; q++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
                }
            }
            if (k == NKS - 1) {
#pragma unroll
                for (int j = 0; j < J; j++) {
                    if (s + 1 < NT) sv[j] = (a.st == 0 ? bf16_to_f32(s16[part][j]) : f16_to_f32(s16[part][j])) * 16777216.0f;
#pragma unroll
                    for (int r = 0; r < 16; r++) tot[i][j][r] = fmaf(sv[j], acc[j][r], tot[i][j][r]);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (kb == kbs || kb % BPC == 0) bias_terms(kb / BPC, g0, g1);
        kb++;
    };
    auto pidx = [&](int sl, int i, int j, int r) {   // [slice][tile][values][thread]: a wave's accesses are contiguous
        return (((size_t)sl * a.ntiles + tile) * (I * J * 16) + (i * J + j) * 16 + r) * (64 * NW) + 64 * wave + lane_now();
    };
    for (int sl = sl0; sl < sl1; sl++) {
        const int kb1 = bound(sl + 1);
        kbs = kb; g0 = kb * GX_K / GS; g1 = kb1 * GX_K / GS;
        while (kb < kb1) step();
        if (a.S > 1) {
            // the slice's partial tile, added by the tile's last workgroup to finish
#pragma unroll
            for (int i = 0; i < I; i++)
#pragma unroll
                for (int j = 0; j < J; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) part_store(a.part + pidx(sl, i, j, r), tot[i][j][r]);
        } else if (SF > 1) {
            // slices added in order, each from zero; their running sum waits in the thread's own outputs
            // (opaque indexes: addresses kept across the block loop would cost it its registers)
            int ln = lane_now(), ys = a.ys;
            asm volatile("" : "+s"(ys));
            const int n1 = n0 + wn * 32 * J + (ln & 31), m1 = m0 + wm * 32 * I + 4 * (ln >> 5);
            float* yb = a.y + (int64_t)m1 * ys + n1;
            if (sl > sl0) {
#pragma unroll
                for (int i = 0; i < I; i++) {
                    f32x16_t v[J];   // 16 J loads in flight (rows past T and O: the last row's, not kept)
#pragma unroll
                    for (int j = 0; j < J; j++)
#pragma unroll
                        for (int r = 0; r < 16; r++) {
                            const int m = i * 32 + 8 * (r >> 2) + (r & 3);
                            v[j][r] = gload(a.y + (int64_t)min(m1 + m, a.T - 1) * ys + min(n1 + j * 32, a.O - 1));
                        }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int j = 0; j < J; j++) tot[i][j] += v[j];
                }
            }
            if (sl + 1 < sl1) {
#pragma unroll
                for (int j = 0; j < J; j++)
#pragma unroll
                    for (int i = 0; i < I; i++)
#pragma unroll
                        for (int r = 0; r < 16; r++) {
                            const int m = i * 32 + 8 * (r >> 2) + (r & 3);
                            if (m1 + m < a.T && n1 + j * 32 < a.O) gstore(yb + (int64_t)m * ys + j * 32, tot[i][j][r]);
                        }
            }
        }
        if (sl + 1 < sl1) {
#pragma unroll
            for (int i = 0; i < I; i++)
#pragma unroll
                for (int j = 0; j < J; j++) tot[i][j] = (f32x16_t)0.0f;
        }
    }
    if (a.S > 1) {
        parts_stored();
        __shared__ int last;
        if (tid == 0) last = part_last(a.cnt + tile, a.S);
        __syncthreads();
        if (!last) return;
        if (tid == 0) part_rearm(a.cnt + tile);
        for (int sl = 0; sl < SF; sl++) {   // in order
#pragma unroll
            for (int i = 0; i < I; i++)
#pragma unroll
                for (int j = 0; j < J; j++) {
                    f32x16_t v;
#pragma unroll
                    for (int r = 0; r < 16; r++) v[r] = part_load(a.part + pidx(sl, i, j, r));
                    tot[i][j] = sl == 0 ? v : tot[i][j] + v;
                }
        }
    }
    const int ln = lane_now(), n1 = n0 + wn * 32 * J + (ln & 31), m1 = m0 + wm * 32 * I + 4 * (ln >> 5);
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int n = n1 + j * 32;
        if (n >= a.O) continue;
        const float bias = a.bias ? (a.st == 0 ? ld_scale<0>(a.bias + n) : ld_scale<1>(a.bias + n)) : 0.0f;
#pragma unroll
        for (int i = 0; i < I; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = m1 + i * 32 + 8 * (r >> 2) + (r & 3);
                if (m < a.T) a.y[(int64_t)m * a.ys + n] = tot[i][j][r] * a.inv[m] + bias;
            }
    }
}

template <int BITS, int GS, class C>
__global__ __launch_bounds__(64 * C::NW, 2) void qgemmx_kernel(QGemmXDev a) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t gx_lds_base[];
    __shared__ int lo_any;
    const int tid = threadIdx.x;
    // XCD x runs workgroups x, x + 8, ...: give it a contiguous run of tiles, token tiles fastest, K
    // slices slowest
    const int total = a.ntiles * a.S, g = blockIdx.x, xcd = g & 7, per = total >> 3, rem = total & 7;
    const int item = xcd * per + min(xcd, rem) + (g >> 3), z = item / a.ntiles, tile = item - z * a.ntiles;
    const int m0 = (tile % a.nT) * C::TOK;
    if (tid == 0) lo_any = 0;
    __syncthreads();
    if (tid < C::TOK && m0 + tid < a.T && a.nz[m0 + tid]) lo_any = 1;
    __syncthreads();
    if (lo_any) qgemmx_body<BITS, GS, C, true>(a, gx_lds_base, tile, z);
    else qgemmx_body<BITS, GS, C, false>(a, gx_lds_base, tile, z);
}

template <int BITS, int GS, class C>
static hipError_t qgemmx_go(QGemmXDev d, hipStream_t s) {
    constexpr int lds = gx_lds<BITS, C>();
    static bool attr = false;
    if (!attr) {
        if (hipError_t e = hipFuncSetAttribute((const void*)qgemmx_kernel<BITS, GS, C>, hipFuncAttributeMaxDynamicSharedMemorySize, lds)) return e;
        attr = true;
    }
    d.nT = (d.T + C::TOK - 1) / C::TOK;
    d.ntiles = d.nT * ((d.O + C::NR - 1) / C::NR);
    hipLaunchKernelGGL((qgemmx_kernel<BITS, GS, C>), dim3(d.ntiles * d.S), dim3(64 * C::NW), lds, s, d);
    return hipGetLastError();
}
// cut 0: GxBig, 1: GxMid, 2: GxSmall. One instantiation per code width (qgemm<width>.hip).
template <int BITS>
static hipError_t qgemmx_width(const QGemmXDev& d, int gs, int cut, hipStream_t s) {
#define GX_GO(GS) return cut == 0 ? qgemmx_go<BITS, GS, GxBig>(d, s) : cut == 1 ? qgemmx_go<BITS, GS, GxMid>(d, s) : qgemmx_go<BITS, GS, GxSmall>(d, s)
    switch (gs) {
        case 32: GX_GO(32);
        case 64: GX_GO(64);
        case 128: GX_GO(128);
    }
#undef GX_GO
    return hipErrorInvalidValue;
}

}  // namespace mlxr
