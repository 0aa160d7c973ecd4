// Causal prefill attention on the matrix cores (flash attention over the bf16 paged KV cache).
//
// Semantics: the reference's flash_prefill (Kernels.swift:1839-2000): query t of the chunk sits at
// position pos0 + t and attends keys 0..pos0+t; scores s = (q * scale) . k, an online softmax over
// key tiles, out = sum p v / sum p, all in fp32 arithmetic. Here q and p enter the bf16 MFMA as a
// hi + lo pair of bf16 values (x = hi + lo exactly to ~2^-16), K and V are the bf16 cache itself,
// and every product accumulates in fp32, so the result matches fp32 arithmetic to ~1e-5 relative.
//
#include "kernels.h"
#include <type_traits>

namespace mlxr {

typedef __bf16 fbf16x8_t __attribute__((ext_vector_type(8)));
typedef float ff32x4_t __attribute__((ext_vector_type(4)));

// MI355X layout: an item is one query head's block of 32 queries; a 256-thread workgroup (a wave per SIMD,
// two workgroups per CU, so that one's softmax runs beside the other's products) takes four items of one
// KV head, heads fastest. All four items read the same K / V tiles, copied from the paged cache straight
// into LDS (buffer -> LDS, [key][128] bf16 with 16-byte chunks XOR-swizzled by (key & 15), two stages).
// A query walks every key tile from position 0 in order, whatever the chunk or its place in it (tiles past
// its last key change nothing), so its output has the same bits however a prompt is cut into chunks. Key
// ranges on workgroups of their own, as many as leave no CU idle, did not keep that (16 tokens after 7000, 40
// heads, took 41 us with them and take 242).
//   S^T = K Q^T   A = K rows (16-byte LDS reads), B = q * scale * log2(e) as bf16 hi + lo (registers)
//   softmax in base 2 (exp2), per query column (lane exchanges for the tile's max and sum; the outputs are
//                 rescaled only where a max grew)
//   O^T += V^T P^T  B = P^T from the S^T accumulators (hi + lo bf16: hardware conversions);
//                 A = V^T read with the LDS transpose read: lane j of a 16-lane group reads key
//                 base + (j >> 2), dims 4 (j & 3) .. + 3, and lane i receives dim i of the four
//                 keys base .. base + 3, so V needs no transposed copy.
// What bounds it: 128 MFMAs (the hi + lo pairs double them) and the softmax's vector work a tile and wave, the
// two overlapped by the CU's other workgroup only in part: 3.45 us a tile for a pair, of which the MFMAs are
// 1.7. The page number and the position go through readfirstlane, or each copy becomes a loop over lanes whose
// buffer descriptors might differ (2048 tokens after 28000: 2990 us so, 2310 now), and whole tiles have a loop
// of their own, without masks and without a branch around each V fragment (130 -> 126 us at 2048 after 0).
// 1000 tokens after 7001, 40 / 8 heads: 475 us with eight items of two query blocks per workgroup (one
// workgroup per CU), 379 in this cut.
typedef short fp_v4s __attribute__((ext_vector_type(4)));
typedef __bf16 fp_bf2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void* fp_lptr;
typedef __attribute__((address_space(3))) fp_v4s* fp_lv4;
constexpr int F2_TILE = 64 * 256;                 // one K (or V) tile: 64 keys x 128 bf16

// (x0, x1) -> packed bf16 hi pair and lo pair, hi + lo = x to ~2^-16 relative
__device__ __forceinline__ void split2(float x0, float x1, uint32_t& hi, uint32_t& lo) {
    const fp_bf2 h = {(__bf16)x0, (__bf16)x1};
    hi = __builtin_bit_cast(uint32_t, h);
    const float r0 = x0 - __uint_as_float(hi << 16), r1 = x1 - __uint_as_float(hi & 0xffff0000u);
    const fp_bf2 l = {(__bf16)r0, (__bf16)r1};
    lo = __builtin_bit_cast(uint32_t, l);
}

struct FlashDev {
    FlashArgs a;
    int nb, nwg, first;   // query blocks, workgroups per KV head, ranks dealt heaviest first
};

__global__ __launch_bounds__(256, 2) void flash_kernel(FlashDev f) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t f2_lds[];   // [2 stages][K tile, V tile]
    const FlashArgs& a = f.a;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G = a.nH / a.nKV;
    // KV heads fastest (with eight of them an XCD keeps to one), then item ranks: heaviest first, the ones
    // past `first` lightest first (they share a CU with the heaviest)
    const int g = (int)blockIdx.x, rank = g / a.nKV, kvh = g % a.nKV;
    const int w = rank < f.first ? f.nwg - 1 - rank : rank - f.first;
    const int items = G * f.nb, item = 4 * w + wave, last = min(4 * w + 3, items - 1);
    const bool active = item < items;
    const int blk = min(item, items - 1) / G, h = kvh * G + min(item, items - 1) % G;
    const int pos0 = __builtin_amdgcn_readfirstlane(*a.dpos);
    const int q0 = blk * 32, nq = min(32, a.T - q0);
    const int kend = pos0 + q0 + nq;                                      // this wave's keys [0, kend)
    const int all = (pos0 + min(last / G * 32 + 32, a.T) + 63) / 64;      // the last item's tiles
    const int ntiles = active ? (kend + 63) / 64 : 0;
    const int r16 = lane & 15, kq = lane >> 4;
    const float qscale = a.scale * 1.4426950408889634f;   // scores in base-2 units

    // copies of tile t: wave w takes 1-KB pieces 8w .. 8w + 7 of the 32 (K: 0-15, V: 16-31)
    auto issue = [&](int t) {
        const int page = __builtin_amdgcn_readfirstlane(a.pt[t]);
        uint8_t* st = f2_lds + (t & 1) * 2 * F2_TILE;
        const size_t off = ((size_t)page * a.nKV + kvh) * (size_t)F2_TILE;
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)((const uint8_t*)(wave < 2 ? a.kc : a.vc) + off), 0, F2_TILE, 0x00020000);
        st += wave < 2 ? 0 : F2_TILE;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int q = 8 * (wave & 1) + i, key = 4 * q + kq;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (fp_lptr)(st + q * 1024), 16, key * 256 + 16 * (r16 ^ (key & 15)), 0, 0, 0);
        }
    };

    // q of this wave's head as B fragments [db][qb] x (hi, lo): dims 32 db + 8 kq .. +8, query 16 qb + r16
    fbf16x8_t qf[4][2][2];
#pragma unroll
    for (int qb = 0; qb < 2; qb++) {
        const int t = min(q0 + 16 * qb + r16, a.T - 1);
        const float* qp = a.q + (size_t)t * a.q_stride + (size_t)h * 128;
#pragma unroll
        for (int db = 0; db < 4; db++) {
            const float4 x0 = *reinterpret_cast<const float4*>(qp + 32 * db + 8 * kq);
            const float4 x1 = *reinterpret_cast<const float4*>(qp + 32 * db + 8 * kq + 4);
            uint32_t hi[4], lo[4];
            split2(x0.x * qscale, x0.y * qscale, hi[0], lo[0]);
            split2(x0.z * qscale, x0.w * qscale, hi[1], lo[1]);
            split2(x1.x * qscale, x1.y * qscale, hi[2], lo[2]);
            split2(x1.z * qscale, x1.w * qscale, hi[3], lo[3]);
            qf[db][qb][0] = __builtin_bit_cast(fbf16x8_t, uint4{hi[0], hi[1], hi[2], hi[3]});
            qf[db][qb][1] = __builtin_bit_cast(fbf16x8_t, uint4{lo[0], lo[1], lo[2], lo[3]});
        }
    }
    ff32x4_t o[8][2];                            // O^T: dims 16 n + 4 kq + i, query 16 qb + r16
#pragma unroll
    for (int n = 0; n < 8; n++)
#pragma unroll
        for (int qb = 0; qb < 2; qb++) o[n][qb] = ff32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    float m[2] = {-INFINITY, -INFINITY}, l[2] = {0.0f, 0.0f};

    auto tile = [&](auto EDGEC, int t) {
        constexpr bool EDGE = decltype(EDGEC)::value;
        const int k0 = t * 64;
        // lane parts of the K and V addresses, opaque: their XORs are taken where used, not kept for all
        // dims and keys across the tiles (registers that the fragments need)
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const uint32_t stage = (uint32_t)(t & 1) * 2 * F2_TILE, l15 = ln & 15, l4 = ln >> 4;
        const uint32_t kaddr = stage + l15 * 256 + 16 * (l4 ^ l15);                 // ^ 64 db + 4096 kb
        const uint32_t v15 = 4 * l4 + (l15 >> 2);                                  // key & 15 of the lane's V reads
        const uint32_t vaddr = stage + F2_TILE + v15 * 256 + 16 * (((l15 & 3) >> 1) ^ v15) + 8 * (l15 & 1);   // ^ 32 n + 4096 (2 st + r)

        // S^T tiles [kb][qb]: keys k0 + 16 kb + 4 kq + i, query 16 qb + r16; the next 16 keys' fragments are
        // read while these keys' products issue
        ff32x4_t s[4][2];
        fbf16x8_t ka[2][4];
        auto kread = [&](int kb) {
#pragma unroll
            for (int db = 0; db < 4; db++) ka[kb & 1][db] = *reinterpret_cast<const fbf16x8_t*>(f2_lds + ((kaddr ^ (64u * db)) + 4096u * kb));
        };
        kread(0);
#pragma unroll
        for (int kb = 0; kb < 4; kb++) {
            __builtin_amdgcn_sched_barrier(0);
            if (kb < 3) kread(kb + 1);
            s[kb][0] = s[kb][1] = ff32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int db = 0; db < 4; db++)
#pragma unroll
                for (int p = 0; p < 2; p++)
#pragma unroll
                    for (int qb = 0; qb < 2; qb++) s[kb][qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[kb & 1][db], qf[db][qb][p], s[kb][qb], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        // V^T fragments of (step st, 16 dims n) f = 8 st + n, two ahead of the products
        uint2 va[3][2];
        auto vread = [&](int f) {
#pragma unroll
            for (int r = 0; r < 2; r++)
                va[f % 3][r] = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((fp_lv4)(f2_lds + ((vaddr ^ (32u * (f & 7))) + 4096u * (2 * (f >> 3) + r)))));
        };
        // causal mask, base-2 online softmax
        uint32_t ph[2][2][4], pl[2][2][4];   // [st][qb] P^T fragments (hi, lo), 4 dwords each
#pragma unroll
        for (int qb = 0; qb < 2; qb++) {
            const int qpos = pos0 + q0 + 16 * qb + r16;
            float mx = -INFINITY;
#pragma unroll
            for (int kb = 0; kb < 4; kb++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if (EDGE && k0 + 16 * kb + 4 * kq + i > qpos) s[kb][qb][i] = -INFINITY;
                    mx = fmaxf(mx, s[kb][qb][i]);
                }
            mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            float alpha = 1.0f;
            if (__any(mx > m[qb])) {
                const float mn = fmaxf(m[qb], mx);
                alpha = mn == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m[qb] - mn);
                m[qb] = mn;
#pragma unroll
                for (int n = 0; n < 8; n++) o[n][qb] *= alpha;
            }
            const float ms = m[qb] == -INFINITY ? 0.0f : m[qb];   // no key yet: every p is 2^-inf
            float p[4][4], sum = 0.0f;
#pragma unroll
            for (int kb = 0; kb < 4; kb++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    p[kb][i] = __builtin_amdgcn_exp2f(s[kb][qb][i] - ms);
                    sum += p[kb][i];
                }
            l[qb] = l[qb] * alpha + xor32_sum(xor16_sum(sum));
            // k-slots of PV step st: 0..3 = keys 16 (2 st) + 4 kq + i, 4..7 = keys 16 (2 st + 1) + 4 kq + i
#pragma unroll
            for (int st = 0; st < 2; st++) {
                split2(p[2 * st][0], p[2 * st][1], ph[st][qb][0], pl[st][qb][0]);
                split2(p[2 * st][2], p[2 * st][3], ph[st][qb][1], pl[st][qb][1]);
                split2(p[2 * st + 1][0], p[2 * st + 1][1], ph[st][qb][2], pl[st][qb][2]);
                split2(p[2 * st + 1][2], p[2 * st + 1][3], ph[st][qb][3], pl[st][qb][3]);
            }
        }
        vread(0);
        vread(1);
#pragma unroll
        for (int st = 0; st < 2; st++) {
            fbf16x8_t pb[2][2];
#pragma unroll
            for (int qb = 0; qb < 2; qb++) {
                pb[qb][0] = __builtin_bit_cast(fbf16x8_t, uint4{ph[st][qb][0], ph[st][qb][1], ph[st][qb][2], ph[st][qb][3]});
                pb[qb][1] = __builtin_bit_cast(fbf16x8_t, uint4{pl[st][qb][0], pl[st][qb][1], pl[st][qb][2], pl[st][qb][3]});
            }
            // keys past the chunk's last key may hold anything: zero their V (their weight is 0, and
            // 0 * NaN is not)
            uint32_t vm[2][2];
            if constexpr (EDGE) {
#pragma unroll
                for (int r = 0; r < 2; r++)
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        const int left = kend - (k0 + 16 * (2 * st + r) + 4 * kq + 2 * e);   // keys of the pair that exist
                        vm[r][e] = left >= 2 ? ~0u : left == 1 ? 0xFFFFu : 0u;
                    }
            }
#pragma unroll
            for (int n = 0; n < 8; n++) {
                const int f = 8 * st + n;
                __builtin_amdgcn_sched_barrier(0);
                if (f + 2 < 16) vread(f + 2);
                if constexpr (EDGE) {
#pragma unroll
                    for (int r = 0; r < 2; r++) { va[f % 3][r].x &= vm[r][0]; va[f % 3][r].y &= vm[r][1]; }
                }
                const fbf16x8_t v8 = __builtin_bit_cast(fbf16x8_t, uint4{va[f % 3][0].x, va[f % 3][0].y, va[f % 3][1].x, va[f % 3][1].y});
#pragma unroll
                for (int p = 0; p < 2; p++)
#pragma unroll
                    for (int qb = 0; qb < 2; qb++) o[n][qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v8, pb[qb][p], o[n][qb], 0, 0, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    issue(0);
    auto next = [&](int t) {
        __builtin_amdgcn_s_waitcnt(0);       // this wave's copies of tile t landed ...
        __builtin_amdgcn_s_barrier();        // ... and every wave's; tile t - 1's stage is free
        if (t + 1 < all) issue(t + 1);
    };
    // whole tiles: every key of theirs is at or before the block's first query
    const int whole = min(ntiles, (pos0 + q0 + 1) / 64);
    int t = 0;
    for (; t < whole; t++) { next(t); tile(std::false_type{}, t); }
    for (; t < ntiles; t++) { next(t); tile(std::true_type{}, t); }
    for (; t < all; t++) next(t);
    if (!active) return;
#pragma unroll
    for (int qb = 0; qb < 2; qb++) {
        const int t = q0 + 16 * qb + r16;
        if (t >= a.T) continue;
        const float inv = 1.0f / l[qb];
        float* op = a.out + (size_t)t * a.out_stride + (size_t)h * 128 + 4 * kq;
#pragma unroll
        for (int n = 0; n < 8; n++)
            *reinterpret_cast<float4*>(op + 16 * n) = float4{o[n][qb][0] * inv, o[n][qb][1] * inv, o[n][qb][2] * inv, o[n][qb][3] * inv};
    }
}

hipError_t launch_flash_prefill(const FlashArgs& a, hipStream_t s) {
    if (a.D != 128 || a.nKV < 1 || a.nH % a.nKV || a.nH / a.nKV > 8 || a.T < 1) return hipErrorInvalidValue;
    FlashDev f{};
    f.a = a;
    f.nb = (a.T + 31) / 32;
    f.nwg = (a.nH / a.nKV * f.nb + 3) / 4;
    const int cus = device_cus(), total = f.nwg * a.nKV;
    f.first = total > cus && total <= 2 * cus ? cus / a.nKV : f.nwg;
    hipLaunchKernelGGL(flash_kernel, dim3(total), dim3(256), 4 * F2_TILE, s, f);
    return hipGetLastError();
}

}  // namespace mlxr
