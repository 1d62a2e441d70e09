// qsa_prefill_full.hip -- prefill attention of queries that attend every block
// up to their position: a dense layer's, and a sparse one's while the sink,
// top-k and window blocks still cover the sequence (a prompt's first
// thousands of tokens).  There neighbouring queries read the same tiles, so a
// workgroup takes a block of queries over each 64-cell tile at once: the
// tile is read and widened to fp16 once for all of them, and every column of
// the matrix cores carries a (query, head).
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "qsa_device.h"

namespace qwfn_qsa {

namespace {

// The page layouts (as qsa_dec_kernel.h): q8_0 with V dim-major per 64-token
// tile, q8_0 with V in the K layout, q4_0 and F16.
constexpr int kPlQ8 = 0, kPlQ8K = 1, kPlQ4 = 2, kPlF16 = 3;

constexpr int kFullPUp = 14;             // the weights enter PV as p * 2^14
constexpr int kFullVTop = 15;            // the V values as V * 2^kv, below 2^15

// A workgroup: GR groups of four waves, group u taking tiles u, u + GR, ... of
// the workgroup's queries; wave w of a group owns NCT 16-column tiles, a
// column one (query, head) of the KV head's group.
template <int HD, int G, int LY>
struct FullCfg {
    static constexpr int NJ = HD / 32, ND = HD / 16, NG = HD / 8;
    static constexpr int NCT = HD <= 128 ? 2 : 1;          // O and the query fragments fit 256 VGPRs
    static constexpr int GR = HD <= 128 && LY != kPlF16 ? 2 : 1;   // two groups' buffers fit the LDS
    static constexpr int COLS = 4 * NCT * 16, QB = COLS / G;   // columns, queries a workgroup
    static constexpr int THREADS = 256 * GR;
    static constexpr bool SCALED = LY != kPlF16;           // K and V are quants times scales
    static constexpr int VP = SCALED ? 2 : 1;              // V planes: fp16 high and low parts
    // bytes of 8 cells of every dim.  The operand reads want groups at the same
    // banks; the K layouts' stores, 16 cell quads a dim at a time, want them
    // spread (64).
    static constexpr int VGRP = HD * 16 + (LY == kPlQ8 ? 0 : 64);
    static constexpr int VPLANE = 8 * VGRP;
    static constexpr int KCH = LY == kPlQ4 ? HD / 32 : LY == kPlF16 ? HD / 8 : HD / 16;   // 16-byte chunks of a row
    static constexpr int KPIECES = KCH * 64 / 256;         // chunks a thread converts a tile
    // kPlQ8: the 32-dim V blocks that a wave's HD / 4 dims lie in (at HD 64 two waves
    // share a block), and the floats of its own strip of their scales, 64 cells each.
    static constexpr int NBW = HD > 128 ? HD / 128 : 1, VSTRIP = 64 * NBW;
    static_assert(G <= COLS && KCH * 64 % 256 == 0, "whole pieces");
};

// A group's tile, in two LDS objects (so the compiler sees that K's traffic and
// V's never meet): K as [dim / 8][cell] 16-byte units of 8 dims (the quants,
// exact in fp16) with its scales, and V as [8 cells][dim] units of the cells a
// lane of the PV operand takes (dequantized, times 2^kv, as fp16 high + low
// parts).
template <int HD, int G, int LY>
struct FullK {
    using C = FullCfg<HD, G, LY>;
    u4v k[C::NG * 64];
    __attribute__((aligned(16))) uint16_t s[C::SCALED ? 64 * C::NJ : 8];
};
template <int HD, int G, int LY>
struct FullV {
    using C = FullCfg<HD, G, LY>;
    float d[LY == kPlQ8 ? 4 * C::VSTRIP : 4];   // kPlQ8: a strip a wave of the tile's V scales times 2^kv
    // (two groups' tiles also hold a group's O at the end)
    static constexpr int BYTES = C::VP * C::VPLANE, XCH = C::GR == 2 ? 4 * C::NCT * C::ND * 1024 / 2 : 0;
    __attribute__((aligned(16))) uint8_t v[BYTES > XCH ? BYTES : XCH];
};
// The tile's bytes as they lie in the pages, where the transfers land: K with its
// scale rows, V with its.
template <int HD, int G, int LY>
struct FullRaw {
    using C = FullCfg<HD, G, LY>;
    static constexpr int SB = C::SCALED ? 64 * C::NJ * 2 : 0;      // bytes of the tile's scales
    u4v k[C::KCH * 64 + (SB > 0 ? 64 : 0)], v[C::KCH * 64 + (SB > 0 ? 64 : 0)];
    static_assert(SB <= 1024 && C::KCH % 4 == 0, "whole transfers a wave");
};
// Cells some queries may not see (a step's parity each): the dims where V is not
// finite, a bit each.
template <int HD>
struct FullBad {
    uint32_t cell[2][64][HD / 32];
    int any[2];
};

// A workgroup barrier that orders LDS traffic only: global loads stay in flight
// across it.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Two quants packed in a word times their V scales (fp32, 2^kv included) as
// packed fp16 high and low parts, hi = f16(d q), lo = f16(d q - hi): d q has at
// most 19 significant bits, so hi + lo is exact while lo is not below fp16's
// smallest step.
__device__ __forceinline__ void dq_split2(float d0, float d1, uint32_t w, uint32_t &hi, uint32_t &lo) {
    asm("v_fma_mixlo_f16 %0, %1, %2, 0 op_sel_hi:[0,1,0]" : "=v"(hi) : "v"(d0), "v"(w));
    asm("v_fma_mixlo_f16 %0, %1, %2, -%3 op_sel_hi:[0,1,1]" : "=v"(lo) : "v"(d0), "v"(w), "v"(hi));
    asm("v_fma_mixhi_f16 %0, %1, %2, 0 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "+v"(hi) : "v"(d1), "v"(w));
    asm("v_fma_mixhi_f16 %0, %1, %2, -%3 op_sel:[0,1,1] op_sel_hi:[0,1,1]" : "+v"(lo) : "v"(d1), "v"(w), "v"(hi));
}

// Two fp32 weights as packed fp16 high and low parts.
__device__ __forceinline__ void p_split(float p0, float p1, uint32_t &hi, uint32_t &lo) {
    asm("v_cvt_f16_f32 %0, %1" : "=v"(hi) : "v"(p0));
    asm("v_fma_mixlo_f16 %0, %1, 1.0, -%2 op_sel_hi:[0,0,1]" : "=v"(lo) : "v"(p0), "v"(hi));
    asm("v_fma_mixhi_f16 %0, %1, 1.0, 0 op_sel_hi:[0,0,0]" : "+v"(hi) : "v"(p1));
    asm("v_fma_mixhi_f16 %0, %1, 1.0, -%2 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "+v"(lo) : "v"(p1), "v"(hi));
}

__device__ __forceinline__ u4v h8_words(h8v x) { return __builtin_bit_cast(u4v, x); }

// Bytes of a q4_0 chunk's four dims 4 r .. 4 r + 3 (r < 8) as nibbles, one a byte.
__device__ __forceinline__ uint32_t q4_nibbles(uint32_t w, bool high) {
    return high ? (w >> 4) & 0x0f0f0f0fu : w & 0x0f0f0f0fu;
}

__device__ __forceinline__ void q4x4_h2(uint32_t w, half2v &lo, half2v &hi) {
    const half2v bias = {(_Float16)-1032.0f, (_Float16)-1032.0f};
    lo = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, w, 0x04010400u)) + bias;
    hi = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, w, 0x04030402u)) + bias;
}

__device__ __forceinline__ bool f16_bad(uint32_t half) { return (half & 0x7c00u) == 0x7c00u; }   // inf or NaN

// grid (ceil(n_q / QB) * Hkv), GR * 256 threads: query block (of QB queries,
// the longest first) and KV head.  Query i of the launch is at position
// pf_pos0 + i and attends every cell up to it; vmax from k_pf_vmax over every
// row (SCALED).  Per 64-cell tile, on v_mfma_f32_16x16x32_f16:
//  - QK: S[cell][column] = sum_j dk(cell, j) (K_j[cell][:] . q_j[:, column])
//    with the key quants exact in fp16 and the query, scaled by a power of
//    two, as fp16 high + low parts: exact products, two MFMAs a 32-dim block,
//    the block's scale applied in fp32 (F16: no scales, one chain, the low parts first);
//  - PV: O[dim][column] += V[dim][cell] P[cell][column] with V = dv q 2^kv and P =
//    p 2^14 each as fp16 high + low parts, hi hi + hi lo + lo hi (lo lo is below
//    2^-24 of the product).  Dequantizing V costs an MFMA more than folding
//    its scale into the weights but is shared by every query of the block, where
//    the weights' fold is not: 64 VALU instructions a wave and tile against 256.
//  - The cells' order along PV's k is the QK accumulator's (cells 4 lg .. 4 lg + 3
//    of two 16-cell groups), so the weights stay in their lanes; V is laid
//    out for it.
// A step of a group has two halves between barriers: softmax and the conversions
// (the tile's V and the next tile's K, from their raw bytes in LDS), then PV
// and the next tile's QK with the next transfers in flight.  The second group
// runs half a step behind, so each SIMD has one wave in either half (in
// phase: 179 against 167 us a 3,001-query call).  A tile some queries may
// not see (the diagonal) has its non-finite V values, at cells past the
// block's first query, replaced by 0 and the columns that do see them set to
// NaN afterwards, so no query reads a later token's row.  The groups' states
// merge through LDS at the end.
// Bound: a step takes about 5 us, 160 MFMAs (2,560 cycles) and 660 VALU
// instructions a wave, each wave's LDS reads and chains exposed at two waves a SIMD
// (its 256 VGPRs hold O, the query and a unit of operands ahead).  Measured: 3,001
// queries from position 0, 16 x 128 heads, 403 -> 155 us the call against one wave a
// (query, KV head) (QK and PV 92 -> 239 TFLOP/s).  Stores of a dim's cells that met
// at one bank took it to 166 us, twelve-MFMA units with twice the operands ahead,
// which spill, to 160 us.
template <int HD, int G, int LY>
__global__ void __launch_bounds__((FullCfg<HD, G, LY>::THREADS))
k_pf_full(Geo g, qwfn_kv_view v, const float *__restrict__ q, int32_t n_q, const float *__restrict__ vmax,
          float *__restrict__ out) {
    using C = FullCfg<HD, G, LY>;
    constexpr int NJ = C::NJ, ND = C::ND, NCT = C::NCT, GR = C::GR, QB = C::QB;
    __shared__ FullK<HD, G, LY> shk[GR];
    __shared__ FullV<HD, G, LY> shv[GR];
    __shared__ FullRaw<HD, G, LY> shr[GR];
    __shared__ FullBad<HD> shb[GR];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
    const int grp = wv >> 2, w = wv & 3, tid = threadIdx.x & 255;
    FullK<HD, G, LY> &TK = shk[grp];
    FullV<HD, G, LY> &TV = shv[grp];
    FullRaw<HD, G, LY> &TR = shr[grp];
    FullBad<HD> &TB = shb[grp];
    const int hn = l & 15, lg = l >> 4;
    const int nqb = (n_q + QB - 1) / QB;
    const int gh = __builtin_amdgcn_readfirstlane((int)blockIdx.x % g.Hkv);
    const int qb = nqb - 1 - __builtin_amdgcn_readfirstlane((int)blockIdx.x / g.Hkv);
    const int q0 = qb * QB, q_last = min(q0 + QB, n_q) - 1;
    const int pos_first = g.pf_pos0 + q0, pos_last = g.pf_pos0 + q_last;

    // ---- the columns: queries, positions, fp16 query fragments
    int lim[NCT];                                    // the column's last visible position
    float lscale[NCT];
    h8v qh[NCT][NJ], ql[NCT][NJ];
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) {
        const int c = 16 * (NCT * w + ct) + hn;
        const int qi = min(q0 + c / G, q_last);
        lim[ct] = g.pf_pos0 + qi;
        const float *qrow = q + ((int64_t)qi * g.H + gh * G + c % G) * HD + 8 * lg;
        float x[NJ][8], amax = 0.0f;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const float4 a = *reinterpret_cast<const float4 *>(qrow + 32 * j);
            const float4 b = *reinterpret_cast<const float4 *>(qrow + 32 * j + 4);
            x[j][0] = a.x; x[j][1] = a.y; x[j][2] = a.z; x[j][3] = a.w;
            x[j][4] = b.x; x[j][5] = b.y; x[j][6] = b.z; x[j][7] = b.w;
#pragma unroll
            for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(x[j][i]));
        }
        amax = col_max4(amax);
        int ex = 0;
        frexpf(amax, &ex);
        const float qs = amax > 0.0f ? ldexpf(1.0f, ex - 14) : 1.0f;   // |q / qs| < 2^14
        const float qinv = 1.0f / qs;                // a power of two: exact
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float y = x[j][i] * qinv;
                const _Float16 hi = (_Float16)y;
                qh[ct][j][i] = hi;
                ql[ct][j][i] = (_Float16)(y - (float)hi);
            }
        lscale[ct] = qs * g.scale_log2;
    }
    // 2^kv brings the head's largest finite V value below 2^15 (|quant| <= 128)
    float v_up = 1.0f, v_down = 1.0f;
    if constexpr (C::SCALED) {
        const float dvm = wave_max(vmax[gh * kVmaxWg + l % kVmaxWg]);
        int e2 = 0;
        frexpf(dvm, &e2);
        if (dvm > 0.0f) {
            v_up = ldexpf(1.0f, kFullVTop - 7 - e2);
            v_down = ldexpf(1.0f, e2 + 7 - kFullVTop);
        }
    }

    f4v o[NCT][ND];
    float m[NCT], lsum[NCT];
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) {
#pragma unroll
        for (int d = 0; d < ND; ++d) o[ct][d] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
        m[ct] = -1e30f;
        lsum[ct] = 0.0f;
    }

    // ---- tile transfers: the group's waves move a tile's bytes to its raw
    // buffer as 1 KB global -> LDS transfers that hold no registers
    const int n_tiles = pos_last / 64 + 1;
    const int cq = tid & 15, dq = tid >> 4;          // V: cells 4 cq .. 4 cq + 3, dims by dq
    const auto lds_addr = [](const void *p) {
        return (uint32_t)__builtin_amdgcn_readfirstlane((int)(uintptr_t)(const __attribute__((address_space(3))) void *)p);
    };
    const uint32_t rk = lds_addr(&TR.k[0]), rv = lds_addr(&TR.v[0]);
    // lane l: the page of the group's tile number base + l (-1: none), looked up
    // for 64 tiles at once.  A tile without a page (past the last, or unmapped)
    // reads page 0, in bounds, and every column is masked.
    int pg_l = -1, tl_l = 0;                         // and the tile's place in the page
    auto look_up = [&](int base) {
        const int t = (base + l) * GR + grp;
        pg_l = -1;
        tl_l = 0;
        if (t < n_tiles) {
            pg_l = phys_page(g, v.page_table, g.pf_seq, t * 64);
            tl_l = t % (g.pt / 64);
            if (pg_l < 0) set_status(v.status, QWFN_STATUS_PAGE_RANGE);
        }
    };
    auto load = [&](int n, const void *pages, uint32_t dst) {
        const int pg = max(__builtin_amdgcn_readlane(pg_l, n & 63), 0);
        const int tl = __builtin_amdgcn_readfirstlane(gh * (g.pt / 64) + __builtin_amdgcn_readlane(tl_l, n & 63));
        const uint8_t *page = (const uint8_t *)pages + (int64_t)pg * g.page_bytes;
        const uint8_t *src = page + (int64_t)tl * C::KCH * 1024;
#pragma unroll
        for (int i = 0; i < C::KCH / 4; ++i) {
            const int c = w * (C::KCH / 4) + i;
            lds_dma16_sv(src + c * 1024, 16 * l, dst + c * 1024);
        }
        if constexpr (C::SCALED)
            if (w == 0 && l < FullRaw<HD, G, LY>::SB / 16)
                lds_dma16_sv(page + g.qbytes + (int64_t)tl * FullRaw<HD, G, LY>::SB, 16 * l, dst + C::KCH * 1024);
    };
    // the group's tile number n
    auto load_k = [&](int n) { load(n, v.k_pages, rk); };
    auto load_v = [&](int n) { load(n, v.v_pages, rv); };
    // ---- conversions into the group's tile
    auto store_k = [&]() {
#pragma unroll
        for (int i = 0; i < C::KPIECES; ++i) {
            const int cell = l, ch = 4 * i + w;      // chunk ch of the tile's cell
            const u4v kr = TR.k[ch * 64 + cell];
            if constexpr (LY == kPlF16) {
                TK.k[ch * 64 + cell] = kr;
            } else if constexpr (LY == kPlQ4) {
#pragma unroll
                for (int n = 0; n < 4; ++n) {        // dims 8 n .. 8 n + 7 of the block
                    half2v a, b, c, d;
                    q4x4_h2(q4_nibbles(kr[2 * (n % 2)], n >= 2), a, b);
                    q4x4_h2(q4_nibbles(kr[2 * (n % 2) + 1], n >= 2), c, d);
                    TK.k[(4 * ch + n) * 64 + cell] =
                        u4v{__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                            __builtin_bit_cast(uint32_t, c), __builtin_bit_cast(uint32_t, d)};
                }
            } else {
                TK.k[(2 * ch) * 64 + cell] = h8_words(q8x8_to_h8(make_uint2(kr[0], kr[1])));
                TK.k[(2 * ch + 1) * 64 + cell] = h8_words(q8x8_to_h8(make_uint2(kr[2], kr[3])));
            }
        }
        if constexpr (C::SCALED)
            if (tid < 64 * NJ * 2 / 16) reinterpret_cast<u4v *>(TK.s)[tid] = TR.k[C::KCH * 64 + tid];
    };
    // four cells' fp16 parts of dim d (high, then low) to their places: cells 4 cq + e
    // are elements 4 (mb % 2) + e of unit (mb / 2, lane group cq % 4), mb = cq / 4
    // A thread's dims are a first one (by dq) plus a constant each, so every address
    // is one register and an immediate.
    uint8_t *const vdst = TV.v + ((cq >> 3) * 4 + (cq & 3)) * C::VGRP + ((cq >> 2) & 1) * 8 + 4 * dq * 16;
    auto put_v = [&](int d, const uint32_t (&x)[2 * C::VP]) {
        *reinterpret_cast<uint2 *>(vdst + d * 16) = make_uint2(x[0], x[1]);
        if constexpr (C::VP == 2) *reinterpret_cast<uint2 *>(vdst + C::VPLANE + d * 16) = make_uint2(x[2], x[3]);
    };
    const uint8_t *const vsrc = reinterpret_cast<const uint8_t *>(&TR.v[0]) + 64 * cq +
                                (LY == kPlF16  ? (dq / 2) * 1024 + 8 * (dq % 2)
                                 : LY == kPlQ4 ? (dq / 8) * 1024 + 4 * (dq % 4)
                                               : (dq / 4) * 1024 + 4 * (dq % 4));
    // kPlQ8: lane (dim l / 4, 16-cell quarter l % 4) of wave w converts the quarter's
    // cells of dims HD / 4 w + l / 4 + 16 i, so the raw rows are read and the units
    // written without bank conflicts and a wave needs the scales of its own dims'
    // blocks alone.  put(16 i, lane group, parts): cells 4 lg .. + 3 of the quarter.
    const int vdim0 = HD / 4 * w + (l >> 2), vquarter = l & 3;
    uint8_t *const vdst8 = TV.v + (vquarter >> 1) * 4 * C::VGRP + (vquarter & 1) * 8 + vdim0 * 16;
    auto put_v8 = [&](int d, int lgx, const uint32_t (&x)[4]) {
        *reinterpret_cast<uint2 *>(vdst8 + lgx * C::VGRP + d * 16) = make_uint2(x[0], x[1]);
        *reinterpret_cast<uint2 *>(vdst8 + C::VPLANE + lgx * C::VGRP + d * 16) = make_uint2(x[2], x[3]);
    };
    auto conv_v8 = [&](auto put) {
        constexpr int NP = HD / 64, NBW = C::NBW;    // dims a thread, blocks a wave
        static_assert(LY != kPlQ8 || (4 * C::VSTRIP <= (int)(sizeof TV.d / sizeof TV.d[0]) && 32 * NBW >= HD / 4),
                      "four waves' strips of scales lie in the array, and hold their dims' blocks");
        const uint16_t *sc = reinterpret_cast<const uint16_t *>(&TR.v[C::KCH * 64]);
        float *strip = TV.d + w * C::VSTRIP;         // the wave's own
#pragma unroll
        for (int b = 0; b < NBW; ++b) strip[64 * b + l] = h2f(sc[l * NJ + HD / 4 * w / 32 + b]) * v_up;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");   // (a wave's LDS operations are in order)
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
#pragma unroll
        for (int b = 0; b < NBW; ++b) {
            f4v ds[4];
#pragma unroll
            for (int lgx = 0; lgx < 4; ++lgx)
                ds[lgx] = *reinterpret_cast<const f4v *>(strip + 64 * b + 16 * vquarter + 4 * lgx);
#pragma unroll
            for (int i = b * (NP / NBW); i < (b + 1) * (NP / NBW); ++i) {
                const u4v x16 = TR.v[(vdim0 + 16 * i) * 4 + vquarter];
#pragma unroll
                for (int lgx = 0; lgx < 4; ++lgx) {
                    half2v a, c;
                    q8x4_to_h2(x16[lgx], a, c);
                    uint32_t x[4];
                    dq_split2(ds[lgx][0], ds[lgx][1], __builtin_bit_cast(uint32_t, a), x[0], x[2]);
                    dq_split2(ds[lgx][2], ds[lgx][3], __builtin_bit_cast(uint32_t, c), x[1], x[3]);
                    put(16 * i, lgx, x);
                }
            }
        }
    };
    // the K layouts: each dim's four cells handed to put(dim - 4 dq, parts)
    auto conv_v = [&](auto put) {
        float ds[C::SCALED ? 4 : 1][NJ];             // dv 2^kv of the four cells
        if constexpr (C::SCALED) {
#pragma unroll
            for (int i = 0; i < NJ / 2; ++i) {
                const h8v x = __builtin_bit_cast(h8v, TR.v[C::KCH * 64 + cq * (NJ / 2) + i]);
#pragma unroll
                for (int k = 0; k < 8; ++k) ds[(8 * i + k) / NJ][(8 * i + k) % NJ] = (float)x[k] * v_up;
            }
        }
        {
#pragma unroll
            for (int i = 0; i < HD / 64; ++i) {
                uint32_t hw[4][2], lw[4][2];         // cell e's dims 4 (dq + 16 i) + {0, 1}, {2, 3}
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if constexpr (LY == kPlF16) {
                        const uint2 x = *reinterpret_cast<const uint2 *>(vsrc + 8 * i * 1024 + 16 * e);
                        hw[e][0] = x.x;
                        hw[e][1] = x.y;
                        lw[e][0] = lw[e][1] = 0u;
                    } else {
                        half2v a, b;
                        // (q4_0: a chunk is a block, its high nibbles dims 16 .. 31)
                        const uint32_t x = *reinterpret_cast<const uint32_t *>(vsrc + (LY == kPlQ4 ? 2 : 4) * i * 1024 + 16 * e);
                        if constexpr (LY == kPlQ4) q4x4_h2(q4_nibbles(x, dq % 8 >= 4), a, b);
                        else                       q8x4_to_h2(x, a, b);
                        // the dims' block is 2 i or 2 i + 1 by dq / 8
                        const float d = dq >= 8 ? ds[e][2 * i + 1] : ds[e][2 * i];
                        dq_split2(d, d, __builtin_bit_cast(uint32_t, a), hw[e][0], lw[e][0]);
                        dq_split2(d, d, __builtin_bit_cast(uint32_t, b), hw[e][1], lw[e][1]);
                    }
                }
#pragma unroll
                for (int k = 0; k < 4; ++k) {        // dim 4 (dq + 16 i) + k of the four cells
                    const uint32_t sel = k % 2 ? 0x07060302u : 0x05040100u;
                    uint32_t x[2 * C::VP];
                    x[0] = __builtin_amdgcn_perm(hw[1][k / 2], hw[0][k / 2], sel);
                    x[1] = __builtin_amdgcn_perm(hw[3][k / 2], hw[2][k / 2], sel);
                    if constexpr (C::VP == 2) {
                        x[2] = __builtin_amdgcn_perm(lw[1][k / 2], lw[0][k / 2], sel);
                        x[3] = __builtin_amdgcn_perm(lw[3][k / 2], lw[2][k / 2], sel);
                    }
                    put(64 * i + k, x);
                }
            }
        }
    };
    auto store_v = [&](int n, bool paged) {
        const int t0 = (n * GR + grp) * 64;
        if (t0 + 63 <= pos_first && paged) {
            if constexpr (LY == kPlQ8) conv_v8(put_v8);
            else                       conv_v(put_v);
            return;
        }
        // a diagonal tile: cells past the block's first query are not every
        // column's, so their non-finite values leave the tile and are flagged (a
        // tile without a page: all of them, unflagged)
        auto clean = [&](int cell0, int dim, uint32_t (&x)[2 * C::VP]) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int cell = cell0 + e;
                if ((t0 + cell > pos_first || !paged) && f16_bad(x[e / 2] >> (16 * (e % 2)))) {
                    const uint32_t keep = e % 2 ? 0x0000ffffu : 0xffff0000u;
                    x[e / 2] &= keep;
                    if constexpr (C::VP == 2) x[2 + e / 2] &= keep;
                    if (paged) {
                        atomicOr(&TB.cell[n & 1][cell][dim / 32], 1u << (dim % 32));
                        TB.any[n & 1] = 1;
                    }
                }
            }
        };
        if constexpr (LY == kPlQ8)
            conv_v8([&](int d, int lgx, uint32_t (&x)[4]) {
                clean(16 * vquarter + 4 * lgx, vdim0 + d, x);
                put_v8(d, lgx, x);
            });
        else
            conv_v([&](int d, uint32_t (&x)[2 * C::VP]) {
                clean(4 * cq, 4 * dq + d, x);
                put_v(d, x);
            });
    };

    f4v sv[NCT][4];                                  // the logits of a tile (before lscale)
    auto qk = [&]() {
        auto read_k = [&](int mb, h8v (&kf)[NJ]) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) kf[j] = __builtin_bit_cast(h8v, TK.k[(4 * j + lg) * 64 + 16 * mb + hn]);
        };
        if constexpr (C::SCALED) {
            // a step (mb, ct) issues its eight MFMAs, independent chains first,
            // with the scale sums of the step before; a 16-cell group's
            // operands are read behind the last MFMAs of the one before
            // it (the compiler's own order waits for every read and
            // product in turn)
            h8v kf[NJ], dk[NJ / 2];              // dk: cells 16 mb + 4 lg .. + 3, every block
            f4v c[NJ];
            auto read_d = [&](int mb) {
#pragma unroll
                for (int i = 0; i < NJ / 2; ++i)
                    dk[i] = reinterpret_cast<const h8v *>(TK.s)[(16 * mb + 4 * lg) * NJ / 8 + i];
            };
            auto sum = [&](int step) {           // step = mb NCT + ct
                const int mb = step / NCT;
                f4v acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int j = 0; j < NJ; ++j)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        acc[i] = __builtin_fmaf((float)dk[(i * NJ + j) / 8][(i * NJ + j) % 8],
                                                c[j][i], acc[i]);
                asm volatile("" : "+v"(acc));    // computed here, not sunk to its use
                sv[step % NCT][mb] = acc;
            };
            read_k(0, kf);
            read_d(0);
#pragma unroll
            for (int step = 0; step < 4 * NCT; ++step) {
                const int mb = step / NCT, ct = step % NCT;
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < NJ; ++j)
                    c[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[j], qh[ct][j],
                                                                            f4v{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
                for (int j = 0; j < NJ; ++j)
                    c[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[j], ql[ct][j], c[j], 0, 0, 0);
                if (ct == NCT - 1 && mb < 3) {
                    __builtin_amdgcn_sched_barrier(0);
                    read_k(mb + 1, kf);
                }
                sum(step);
                if (ct == NCT - 1 && mb < 3) read_d(mb + 1);
            }
        } else {
#pragma unroll
            for (int mb = 0; mb < 4; ++mb) {
                h8v kf[NJ];
                read_k(mb, kf);
#pragma unroll
                for (int ct = 0; ct < NCT; ++ct) sv[ct][mb] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
                // the low parts' sum first: a product of the high parts' sums rounds at the
                // logit's size, one of the low parts' at 2^-11 of it
#pragma unroll
                for (int j = 0; j < NJ; ++j)
#pragma unroll
                    for (int ct = 0; ct < NCT; ++ct)
                        sv[ct][mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[j], ql[ct][j], sv[ct][mb], 0, 0, 0);
#pragma unroll
                for (int j = 0; j < NJ; ++j)
#pragma unroll
                    for (int ct = 0; ct < NCT; ++ct)
                        sv[ct][mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[j], qh[ct][j], sv[ct][mb], 0, 0, 0);
            }
        }
    };

    auto clear_bad = [&](int par) {
        for (int i = tid; i < 64 * NJ; i += 256) (&TB.cell[par][0][0])[i] = 0u;
        if (tid == 0) TB.any[par] = 0;
    };
    clear_bad(0);
    clear_bad(1);
    const int steps = (n_tiles + GR - 1) / GR;
    look_up(0);
    load_k(0);
    load_v(0);
    bool mine = __builtin_amdgcn_readlane(pg_l, 0) >= 0;   // (uniform over the group) step st's tile has a page
    wait_vmem_all();
    lds_barrier();                                   // the tile's bytes are in place, the flags are clear
    store_k();
    lds_barrier();                                   // K is in place, its bytes are read
    load_k(1);
    qk();
    wait_vmem_all();
    lds_barrier();                                   // K is read, the next one's bytes are in place
    // the second group runs half a step behind: its vector half beside the
    // first one's matrix half
    if (GR == 2 && grp == 1) lds_barrier();
    for (int st = 0; st < steps; ++st) {
        const int t = st * GR + grp;
        const bool diag = t * 64 + 63 > pos_first || !mine;   // not every column sees every cell
        uint32_t ph[NCT][4][2], pl[NCT][4][2];       // the weights' parts, a 16-cell group's four cells a pair of words
        // ---- the vector half: softmax, then the tiles' conversions (V's and
        // K's last readers passed the barrier before it) and the next loads
        if (diag) {                                  // cells past a column's query
            asm volatile("" ::);                     // (a branch, not 32 selects every tile)
#pragma unroll
            for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
                for (int mb = 0; mb < 4; ++mb)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (!mine || t * 64 + 16 * mb + 4 * lg + i > lim[ct]) sv[ct][mb][i] = -INFINITY;
        }
        // ---- online softmax
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) {
            float tm = -INFINITY;
#pragma unroll
            for (int mb = 0; mb < 4; ++mb)
#pragma unroll
                for (int i = 0; i < 4; ++i) tm = fmaxf(tm, sv[ct][mb][i]);
            tm = col_max4(tm) * lscale[ct];      // lscale > 0: the max commutes
            const float m_new = fmaxf(m[ct], tm);
            const float alpha = __builtin_amdgcn_exp2f(m[ct] - m_new);
            const float bias = (float)kFullPUp - m_new;
            float tsum = 0.0f;
#pragma unroll
            for (int mb = 0; mb < 4; ++mb) {
                float p[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    p[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[ct][mb][i], lscale[ct], bias));
                    tsum += p[i];
                }
                p_split(p[0], p[1], ph[ct][mb][0], pl[ct][mb][0]);
                p_split(p[2], p[3], ph[ct][mb][1], pl[ct][mb][1]);
            }
            lsum[ct] = lsum[ct] * alpha + col_sum4(tsum);
            m[ct] = m_new;
            if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
                for (int d = 0; d < ND; ++d) o[ct][d] *= alpha;
            }
        }
        store_v(st, mine);
        store_k();
        mine = __builtin_amdgcn_readlane(pg_l, (st + 1) & 63) >= 0;
        lds_barrier();                               // this tile's V and the next one's K are in place, their bytes read
        load_v(st + 1);
        if (((st + 2) & 63) == 0) look_up(st + 2);
        load_k(st + 2);
        // ---- the matrix half: PV, then the next tile's QK
        // ---- PV: unit u = (16 dims u / 2, 32 cells u % 2), operands read one unit
        // ahead of their MFMAs
        h8v va[2][C::VP];
        auto read_v = [&](int u) {
#pragma unroll
            for (int x = 0; x < C::VP; ++x)
                va[u % 2][x] = *reinterpret_cast<const h8v *>(TV.v + x * C::VPLANE + (4 * (u % 2) + lg) * C::VGRP +
                                                              (16 * (u / 2) + hn) * 16);
        };
        read_v(0);
#pragma unroll
        for (int u = 0; u < 2 * ND; ++u) {
            if (u + 1 < 2 * ND) read_v(u + 1);
            __builtin_amdgcn_sched_barrier(0);
            const int d = u / 2, ks = u % 2;
            h8v bh[NCT], bl[NCT];
#pragma unroll
            for (int ct = 0; ct < NCT; ++ct) {
                bh[ct] = __builtin_bit_cast(
                    h8v, u4v{ph[ct][2 * ks][0], ph[ct][2 * ks][1], ph[ct][2 * ks + 1][0], ph[ct][2 * ks + 1][1]});
                bl[ct] = __builtin_bit_cast(
                    h8v, u4v{pl[ct][2 * ks][0], pl[ct][2 * ks][1], pl[ct][2 * ks + 1][0], pl[ct][2 * ks + 1][1]});
            }
            const h8v *vu = va[u % 2];
#pragma unroll
            for (int ct = 0; ct < NCT; ++ct) o[ct][d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vu[0], bh[ct], o[ct][d], 0, 0, 0);
#pragma unroll
            for (int ct = 0; ct < NCT; ++ct) o[ct][d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vu[0], bl[ct], o[ct][d], 0, 0, 0);
            if constexpr (C::VP == 2)
#pragma unroll
                for (int ct = 0; ct < NCT; ++ct)
                    o[ct][d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vu[1], bh[ct], o[ct][d], 0, 0, 0);
        }
        if (diag && TB.any[st & 1]) {            // (rare) non-finite rows some columns see
            for (int cell = 0; cell < 64; ++cell) {
#pragma unroll
                for (int d = 0; d < ND; ++d) {
                    // this lane's dims 16 d + 4 lg .. + 3
                    const uint32_t b = TB.cell[st & 1][cell][d / 2] >> (16 * (d % 2) + 4 * lg) & 15u;
#pragma unroll
                    for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            if ((b >> i & 1u) && t * 64 + cell <= lim[ct]) o[ct][d][i] = NAN;
                }
            }
        }
        clear_bad((st + 1) & 1);                     // (read a step ago, set past the next barrier)
        if (st + 1 < steps) qk();
        wait_vmem_all();
        lds_barrier();                               // both are read, the next bytes in place
    }
    if (GR == 2 && grp == 0) lds_barrier();
    // ---- the groups' states: group 1's into group 0's
    if constexpr (GR == 2) {
        float *xo = reinterpret_cast<float *>(&shv[0]), *xm = reinterpret_cast<float *>(&shk[0]);
        static_assert(4 * NCT * ND * 1024 <= (int)sizeof shv && 4 * NCT * 512 <= (int)sizeof shk,
                      "the exchange fits the tiles");
        if (grp == 1) {
#pragma unroll
            for (int ct = 0; ct < NCT; ++ct) {
                const int at = w * NCT + ct;
#pragma unroll
                for (int d = 0; d < ND; ++d) *reinterpret_cast<f4v *>(xo + (at * ND + d) * 256 + 4 * l) = o[ct][d];
                xm[at * 128 + l] = m[ct];
                xm[at * 128 + 64 + l] = lsum[ct];
            }
        }
        lds_barrier();
        if (grp == 1) return;
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) {
            const int at = w * NCT + ct;
            const float m1 = xm[at * 128 + l], l1 = xm[at * 128 + 64 + l];
            const float mx = fmaxf(m[ct], m1);
            const float a0 = __builtin_amdgcn_exp2f(m[ct] - mx), a1 = __builtin_amdgcn_exp2f(m1 - mx);
            lsum[ct] = lsum[ct] * a0 + l1 * a1;
#pragma unroll
            for (int d = 0; d < ND; ++d)
                o[ct][d] = o[ct][d] * a0 + *reinterpret_cast<const f4v *>(xo + (at * ND + d) * 256 + 4 * l) * a1;
        }
    }
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) {
        const int c = 16 * (NCT * w + ct) + hn;
        if (c >= QB * G || q0 + c / G > q_last) continue;
        const float inv = lsum[ct] > 0.0f ? v_down / lsum[ct] : 0.0f;
        float *orow = out + ((int64_t)(q0 + c / G) * g.H + gh * G + c % G) * HD;
#pragma unroll
        for (int d = 0; d < ND; ++d) *reinterpret_cast<f4v *>(orow + 16 * d + 4 * lg) = o[ct][d] * inv;
    }
}
template <int HD, int G, int LY>
void launch_full_t(const Geo &g, const qwfn_kv_view &v, const float *q, int32_t n_q, const float *vmax, float *out,
                   hipStream_t st) {
    using C = FullCfg<HD, G, LY>;
    const unsigned nqb = (unsigned)((n_q + C::QB - 1) / C::QB);
    hipLaunchKernelGGL((k_pf_full<HD, G, LY>), dim3(nqb * (unsigned)g.Hkv), dim3(C::THREADS), 0, st, g, v, q, n_q, vmax,
                       out);
}

// The layout of a shape with an instance, or -1.
int full_layout(const Geo &g) {
    if (g.kt == QWFN_KV_Q8_0) return g.vdim ? kPlQ8 : g.hd == 256 && g.G == 12 ? kPlQ8K : -1;
    return g.hd == 128 && g.G == 8 ? (g.kt == QWFN_KV_Q4_0 ? kPlQ4 : kPlF16) : -1;
}

}  // namespace

// Measured against the per-query kernels (us a call, whole calls of 2 KV heads on
// 256 CUs; per-query kernel / this one).  A workgroup here walks its tiles in series, 5
// us a step of two tiles, so a call of few queries is better split over them.
//   q8_0, whose per-query kernel splits a query over waves while a call leaves CUs
//     idle: 16 x 128 dense 512 after 9,000 tokens 306 / 396, 520 388 / 398, 700 455 /
//     405, 1,000 611 / 418, 3,001 from 0 403 / 155; 16 x 64 dense 512 after 9,000 191 /
//     244, 520 244 / 244; 16 x 256 512 after 9,000 796 / 662, 24 x 256 925 / 672.  The
//     line is where that kernel stops sharing pairs: past four a CU, at 256 dims (half
//     the waves a CU) from four.
//   The K layouts' per-query kernel (k_dec_loop) is a workgroup a pair whose time goes
//     in steps with the workgroups a CU, and a call whose every query attends every
//     block also saves its selection here, so the line moves with the length: dense F16
//     512 after 9,000 368 / 441, 520 469 / 441, 700 from 0 49 / 50, 1,000 75 / 65; dense
//     q4_0 512 from 0 38 / 50, 1,000 81 / 75, 512 after 1,500 109 / 118, 600 130 / 124,
//     512 after 15,000 725 / 700; the checkpoint layer 384 after 1,000 130 / 138, 450
//     158 / 142, 1,000 329 / 264.  Both sides' times are estimated.
constexpr int64_t kFullPairsCu = 4, kFullPairsCuK = 3;    // (query, KV head) pairs a CU: the lines (K: no fewer)

// What the estimates are made of, us: this kernel's start and its time a tile, and
// k_dec_loop's time a tile, a part of its own and a part for each pair a CU.
// Fitted over 240 calls of 1, 2 and 8 KV heads, 64 to 2,000 queries after 0 to 30,000
// tokens: the side taken is the faster one or within 8% of it in all but eight.
struct FullCost { float full0, full, loop, loop_cu; };
constexpr FullCost kFullCostQ8K = {23.0f, 4.95f, 0.6f, 1.15f}, kFullCostQ4 = {28.0f, 2.8f, 0.5f, 0.62f},
                   kFullCostF16 = {18.0f, 2.86f, 0.1f, 0.58f};
constexpr float kLoop0 = 14.0f;          // k_dec_loop's start

// This kernel over n queries from position pos0, `wgs` workgroups, the longest first:
// the rounds before the last one at the mean length of theirs, the last one at its own.
float full_us(const FullCost &c, int64_t pos0, int64_t n, int64_t wgs) {
    const int64_t cus = device_cus(), rounds = (wgs + cus - 1) / cus;
    const float t = (float)((pos0 + n + 63) / 64), t0 = (float)(pos0 / 64);
    const float before = (float)((rounds - 1) * cus) / (float)wgs;
    const float walk = (float)(rounds - 1) * (t - (t - t0) * before * 0.5f) + t0 + (t - t0) * (1.0f - before) * 0.5f;
    return c.full0 + c.full * std::max(t, rounds > 1 ? walk : 0.0f);
}

// k_dec_loop over `pairs` of tiles t0 .. t: up to four workgroups a CU side by side, the
// ones after them at the mean length.
float loop_us(const FullCost &c, int64_t pairs, int64_t pos0, int64_t end) {
    if (pairs <= 0) return 0.0f;
    const int64_t cus = device_cus(), a_cu = (pairs + cus - 1) / cus;
    const float t = (float)((end + 63) / 64), t0 = (float)(pos0 / 64);
    return kLoop0 + t * (c.loop + c.loop_cu * (float)std::min<int64_t>(a_cu, 4)) +
           c.loop_cu * (float)std::max<int64_t>(a_cu - 4, 0) * 0.5f * (t0 + t);
}

int32_t pf_full_queries(const Geo &g, int32_t pos0, int32_t n_q, float sel_us) {
    const int ly = full_layout(g);
    if (ly < 0) return 0;
    const int64_t most = g.topk <= 0 ? (int64_t)pos0 + n_q : all_kept_len(g);
    const int64_t n = std::max<int64_t>(0, std::min<int64_t>(n_q, most - pos0));
    const int64_t pairs = n * g.Hkv, cus = device_cus();
    if (ly == kPlQ8) return pairs > kFullPairsCu * cus - (g.hd > 128 ? 1 : 0) ? (int32_t)n : 0;
    if (pairs < kFullPairsCuK * cus) return 0;
    const FullCost &c = ly == kPlQ8K ? kFullCostQ8K : ly == kPlQ4 ? kFullCostQ4 : kFullCostF16;
    const int qb = (g.hd > 128 ? 64 : 128) / g.G;          // FullCfg's queries a workgroup
    // a call's other queries (they attend a selection) take k_dec_loop either way
    const int64_t rest = (int64_t)n_q - n, end = std::min((int64_t)pos0 + n_q, most);
    const float full = full_us(c, pos0, n, (n + qb - 1) / qb * g.Hkv) + loop_us(c, rest * g.Hkv, end, end);
    const float loop = loop_us(c, (int64_t)n_q * g.Hkv, pos0, end) + (rest == 0 ? sel_us : 0.0f);
    return full <= loop ? (int32_t)n : 0;
}

hipError_t launch_prefill_full(const Geo &g, const qwfn_kv_view &v, const float *q, int32_t n_q, const float *vmax,
                               float *out, hipStream_t st) {
#define QWFN_FULL(HD_, G_, LY_)                                             \
    if (g.hd == HD_ && g.G == G_ && full_layout(g) == LY_) {                \
        launch_full_t<HD_, G_, LY_>(g, v, q, n_q, vmax, out, st);           \
        return hipGetLastError();                                           \
    }
    QWFN_FULL(128, 8, kPlQ8)
    QWFN_FULL(128, 4, kPlQ8)
    QWFN_FULL(128, 2, kPlQ8)
    QWFN_FULL(64, 8, kPlQ8)
    QWFN_FULL(256, 12, kPlQ8)
    QWFN_FULL(256, 8, kPlQ8)
    QWFN_FULL(256, 12, kPlQ8K)
    QWFN_FULL(128, 8, kPlQ4)
    QWFN_FULL(128, 8, kPlF16)
#undef QWFN_FULL
    return hipErrorInvalidValue;
}

}  // namespace qwfn_qsa
