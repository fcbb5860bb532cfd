// gemm_tile.hpp -- the tiled MFMA dequant-GEMM of the prompt pass, gfx950.
//
// y[M, N] = x[M, K] . W[N, K]^T, K % 32 == 0, W packed Q4_0 / Q8_0 or f16.
// A workgroup of 8 waves owns a BM x BN output tile: WM x WN waves side by
// side, each 32 TM x 32 TN in v_mfma_f32_32x32x16_f16 tiles, and G = 8 /
// (WM WN) groups of them that share the tile and split each K step (a
// 32-element quant block per wave and step).  What bounds it: the LDS
// ports, the address unit of the direct-to-LDS loads and the matrix cores are
// each 60 - 80 % busy in the K loop at 128 x 128, so the design spends as
// little as it can on the first two:
//  - The waves split K instead of a narrower tile each: an activation or
//    weight block then enters registers WN or WM times and not 4 and 2 times
//    (8 waves of 64 x 32 read 80 KB of LDS per 64 k at 128 x 128; two groups
//    of 2 x 2 waves of 64 x 64 read 48 KB; four groups of 1 x 2 waves of
//    128 x 64 read 40 KB and dequantise every weight once).
//  - K steps of 128 or 256: a row's piece is 256 or 512 consecutive bytes
//    (direct loads of 128-byte pieces reached 100 GB/s per CU, of 256-byte
//    pieces 166).
//  - The loads that refill a stage are spread over the MFMAs of the next
//    step; issued back to back after the barrier they stalled every wave at
//    the address unit (M = 512, [5632 x 2048] Q8_0: 23.7 -> 20.7 us).
//  - A step's scales are few bytes of many rows, and the load that brings
//    them costs the address unit and the memory as much as 1 KB of weights
//    does: they come for four steps at once, and the K loop is written four
//    steps to a round, so that nothing branches on it.  Weights out of HBM /
//    in the caches, a load of scales per step -> now, M = 512, K not split: Q8_0 [2560 x
//    10240] 86.5 / 62.5 -> 70.9 / 59.4 us, [7680 x 2560] 29.5 / 25.1 -> 27.5 /
//    25.1, Q4_0 [2560 x 10240] 70.2 / 61.8 -> 63.6 / 58.0 us (the short
//    [5632 x 2048] out of the caches went from 18.7 to 19.4, out of HBM from
//    23.0 to 21.5).
//  - The weights stay packed in LDS and are dequantised into registers
//    between the MFMAs of the sub-step before (RNE_f16((q - 8) d) /
//    RNE_f16(q d), the exact values of gguf.rs:22-112).
//  - The fp32 tiles of the groups meet in LDS and are added in group order by
//    an epilogue of 8 consecutive outputs per thread: 16-byte stores, and a
//    few hundred instructions where one unrolled over the accumulators was
//    7,800 (fetching them cost more than 10 us per launch).
// Measured (MI355X, back to back over three weight copies), a kernel
// of 64 x 32 waves / this one: M = 512 Q8_0 [5632 x 2048] 29.5 / 20.7 us (an
// f16 GEMM of the platform's library takes 20.1; out of HBM, over 24 copies, it
// takes 23.9 and this one 22.8), [7680 x 2560] 48 / 27, [2560 x 10240] 54 / 38 (in
// 4 and 3 slices of K), [2560 x 2560] 28 / 16; M = 400 Q4_0 [2048 x 2048]
// 24 / 9.5; M = 2048 Q4_0 [2048 x 5632] 74 / 49.
#pragma once

#include <type_traits>

#include "device_common.hpp"
#include "internal.hpp"

namespace tlhip {

struct TileParams {
    const uint16_t* x;
    const uint8_t* wq;
    const uint16_t* wd;
    const uint16_t* bias;
    const uint16_t* resid;
    uint16_t* y;
    float* part;   // fp32 partials [splits][M][N rounded up to 8] of a K split, else null
    int M, N, K, ldy, epi;
    int mT, nT, splits;
    int vec;       // EPI_QKV_ROPE: 8-column items share a head and a side of rot
    // EPI_QKV_ROPE: columns [0, nq) are q, [nq, nq + nk) k, the rest v; row m
    // is position pos0 + m (as the GEMV's fused epilogue)
    int nq, nk, head_dim, rot, layout, pos0;
    const float* rope_tab;
    uint16_t *q_out, *kc, *vc;
};

// sk_dma<16> with a scalar byte offset added to every lane's.
__device__ __forceinline__ void tile_dma(__amdgpu_buffer_rsrc_t r, uint32_t lds, uint32_t off, uint32_t soff) {
    lds = __builtin_amdgcn_readfirstlane(lds);
    soff = __builtin_amdgcn_readfirstlane(soff);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(off), "s"(r),
                 "s"(soff)
                 : "memory");
}

constexpr uint32_t SK_OOB = 0x80000000u;   // a buffer offset past every range

// Four payload bytes -> two f16 pairs in element order (e0,e1) (e2,e3).
__device__ __forceinline__ void q8_pairs(uint32_t w, h2 dd, uint32_t& p01, uint32_t& p23) {
    const h2 bias = {(h16)-1152.0f, (h16)-1152.0f};
    const uint32_t v = w ^ 0x80808080u;
    p01 = as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, v, 0x04010400u)) + bias) * dd);
    p23 = as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, v, 0x04030402u)) + bias) * dd);
}
__device__ __forceinline__ void q4_pairs(uint32_t nib, h2 dd, uint32_t& p01, uint32_t& p23) {
    const h2 bias = {(h16)-1032.0f, (h16)-1032.0f};
    p01 = as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, nib, 0x04010400u)) + bias) * dd);
    p23 = as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, nib, 0x04030402u)) + bias) * dd);
}
// The same for nibbles left in the high half of each byte (16 q under the
// exponent of 64: 64 + q, mantissa step 1/16).
__device__ __forceinline__ void q4_pairs_hi(uint32_t nib, h2 dd, uint32_t& p01, uint32_t& p23) {
    const h2 bias = {(h16)-72.0f, (h16)-72.0f};
    p01 = as_u32((as_h2(__builtin_amdgcn_perm(0x54545454u, nib, 0x04010400u)) + bias) * dd);
    p23 = as_u32((as_h2(__builtin_amdgcn_perm(0x54545454u, nib, 0x04030402u)) + bias) * dd);
}

// XOR applied to the 16-byte slot index of row r in an LDS region of rows
// of R bytes: 16 consecutive rows read at one chunk index fall in distinct
// 16-byte slots of the 256 bytes the banks serve at once.
template <int R>
__device__ __forceinline__ constexpr int tile_swz(int r) {
    constexpr int per_line = R >= 256 ? 1 : 256 / R;
    constexpr int mask = (R >= 256 ? 16 : R / 16) - 1;
    return (r / per_line) & mask;
}

template <int WT, int TM, int TN, int WM, int WN>
struct Tile {
    static constexpr int G = 8 / (WM * WN);            // K groups: waves that share an output tile
    static constexpr int NBK = G;                      // 32-element blocks of K per step, one per group
    static constexpr int BM = 32 * TM * WM, BN = 32 * TN * WN, BK = 32 * NBK;
    static constexpr int WB = WT == TLHIP_F16 ? 64 : (WT == TLHIP_Q8_0 ? 32 : 16);   // bytes of one 32-weight block
    static constexpr int AR = 64 * NBK, BR = WB * NBK; // LDS row bytes
    // The scales come a group of 4 steps at a time, in a ring of 2 groups: a
    // load instruction costs the address unit the same whether it brings 1 KB
    // or a step's few scales
    static constexpr int SG = 4;   // (the K loop spells its four steps out)
    static constexpr int SP = (SG * NBK / 2 + 1 + 3) / 4;   // 16-byte pieces that hold a row's scales, even or odd start
    static constexpr int SR = 16 * SP;                      // LDS row bytes
    static constexpr int A_BYTES = BM * AR, B_BYTES = BN * BR;
    static constexpr int SL = WT == TLHIP_F16 ? 0 : BN * SP / 8;   // pieces per wave and group
    static constexpr int NA = A_BYTES / 8192;          // 16-byte-per-lane loads per wave and stage
    static constexpr int BL = B_BYTES / 128;           // 16-byte pieces of B per wave
    static constexpr int NB = (BL + 63) / 64;
    static constexpr int C = NA + NB;                  // loads per wave and stage, without the scales
    // every load runs on all 64 lanes: lanes past a wave's part fetch the next
    // wave's first pieces (the same data to the same place), the last wave's
    // go to the padding after its region
    static constexpr int STAGE = A_BYTES + B_BYTES + 16 * (64 * NB - BL);
    static constexpr int SGROUP = SL ? 16 * (8 * SL + 64 - SL) : 0;
    static constexpr int ETM = TM < 2 ? TM : 2;        // M tiles of a wave that one pass of the epilogue takes
    static constexpr int EPI = 8 * ETM * TN * 4096;    // fp32 tiles of the 8 waves in one pass
    static constexpr int NS0 = (160 * 1024 - 2 * SGROUP) / STAGE;
    static constexpr int NS = NS0 < SG ? NS0 : SG;   // (the next group's scales go before its first stage)
    static constexpr int S_AT = NS * STAGE;
    static constexpr int LDS = S_AT + 2 * SGROUP > EPI ? S_AT + 2 * SGROUP : EPI;
    static_assert(A_BYTES % 8192 == 0 && B_BYTES % 128 == 0 && SL <= 64 && BN * SP % 8 == 0 && NBK % 2 == 0, "load shapes");
    static_assert(NS >= 2 && (NS - 1) * C + 2 < 64, "ring");
};

// EPI_QKV_ROPE of 8 consecutive projections n .. n + 7 (f16) of row m: the
// bias added, q and k pairs rotated and stored as the GEMV's fused epilogue
// does (layout 0: pairs in place; 1: columns 2i, 2i + 1 of a head are dims i
// and i + rot / 2), k and v into the cache rows.  p.vec: head_dim and rot
// multiples of 8, so the 8 columns share a head and a side of rot.
__device__ __forceinline__ void tile_rope8(const TileParams& p, int m, int n, uint16_t (&h)[8]) {
    const int pos = p.pos0 + m, D = p.head_dim, half = p.rot >> 1;
    if (p.bias) {
#pragma unroll
        for (int e = 0; e < 8; e++)
            if (n + e < p.N) h[e] = add_h(h[e], p.bias[n + e]);
    }
#pragma unroll
    for (int e = 0; e < 8; e += 2) {   // (p.vec: the addresses below advance by a constant)
        const int c = n + e;
        if (c + 1 >= p.N) break;
        if (c >= p.nq + p.nk) {
            if (p.vec && e == 0) {   // (N, nq and nk are then multiples of 8)
                u4 o;
#pragma unroll
                for (int k = 0; k < 4; k++) o[k] = (uint32_t)h[2 * k] | ((uint32_t)h[2 * k + 1] << 16);
                *(u4*)(p.vc + (size_t)pos * p.nk + c - p.nq - p.nk) = o;
                return;
            }
            p.vc[(size_t)pos * p.nk + c - p.nq - p.nk] = h[e];
            p.vc[(size_t)pos * p.nk + c - p.nq - p.nk + 1] = h[e + 1];
            continue;
        }
        const bool is_k = c >= p.nq;
        const int cc = is_k ? c - p.nq : c, el = cc % D;
        uint16_t* dst = is_k ? p.kc + (size_t)pos * p.nk + cc - el : p.q_out + (size_t)m * p.nq + cc - el;
        const bool turn = el < p.rot;
        if (p.vec && e == 0) {
            uint16_t a[4], b[4];   // first and second of each pair
#pragma unroll
            for (int k = 0; k < 4; k++) {
                a[k] = h[2 * k];
                b[k] = h[2 * k + 1];
                if (turn) {
                    const float* t = p.rope_tab + 2 * ((size_t)pos * half + (el >> 1) + k);
                    const float x0 = h2f(a[k]), x1 = h2f(b[k]), cs = t[0], sn = t[1];
                    a[k] = f2h(__fsub_rn(__fmul_rn(x0, cs), __fmul_rn(x1, sn)));
                    b[k] = f2h(__fadd_rn(__fmul_rn(x0, sn), __fmul_rn(x1, cs)));
                }
            }
            if (turn && p.layout) {
                const int i = el >> 1;
                *(uint2*)(dst + i) = uint2{(uint32_t)a[0] | ((uint32_t)a[1] << 16), (uint32_t)a[2] | ((uint32_t)a[3] << 16)};
                *(uint2*)(dst + i + half) = uint2{(uint32_t)b[0] | ((uint32_t)b[1] << 16), (uint32_t)b[2] | ((uint32_t)b[3] << 16)};
            } else {
                u4 o;
#pragma unroll
                for (int k = 0; k < 4; k++) o[k] = (uint32_t)a[k] | ((uint32_t)b[k] << 16);
                *(u4*)(dst + el) = o;
            }
            return;
        }
        if (turn) {
            const int i = el >> 1;
            const float* t = p.rope_tab + 2 * ((size_t)pos * half + i);
            const float x0 = h2f(h[e]), x1 = h2f(h[e + 1]), cs = t[0], sn = t[1];
            dst[p.layout ? i : el] = f2h(__fsub_rn(__fmul_rn(x0, cs), __fmul_rn(x1, sn)));
            dst[p.layout ? i + half : el + 1] = f2h(__fadd_rn(__fmul_rn(x0, sn), __fmul_rn(x1, cs)));
        } else {
            dst[el] = h[e];
            dst[el + 1] = h[e + 1];
        }
    }
}

// The epilogue (GemvEpi) of 8 consecutive outputs n .. n + 7 of row m (the
// last item of a row may hold fewer).
__device__ __forceinline__ void tile_store8(const TileParams& p, int m, int n, const float (&v)[8]) {
    const bool full = n + 8 <= p.N;
    uint16_t h[8];
#pragma unroll
    for (int e = 0; e < 8; e++) h[e] = f2h(v[e]);
    if (p.epi == EPI_SWIGLU_PAIR) {
        uint16_t* d = p.y + (size_t)m * p.ldy + n / 2;
        uint16_t o[4];
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = swiglu_h(h[2 * e], h[2 * e + 1]);
        if (full) {
            *(h4_any*)d = h4_any{{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16)}};
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n + 2 * e + 1 < p.N) d[e] = o[e];
        }
        return;
    }
    if (p.epi == EPI_QKV_ROPE) {
        tile_rope8(p, m, n, h);
        return;
    }
    const bool ub = p.epi == EPI_BIAS || p.epi == EPI_BIAS_RESID || p.epi == EPI_BIAS_GELU;
    const bool ur = p.epi == EPI_RESID || p.epi == EPI_BIAS_RESID;
    uint16_t* d = p.y + (size_t)m * p.ldy + n;
    const uint16_t* rs = p.resid + (size_t)m * p.N + n;
    h8_any b = {}, r = {};
    if (full) {
        if (ub) b = *(const h8_any*)(p.bias + n);
        if (ur) r = *(const h8_any*)rs;
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) {   // (columns past the row repeat its last)
            const int c = min(e, p.N - 1 - n);
            if (ub) b.w[e / 2] |= (uint32_t)p.bias[n + c] << (16 * (e & 1));
            if (ur) r.w[e / 2] |= (uint32_t)rs[c] << (16 * (e & 1));
        }
    }
    if (ub) {
#pragma unroll
        for (int e = 0; e < 8; e++) h[e] = add_h(h[e], (uint16_t)(b.w[e / 2] >> (16 * (e & 1))));
    }
    if (p.epi == EPI_BIAS_GELU) {
#pragma unroll
        for (int e = 0; e < 8; e++) h[e] = gelu_h(h[e]);
    }
    if (ur) {
#pragma unroll
        for (int e = 0; e < 8; e++) h[e] = add_h((uint16_t)(r.w[e / 2] >> (16 * (e & 1))), h[e]);
    }
    if (full) {
        h8_any o;
#pragma unroll
        for (int e = 0; e < 4; e++) o.w[e] = (uint32_t)h[2 * e] | ((uint32_t)h[2 * e + 1] << 16);
        *(h8_any*)d = o;
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++)
            if (n + e < p.N) d[e] = h[e];
    }
}

template <int V>
using Int = std::integral_constant<int, V>;

template <int WT, int TM, int TN, int WM, int WN>
__global__ __launch_bounds__(512) void gemm_tile_kernel(TileParams p) {
    using L = Tile<WT, TM, TN, WM, WN>;
    constexpr int G = L::G, BM = L::BM, BN = L::BN, NS = L::NS;
    __shared__ __attribute__((aligned(1024))) uint8_t smem[L::LDS];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = wave / (WM * WN), wm = wave % (WM * WN) / WN, wn = wave % WN;
    const int hh = lane >> 5, l32 = lane & 31;

    // workgroup -> tile: each XCD (workgroup id mod 8) takes a run of tiles;
    // a run walks groups of up to 4 M tiles, M fastest, so the tiles of one
    // XCD share their activation and weight rows in its L2
    const int T = p.mT * p.nT, total = T * p.splits;
    int q;
    {
        const int id = blockIdx.x, xcd = id & 7, s = id >> 3, per = total >> 3, rem = total & 7;
        q = xcd * per + min(xcd, rem) + s;
    }
    const int z = q / T, qt = q % T;
    const int g0 = qt / (4 * p.nT) * 4, gm = min(4, p.mT - g0), qg = qt - g0 * p.nT;
    const int m0 = (g0 + qg % gm) * BM, n0 = qg / gm * BN;
    const int nkt = (p.K + L::BK - 1) / L::BK;
    const int kt0 = (int)((int64_t)nkt * z / p.splits), nk = (int)((int64_t)nkt * (z + 1) / p.splits) - kt0;
    const int nbr = p.K >> 5;
    const uint32_t xrow = 2u * p.K, wrow = (uint32_t)nbr * L::WB;
    const int mrows = min(BM, p.M - m0), nrows = min(BN, p.N - n0);

    // rows past M / N lie past the buffers' ranges: zeros, no memory access
    const __amdgpu_buffer_rsrc_t rx = sk_rsrc(p.x + (size_t)m0 * p.K, (uint32_t)mrows * xrow);
    const __amdgpu_buffer_rsrc_t rw = sk_rsrc(p.wq + (size_t)n0 * wrow, (uint32_t)nrows * wrow);
    // (n0 is even: 4-byte aligned)
    const __amdgpu_buffer_rsrc_t rd = sk_rsrc(WT == TLHIP_F16 ? (const void*)p.wq : (const void*)(p.wd + (size_t)n0 * nbr),
                                              WT == TLHIP_F16 ? 0u : (uint32_t)(nrows * nbr * 2 + 3) & ~3u);

    // source offset of this lane's piece of each load at step kt0
    uint32_t asrc[L::NA], bsrc[L::NB], ssrc = 0;
#pragma unroll
    for (int u = 0; u < L::NA; u++) {
        const int P = (u * 8 + wave) * 64 + lane, r = P / (L::AR / 16), c = (P % (L::AR / 16)) ^ tile_swz<L::AR>(r);
        asrc[u] = (uint32_t)r * xrow + 16u * c + (uint32_t)kt0 * L::AR;
    }
#pragma unroll
    for (int u = 0; u < L::NB; u++) {
        const int P = wave * L::BL + 64 * u + lane;
        const int r = P / (L::BR / 16), c = (P % (L::BR / 16)) ^ tile_swz<L::BR>(r);
        bsrc[u] = (uint32_t)r * wrow + 16u * c + (uint32_t)kt0 * L::BR;
    }
    if constexpr (L::SL > 0) {
        const int P = wave * L::SL + lane, n = P / L::SP, c = P % L::SP;
        ssrc = 4u * ((uint32_t)(n * nbr + kt0 * L::NBK) / 2u) + 16u * c;
    }
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(gl_lds_t)smem);

    // Load d (of L::C) of step kt0 + step into ring slot `slot`: fixed lane
    // offsets, the step in the scalar offset.  Steps past the last go to an
    // offset outside the buffers (zeros, no memory access), so that every
    // wait counts the same loads; the scales of a group of steps go before its
    // first stage.  (Pieces past K in a partial last step hold
    // whatever follows in the tile's buffer; no wave computes on those blocks.)
    auto issue = [&](int d, int step, int slot) {
        const uint32_t base = lds0 + (uint32_t)slot * L::STAGE;
        const uint32_t dead = step < nk ? 0u : SK_OOB;
        const uint32_t st = step < nk ? (uint32_t)step : 0u;
        if (d < L::NA)
            tile_dma(rx, base + 1024u * (d * 8 + wave), asrc[d < L::NA ? d : 0] | dead, st * L::AR);
        else
            tile_dma(rw, base + L::A_BYTES + 16u * (wave * L::BL + 64 * (d - L::NA)),
                         bsrc[d >= L::NA && d < L::NA + L::NB ? d - L::NA : 0] | dead, st * L::BR);
    };

    auto issue_scales = [&](int grp) {
        if constexpr (L::SL > 0)
            tile_dma(rd, lds0 + L::S_AT + (uint32_t)(grp & 1) * L::SGROUP + 16u * L::SL * wave,
                         ssrc | (grp * L::SG < nk ? 0u : SK_OOB), (grp * L::SG < nk ? (uint32_t)grp : 0u) * (2u * L::SG * L::NBK));
    };

    // operand offsets inside a stage.  This wave's block of a step is g; at
    // MFMA sub-step t lane half hh holds 8 of its 32 elements, A and B alike:
    //   f16   16 t + 8 hh ..   (16 bytes per sub-step)
    //   Q8_0  16 hh + 8 t ..   (16 bytes give both sub-steps)
    //   Q4_0  16 t + 8 hh ..   (8 bytes: low nibbles t = 0, high t = 1)
    int aoff[TM][2], boff[TN][2], soff[TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int m = 32 * (wm * TM + i) + l32;
            const int c = 4 * g + (WT == TLHIP_Q8_0 ? 2 * hh + t : 2 * t + hh);
            aoff[i][t] = m * L::AR + 16 * (c ^ tile_swz<L::AR>(m));
        }
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int n = 32 * (wn * TN + j) + l32;
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int c = WT == TLHIP_F16 ? 4 * g + 2 * t + hh : (WT == TLHIP_Q8_0 ? 2 * g + hh : g);
            boff[j][t] = L::A_BYTES + n * L::BR + 16 * (c ^ tile_swz<L::BR>(n)) + (WT == TLHIP_Q4_0 ? 8 * hh : 0);
        }
        soff[j] = L::S_AT + L::SR * n + 2 * ((n * nbr & 1) + g);
    }

    // Operands of the block in registers: activations and dequantised weights
    // of both MFMA sub-steps, and the block's packed weights and scales.
    h8 oa[TM][2], ob[TN][2];
    u4 rawb[TN];
    uint32_t raws[TN];
    auto read = [&](int soffs, int slot, int t) {
        const uint8_t* st = smem + slot * L::STAGE;
#pragma unroll
        for (int j = 0; j < TN; j++) {
            if constexpr (WT == TLHIP_F16) {
                ob[j][t] = *(const h8*)(st + boff[j][t]);
            } else if (t == 0) {
                if constexpr (WT == TLHIP_Q8_0) {
                    rawb[j] = *(const u4*)(st + boff[j][0]);
                } else {
                    const uint2 v = *(const uint2*)(st + boff[j][0]);
                    rawb[j][0] = v.x;
                    rawb[j][1] = v.y;
                }
                raws[j] = *(const uint16_t*)(smem + soff[j] + soffs);
            }
        }
#pragma unroll
        for (int i = 0; i < TM; i++) oa[i][t] = *(const h8*)(st + aoff[i][t]);
    };
    // piece q (two per weight tile: four weights each) of sub-step t
    auto dequant = [&](int q, int t) {
        const int j = q / 2, h = q % 2;
        const h16 dh = __builtin_bit_cast(h16, (uint16_t)raws[j]);
        const h2 dd = {dh, dh};
        uint32_t p01, p23;
        if (WT == TLHIP_Q8_0) q8_pairs(rawb[j][2 * t + h], dd, p01, p23);
        else if (t == 0) q4_pairs(rawb[j][h] & 0x0F0F0F0Fu, dd, p01, p23);
        else q4_pairs_hi(rawb[j][h] & 0xF0F0F0F0u, dd, p01, p23);
        asm volatile("" : "+v"(p01), "+v"(p23));   // here, not where the MFMA wants it
        u4 v = __builtin_bit_cast(u4, ob[j][t]);
        v[2 * h] = p01;
        v[2 * h + 1] = p23;
        ob[j][t] = __builtin_bit_cast(h8, v);
    };

    f16v acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = f16v{0};

    // The MFMAs of sub-step t (consecutive ones on different accumulators);
    // between the later ones the dequantisation of the next sub-step, whose
    // LDS reads were issued before (an MFMA holds the matrix core for eight
    // vector issue slots), and loads [d0, d1) of stage `step`, spread out
    // because back to back they would stall the wave at the address unit.
    constexpr int NM = TM * TN, NP = WT == TLHIP_F16 ? 0 : 2 * TN;
    auto mma = [&](int t, bool next, int d0, int d1, int step, int dslot, int grp = -1) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < NM; e++) {
            const int j = e / TM, i = e % TM;
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ob[j][t], oa[i][t], acc[i][j], 0, 0, 0);
            if (grp >= 0 && e == 0) issue_scales(grp);
#pragma unroll
            for (int d = d0 + e * (d1 - d0) / NM; d < d0 + (e + 1) * (d1 - d0) / NM; d++) issue(d, step, dslot);
            constexpr int E0 = NM / 2 - 1;
            if (next && e >= E0) {
#pragma unroll
                for (int q = (e - E0) * NP / (NM - E0); q < (e - E0 + 1) * NP / (NM - E0); q++) dequant(q, 1 - t);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // K loop.  Ring of NS stages.  During a step's last sub-step the next
    // stage's first operands are read, after a barrier at which every wave
    // has read the whole stage: its slot is then refilled with the stage NS
    // steps on, over the sub-steps up to the next barrier.
    // Four steps to a round of the loop: where a group of scales is issued and
    // read is then fixed, and nothing branches inside.
    constexpr int D1 = L::C / 2, W = (NS - 2) * L::C;
    issue_scales(0);
#pragma unroll
    for (int s = 0; s < NS; s++)
#pragma unroll
        for (int d = 0; d < (s + 1 < NS ? L::C : D1); d++) issue(d, s, s);
    sk_wait_vm<W + D1>();
    lds_barrier();
    read(0, 0, 0);
#pragma unroll
    for (int q = 0; q < NP; q++) dequant(q, 0);
    int slot = 0, prev = NS - 1, i = 0, sgo = 0;   // sgo: LDS offset of the group of step i
    auto step = [&](auto wait, int ph, bool scales) {
        const int nslot = slot + 1 == NS ? 0 : slot + 1;
        read(0, slot, 1);
        mma(0, true, D1, L::C, i - 1 + NS, prev);
        sk_wait_vm<decltype(wait)::value>();   // stage i + 1 has landed (loads complete in order)
        lds_barrier();
        read(ph + 1 == L::SG ? L::SGROUP - sgo : sgo + (ph + 1) * 2 * L::NBK, nslot, 0);
        mma(1, true, 0, D1, i + NS, slot, scales ? i / L::SG + 1 : -1);
        prev = slot;
        slot = nslot;
        i++;
    };
    while (i + L::SG < nk) {
        // the scales that step 0 issues may still be under way at the waits
        // for the stages issued before them
        constexpr int S = L::SL ? 1 : 0;
        step(Int<W>{}, 0, true);
        step(Int<W + (NS > 2 ? S : 0)>{}, 1, false);
        step(Int<W + (NS > 3 ? S : 0)>{}, 2, false);
        step(Int<W>{}, 3, false);
        sgo = L::SGROUP - sgo;
    }
    for (int ph = 0, left = nk - 1 - i; ph < left; ph++) step(Int<W>{}, ph, false);
    // the last step, if this wave's block lies inside K
    if (g < nbr - (kt0 + nk - 1) * L::NBK) {
        read(0, slot, 1);
        mma(0, true, 0, 0, 0, 0);
        mma(1, false, 0, 0, 0, 0);
    }
    sk_wait_vm<0>();   // the ring becomes the epilogue's buffer

    // The waves' fp32 tiles to LDS as [group][m][n] rows (C layout of the
    // transposed product: lane = activation row, 4 consecutive n per
    // register quad), then 8 consecutive n per thread: the groups summed in
    // order, the epilogue, 16-byte stores.
    constexpr int ER = BN * 4, VPR = BN / 8;   // row bytes, 8-column items per row
    constexpr int ETM = L::ETM, EM = 32 * ETM * WM;
#pragma unroll
    for (int ps = 0; ps < TM / ETM; ps++) {
        lds_barrier();
#pragma unroll
        for (int ii = 0; ii < ETM; ii++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const f16v& c = acc[ps * ETM + ii][j];
                    const int m = 32 * (wm * ETM + ii) + l32, s = 8 * (wn * TN + j) + 2 * r + hh;
                    *(f4*)(smem + (size_t)(g * EM + m) * ER + 16 * (s ^ tile_swz<ER>(m))) =
                        f4{c[4 * r], c[4 * r + 1], c[4 * r + 2], c[4 * r + 3]};
                }
        lds_barrier();
#pragma unroll 1
        for (int it = tid; it < EM * VPR; it += 512) {
            const int er = it / VPR, c8 = it % VPR;
            const int m = m0 + er / (32 * ETM) * (32 * TM) + ps * 32 * ETM + er % (32 * ETM), n = n0 + 8 * c8;
            float v[8];
#pragma unroll
            for (int gi = 0; gi < G; gi++) {
                const uint8_t* row = smem + (size_t)(gi * EM + er) * ER;
                const f4 a = *(const f4*)(row + 16 * ((2 * c8) ^ tile_swz<ER>(er)));
                const f4 b = *(const f4*)(row + 16 * ((2 * c8 + 1) ^ tile_swz<ER>(er)));
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    v[e] = gi ? v[e] + a[e] : a[e];
                    v[4 + e] = gi ? v[4 + e] + b[e] : b[e];
                }
            }
            if (m >= p.M || n >= p.N) continue;
            if (p.part) {
                float* d = p.part + ((size_t)z * p.M + m) * ((p.N + 7) & ~7) + n;
                *(f4*)d = f4{v[0], v[1], v[2], v[3]};
                *(f4*)(d + 4) = f4{v[4], v[5], v[6], v[7]};
                continue;
            }
            tile_store8(p, m, n, v);
        }
    }
}

}  // namespace tlhip
