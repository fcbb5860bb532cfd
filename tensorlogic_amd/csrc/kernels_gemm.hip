// kernels_gemm.hip -- dequant-GEMM for prefill (M > 4) on MFMA, gfx950.
//
// y[M, N] = x[M, K] . W[N, K]^T, W packed Q4_0 / Q8_0 or f16: activation and
// weight tiles staged in LDS, weights dequantised to RNE_f16((q-8)*d) /
// RNE_f16(q*d) (the exact values of gguf.rs:22-112), fp32 accumulation on the
// matrix cores as the reference's tiled matmul does (unified.metal:
// 4291-4348), output f16 with the same epilogues as the GEMV (bias, residual
// add, SwiGLU on interleaved gate/up rows, QKV + RoPE + cache).
//
// gemm_tile_kernel (gemm_tile.hpp, kernels_gemm_tile.hip) takes every K that
// is a multiple of 32; gemm_skinny_kernel (below) the M <= 64 shapes where it
// is the faster one: a ring of LDS stages per wave filled by direct
// global->LDS loads, split over K with a fence-free exchange;
// gemm_staged_kernel (kernels_gemm_staged.hip) many tiles of a short K.  gemm_kernel
// (64 x 64 x 32 tiles) covers rows too long for the tiled kernel's buffer
// ranges, gemm_naive_kernel f16 weights whose K is no multiple of 32.  Here
// too: linear() on f32 tensors.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "gemm_tile.hpp"

namespace tlhip {

struct GemmParams {
    const uint16_t* x;
    const uint8_t* wq;
    const uint16_t* wd;
    const uint16_t* bias;
    const uint16_t* resid;
    uint16_t* y;
    int M, N, K, ldy, epi;
    // skinny GEMM split over K: fp32 partials [splits][M][N] and one arrival
    // counter per 32-row tile (zero between launches)
    float* part = nullptr;
    uint32_t* flags = nullptr;
    int splits = 1;
    int mtiles = 1;   // skinny GEMM: workgroups along M
    // skinny GEMM, EPI_QKV_ROPE: columns [0, nq) are q, [nq, nq + nk) k, the
    // rest v; row m is position pos0 + m (as the GEMV's fused epilogue)
    int nq = 0, nk = 0, head_dim = 0, rot = 0, layout = 0, pos0 = 0;
    const float* rope_tab = nullptr;
    uint16_t* q_out = nullptr;
    uint16_t* kc = nullptr;
    uint16_t* vc = nullptr;
};

constexpr int GBM = 64, GBN = 64, GBK = 32, GPAD = 8;

typedef h16 h4 __attribute__((ext_vector_type(4)));

template <int WT>
__global__ __launch_bounds__(256) void gemm_kernel(GemmParams p) {
    __shared__ __attribute__((aligned(16))) uint16_t As[GBM][GBK + GPAD];
    __shared__ __attribute__((aligned(16))) uint16_t Bs[GBN][GBK + GPAD];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int m0 = blockIdx.y * GBM, n0 = blockIdx.x * GBN;
    const int nbr = p.K >> 5;
    f16v acc = {0};

    const int lr = tid >> 2, lq = tid & 3;   // loader row, quarter
    for (int kb = 0; kb < nbr; kb++) {
        // activation tile: 64 rows x 32 halves, 16 B per thread
        {
            const int m = m0 + lr;
            u4 v = {0u, 0u, 0u, 0u};
            if (m < p.M) v = *(const u4*)(p.x + (size_t)m * p.K + (size_t)kb * 32 + lq * 8);
            *(u4*)&As[lr][lq * 8] = v;
        }
        // weight tile: 64 rows x one block, dequantised into LDS
        {
            const int n = min(n0 + lr, p.N - 1);
            if (WT == TLHIP_Q4_0) {
                const uint8_t* qb = p.wq + (size_t)n * (p.K / 2) + (size_t)kb * 16;
                uint32_t w = *(const uint32_t*)(qb + 4 * lq);
                h16 dh = __builtin_bit_cast(h16, p.wd[(size_t)n * nbr + kb]);
                h2 dd = {dh, dh}, r[4];
                q4_unpack(w, dd, r);
                // r0=(e4q,e4q+2) r1=(e4q+1,e4q+3) r2/r3 the same at +16
                *(uint32_t*)&Bs[lr][4 * lq + 0] = pack_lo(as_u32(r[0]), as_u32(r[1]));
                *(uint32_t*)&Bs[lr][4 * lq + 2] = pack_hi(as_u32(r[0]), as_u32(r[1]));
                *(uint32_t*)&Bs[lr][16 + 4 * lq + 0] = pack_lo(as_u32(r[2]), as_u32(r[3]));
                *(uint32_t*)&Bs[lr][16 + 4 * lq + 2] = pack_hi(as_u32(r[2]), as_u32(r[3]));
            } else if (WT == TLHIP_Q8_0) {
                const uint8_t* qb = p.wq + (size_t)n * p.K + (size_t)kb * 32 + 8 * lq;
                uint32_t w0 = *(const uint32_t*)qb, w1 = *(const uint32_t*)(qb + 4);
                h16 dh = __builtin_bit_cast(h16, p.wd[(size_t)n * nbr + kb]);
                h2 dd = {dh, dh}, r[2];
                q8_unpack(w0, dd, r);
                *(uint32_t*)&Bs[lr][8 * lq + 0] = pack_lo(as_u32(r[0]), as_u32(r[1]));
                *(uint32_t*)&Bs[lr][8 * lq + 2] = pack_hi(as_u32(r[0]), as_u32(r[1]));
                q8_unpack(w1, dd, r);
                *(uint32_t*)&Bs[lr][8 * lq + 4] = pack_lo(as_u32(r[0]), as_u32(r[1]));
                *(uint32_t*)&Bs[lr][8 * lq + 6] = pack_hi(as_u32(r[0]), as_u32(r[1]));
            } else {
                const uint16_t* wr = (const uint16_t*)p.wq + (size_t)n * p.K + (size_t)kb * 32 + 8 * lq;
                *(u4*)&Bs[lr][8 * lq] = *(const u4*)wr;
            }
        }
        __syncthreads();
        // 4 x mfma 32x32x8: A rows (wm*32 + lane%32), B rows (wn*32 + lane%32)
#pragma unroll
        for (int ks = 0; ks < GBK; ks += 8) {
            const int kk = ks + 4 * (lane >> 5);
            h4 a = *(const h4*)&As[wm * 32 + (lane & 31)][kk];
            h4 b = *(const h4*)&Bs[wn * 32 + (lane & 31)][kk];
            acc = __builtin_amdgcn_mfma_f32_32x32x8f16(a, b, acc, 0, 0, 0);
        }
        __syncthreads();
    }

    // C layout: col j = lane%32 (weight row), row i = 8*(r/4) + 4*(lane/32) + r%4
    const int n = n0 + wn * 32 + (lane & 31);
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int m = m0 + wm * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        float v = acc[r];
        if (p.epi == EPI_SWIGLU_PAIR) {
            float up = __shfl_down(v, 1, 64);
            if (m < p.M && n + 1 < p.N && (n & 1) == 0)
                p.y[(size_t)m * p.ldy + n / 2] = swiglu_h(f2h(v), f2h(up));
        } else if (m < p.M && n < p.N) {
            p.y[(size_t)m * p.ldy + n] = epilogue_h(p.epi, v, p.bias, p.resid, (size_t)m * p.N + n, n);
        }
    }
}

// ---------------------------------------------------------------------------
// Skinny dequant-GEMM (4 < M <= 64, K % 64 == 0) on v_mfma_f32_16x16x32_f16:
// one launch, no workspace by default.  A workgroup reads its activation
// rows and weight rows once; both enter the CU as whole 64-byte pieces,
// because the vector L1 handles a load one piece per lane-run of adjacent
// addresses: an MFMA operand read straight from a row-major matrix (one row
// per lane) costs one L1 access per lane, here one per 64 bytes.  What
// bounds it is the bytes each CU takes in: the activation rows (which every
// workgroup of the same rows re-reads) plus its own weight rows.  The host
// plan (sk_plan) picks per shape how many 16-row M tiles a workgroup covers
// (MT) and how many 16-row weight tiles (NT), so that the largest per-CU
// byte count is smallest.
//
// A workgroup (4 waves) owns MT x 16 activation rows and 16 NT weight rows;
// wave w takes K part w (the workgroup's 64-k steps split into 4 ranges) for
// all of them.  Each wave streams its part through a private ring of L::ST
// LDS stages with buffer loads to LDS (16 bytes per lane, adjacent lanes on
// adjacent bytes; the 16-byte pieces of a row XOR-swizzled by row so the
// operand reads below spread over the banks), then reads the operands of
// sub-step t = 0, 1 in the natural 16 x 16 x 32 layout -- lane l (tile row /
// column l % 16, group g = l / 16) holds k = 64 q + 32 t + 8 g + i:
//   A (activation row 16 mt + l % 16): 16 bytes;
//   B (weight row): f16 16 bytes; Q8_0 8 bytes of block 2q + t; Q4_0 8
//   bytes of block 2q + t (low nibbles for g < 2, high for g >= 2), with the
//   block's scale,
// dequantised with the correctly rounded RNE_f16((q - 8) d) / RNE_f16(q d)
// of every other path.  A wave issues only the stages of its own range and
// waits for a stage with the exact count of loads issued after it.  Rows
// past M and weight rows past N are read from offsets outside the buffers
// (zeros, no memory access).  The four K parts' fp32 accumulators meet in
// LDS and are added in a fixed order (part 0 + 1 + 2 + 3) before the
// epilogue.  C layout of a 16 x 16 tile: lane l holds column (weight row)
// l % 16 and activation rows 4 (l / 16) + r.
//
// K may also be split over p.splits workgroups per tile (block b: slice
// b % splits).  Each writes its fp32 tile to p.part and counts itself in on
// the tile's counter; the last to arrive adds the slices in slice order --
// the same bits whichever arrives last -- applies the epilogue and resets
// the counter to zero for the next launch, so no second kernel runs.  The
// exchange costs a few microseconds of memory round trips, so the plan
// splits only where that pays.  Every choice but the split leaves each
// output's summation order, and so its bits, unchanged.
// ---------------------------------------------------------------------------
constexpr int SK_LDS = 160 * 1024 - 1024;   // LDS the rings may take
constexpr int SK_MAX_SPLITS = 8;

template <int WT, int MT, int NT, int KP>
struct SkL {   // LDS bytes of one stage (one 64-k step) of one wave
    static constexpr int ROWS = 16 * NT;      // weight rows per workgroup
    static constexpr int X = MT * 16 * 128;   // activation rows, 128 bytes each
    static constexpr int WROW = WT == TLHIP_F16 ? 128 : (WT == TLHIP_Q8_0 ? 64 : 32);
    static constexpr int W = ROWS * WROW;
    static constexpr int S = WT == TLHIP_F16 ? 0 : 256;   // ROWS x 2 scales, one 4-byte load per lane
    static constexpr int STAGE = X + W + S;
    static constexpr int NX = X / 1024, NW = W / 1024, NS = S ? 1 : 0;
    static constexpr int C = NX + NW + NS;   // loads per stage
    // stages per wave: as many as the LDS holds (the deeper the ring, the
    // fewer memory round trips a wave's part takes), at most 6; a shape with
    // fewer than 2 is not launched (sk_plan)
    static constexpr int ST0 = SK_LDS / (KP * STAGE);
    static constexpr int ST = ST0 < 6 ? ST0 : 6;
    static constexpr bool OK = ST >= 2 && (ST - 1) * C < 64;
    static_assert(X % 1024 == 0 && W % 1024 == 0 && ROWS * 4 <= 256, "load shapes");
};

// wait until at most `ahead` stages of C loads each are outstanding
template <int C, int K>
__device__ __forceinline__ void sk_wait_stages(int ahead) {
    if constexpr (K == 0) {
        sk_wait_vm<0>();
    } else {
        if (ahead >= K) sk_wait_vm<K * C>();
        else sk_wait_stages<C, K - 1>(ahead);
    }
}

// Operand layout of one 64-k step (the k order inside an MFMA is free as
// long as both operands follow it).  Lane l = (column / row l % 16, group
// g = l / 16) holds at sub-step t the 8 elements k = 64 q + 8 c + i of its
// activation row, c = sk_piece(g, t), and of its weight row:
//   f16:  c = 4t + g, 16 bytes per sub-step;
//   Q8_0: c = 4(g/2) + 2(g%2) + t -- 16 bytes of block 2q + g/2 (elements
//         16(g%2) .. +15) give both sub-steps;
//   Q4_0: c = 4(g/2) + 2t + g%2 -- 8 bytes of block 2q + g/2 (bytes
//         8(g%2) .. +7) give both: low nibbles (elements 8(g%2) .. +7) at
//         t = 0, high nibbles (elements 16 + 8(g%2) .. +7) at t = 1;
// each block dequantised with its scale as RNE_f16((q - 8) d) / RNE_f16(q d).
template <int WT>
__device__ __forceinline__ int sk_piece(int g, int t) {
    if constexpr (WT == TLHIP_F16) return 4 * t + g;
    else if constexpr (WT == TLHIP_Q8_0) return 4 * (g >> 1) + 2 * (g & 1) + t;
    else return 4 * (g >> 1) + 2 * t + (g & 1);
}

template <int WT, int MT, int NT, int KP>
__global__ __launch_bounds__(64 * KP) void gemm_skinny_kernel(GemmParams p) {
    using L = SkL<WT, MT, NT, KP>;
    static_assert(L::OK, "ring");
    __shared__ __attribute__((aligned(1024))) uint8_t smem[KP * L::ST * L::STAGE];
    const int lane = threadIdx.x & 63;
    const int kp = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);   // wave-uniform
    const int nl = lane & 15, g = lane >> 4;
    const int z = (int)blockIdx.x % p.splits, mn = (int)blockIdx.x / p.splits;   // K slice, (M tile, N tile)
    const int m0 = mn % p.mtiles * 16 * MT, n0 = mn / p.mtiles * L::ROWS;
    const int nq = p.K >> 6;
    const int za = nq * z / p.splits, nz = nq * (z + 1) / p.splits - za;   // this workgroup's K slice (steps)
    const int qa = za + nz * kp / KP, nst = za + nz * (kp + 1) / KP - qa;
    uint8_t* const ring = smem + kp * L::ST * L::STAGE;
    const uint32_t ring_lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(gl_lds_t)ring);
    const uint32_t K = (uint32_t)p.K;

    constexpr uint32_t WSTEP = WT == TLHIP_F16 ? 128u : (WT == TLHIP_Q8_0 ? 64u : 32u);   // weight bytes per row and step
    const uint32_t wrow = WT == TLHIP_F16 ? 2u * K : (WT == TLHIP_Q8_0 ? K : K / 2u);
    const __amdgpu_buffer_rsrc_t rx = sk_rsrc(p.x, (uint32_t)p.M * K * 2u);
    const __amdgpu_buffer_rsrc_t rw = sk_rsrc(p.wq, (uint32_t)p.N * wrow);
    const __amdgpu_buffer_rsrc_t rd = sk_rsrc(WT == TLHIP_F16 ? (const void*)p.wq : (const void*)p.wd,
                                              WT == TLHIP_F16 ? 0u : (uint32_t)p.N * (K / 32u) * 2u);

    // source byte offsets (step 0) of this lane's 16 bytes in each load:
    // LDS piece P = 64 u + lane of the region, rows of 8 (x, f16 weights),
    // 4 (Q8_0) or 2 (Q4_0) pieces, XOR-swizzled by row
    uint32_t xsrc[L::NX], wsrc[L::NW], dsrc = SK_OOB;
#pragma unroll
    for (int u = 0; u < L::NX; u++) {
        const int P = 64 * u + lane, r = P >> 3, c = (P & 7) ^ (r & 7);
        xsrc[u] = m0 + r < p.M ? (uint32_t)(m0 + r) * K * 2u + 16u * c : SK_OOB;
    }
#pragma unroll
    for (int u = 0; u < L::NW; u++) {
        const int P = 64 * u + lane;
        int n, c;
        if (WT == TLHIP_F16) { n = P >> 3; c = (P & 7) ^ (n & 7); }
        else if (WT == TLHIP_Q8_0) { n = P >> 2; c = (P & 3) ^ ((n >> 1) & 3); }
        else { n = P >> 1; c = (P & 1) ^ ((n >> 2) & 1); }
        wsrc[u] = n0 + n < p.N ? (uint32_t)(n0 + n) * wrow + 16u * c : SK_OOB;
    }
    if (L::NS && lane < L::ROWS && n0 + lane < p.N) dsrc = (uint32_t)(n0 + lane) * (K / 32u) * 2u;

    // operand offsets inside a stage
    int xrd[MT][2], wrd[NT][2], drd[NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int r = 16 * mt + nl;
            xrd[mt][t] = r * 128 + 16 * (sk_piece<WT>(g, t) ^ (r & 7));
        }
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const int n = 16 * j + nl;
#pragma unroll
        for (int t = 0; t < 2; t++) {
            if (WT == TLHIP_F16) wrd[j][t] = L::X + n * 128 + 16 * ((4 * t + g) ^ (n & 7));
            else if (WT == TLHIP_Q8_0) wrd[j][t] = L::X + n * 64 + 16 * ((2 * (g >> 1) + (g & 1)) ^ ((n >> 1) & 3));
            else wrd[j][t] = L::X + n * 32 + 16 * ((g >> 1) ^ ((n >> 2) & 1)) + 8 * (g & 1);
        }
        drd[j] = L::X + L::W + 4 * n + 2 * (g >> 1);   // this lane's block's scale
    }

    // one stage's loads: step q into stage st
    auto issue = [&](int q, int st) {
        const uint32_t base = ring_lds + (uint32_t)(st * L::STAGE);
#pragma unroll
        for (int u = 0; u < L::NX; u++) sk_dma<16>(rx, base + 1024u * u, xsrc[u] + (uint32_t)q * 128u);
#pragma unroll
        for (int u = 0; u < L::NW; u++) sk_dma<16>(rw, base + L::X + 1024u * u, wsrc[u] + (uint32_t)q * WSTEP);
        if constexpr (L::NS > 0) sk_dma<4>(rd, base + L::X + L::W, dsrc + (uint32_t)q * 4u);
    };

    const bool rope = p.epi == EPI_QKV_ROPE;
    const bool use_b = p.epi == EPI_BIAS || p.epi == EPI_BIAS_RESID || p.epi == EPI_BIAS_GELU || (rope && p.bias);
    const bool use_r = p.epi == EPI_RESID || p.epi == EPI_BIAS_RESID;
    constexpr int NP = (NT * MT + KP - 1) / KP;   // pairs per wave
    uint32_t bv[NP], rv[NP][4];
    float rc[NP][4], rsn[NP][4];   // EPI_QKV_ROPE: the rotation of this lane's column pair at each row
#pragma unroll
    for (int i = 0; i < NP; i++) {   // epilogue operands, loaded while the K loop runs
        const int pr = kp + KP * i, j = pr % NT, mt = pr / NT;
        const int n = min(n0 + 16 * j + nl, p.N - 1);
        bv[i] = use_b && mt < MT ? (uint32_t)p.bias[n] : 0u;
        // EPI_QKV_ROPE: this column pair's place in its head (one division
        // per column, not per row)
        int re = -1;
        if (rope && mt < MT) {
            const int ne = n & ~1, D = p.head_dim;
            re = ne < p.nq ? ne % D : (ne < p.nq + p.nk ? (ne - p.nq) % D : -1);
            if (re >= p.rot) re = -1;
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = min(m0 + 16 * mt + 4 * g + r, p.M - 1);
            rv[i][r] = use_r && mt < MT ? (uint32_t)p.resid[(size_t)m * p.N + n] : 0u;
            rc[i][r] = 1.0f;
            rsn[i][r] = 0.0f;
            if (re >= 0) {
                const size_t ti = 2 * ((size_t)(p.pos0 + m) * (p.rot >> 1) + (re >> 1));
                rc[i][r] = p.rope_tab[ti];
                rsn[i][r] = p.rope_tab[ti + 1];
            }
        }
    }

    f4 acc[NT][MT];
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) acc[j][mt] = f4{0.0f, 0.0f, 0.0f, 0.0f};

    // the operands of one stage and its MFMAs
    auto compute = [&](int st) {
        const uint8_t* base = ring + st * L::STAGE;
        h8 a[MT][2], b[NT][2];
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int t = 0; t < 2; t++) a[mt][t] = *(const h8*)(base + xrd[mt][t]);
        if constexpr (WT == TLHIP_F16) {
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int t = 0; t < 2; t++) b[j][t] = *(const h8*)(base + wrd[j][t]);
        } else {
#pragma unroll
            for (int j = 0; j < NT; j++) {
                const h16 dh = *(const h16*)(base + drd[j]);
                const h2 dd = {dh, dh};
                uint32_t o[8];
                if constexpr (WT == TLHIP_Q8_0) {
                    const u4 w = *(const u4*)(base + wrd[j][0]);   // 16 elements: t = 0 bytes 0-7, t = 1 bytes 8-15
                    q8_pairs(w[0], dd, o[0], o[1]);
                    q8_pairs(w[1], dd, o[2], o[3]);
                    q8_pairs(w[2], dd, o[4], o[5]);
                    q8_pairs(w[3], dd, o[6], o[7]);
                } else {
                    const uint2 w = *(const uint2*)(base + wrd[j][0]);   // low nibbles t = 0, high nibbles t = 1
                    q4_pairs(w.x & 0x0F0F0F0Fu, dd, o[0], o[1]);
                    q4_pairs(w.y & 0x0F0F0F0Fu, dd, o[2], o[3]);
                    q4_pairs((w.x >> 4) & 0x0F0F0F0Fu, dd, o[4], o[5]);
                    q4_pairs((w.y >> 4) & 0x0F0F0F0Fu, dd, o[6], o[7]);
                }
                b[j][0] = __builtin_bit_cast(h8, u4{o[0], o[1], o[2], o[3]});
                b[j][1] = __builtin_bit_cast(h8, u4{o[4], o[5], o[6], o[7]});
            }
        }
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int j = 0; j < NT; j++)
                    acc[j][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[mt][t], b[j][t], acc[j][mt], 0, 0, 0);
    };

#pragma unroll
    for (int st = 0; st < L::ST; st++)
        if (st < nst) issue(qa + st, st);
    // steady state: every step refills its stage, so L::ST - 1 stages are
    // always in flight after it; then the last L::ST - 1 steps (fewer if the
    // part is short) drain the ring
    int st = 0, i = 0;
    for (; i + L::ST < nst; i++) {
        sk_wait_vm<(L::ST - 1) * L::C>();   // this step's stage has landed (loads complete in order)
        compute(st);
        // the stage's reads have returned before its refill is issued
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        issue(qa + i + L::ST, st);
        __builtin_amdgcn_sched_barrier(0);
        st = st + 1 == L::ST ? 0 : st + 1;
    }
    for (; i < nst; i++) {
        sk_wait_stages<L::C, L::ST - 1>(nst - 1 - i);
        compute(st);
        st = st + 1 == L::ST ? 0 : st + 1;
    }

    // every part's partial tiles to LDS (over the rings: every wave's loads
    // have landed); wave w then reduces (weight tile, M tile) pairs w,
    // w + KP, ... in part order and applies the epilogue
    __syncthreads();
    float (*red)[NT][MT * 4][64] = (float (*)[NT][MT * 4][64])smem;
    static_assert(sizeof(float) * KP * NT * MT * 4 * 64 <= sizeof(smem), "reduction fits the rings");
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int r = 0; r < 4; r++) red[kp][j][mt * 4 + r][lane] = acc[j][mt][r];
    __syncthreads();
    float vs[NP][4];
#pragma unroll
    for (int i = 0; i < NP; i++) {
        const int pr = kp + KP * i, j = pr % NT, mt = pr / NT;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            float v = 0.0f;
            if (mt < MT) {
                v = red[0][j][mt * 4 + r][lane];
#pragma unroll
                for (int u = 1; u < KP; u++) v += red[u][j][mt * 4 + r][lane];
            }
            vs[i][r] = v;
        }
    }
    if (p.splits > 1) {
        // This slice's tile to the partials; the last slice to arrive sums
        // them.  Partials and counter are written and read as device-scope
        // relaxed atomics, which go past this XCD's L2 to the memory every
        // XCD sees; waiting for the stores to complete before the count
        // orders them.  (Device-scope fences would instead write back and
        // invalidate the whole L2, which the other workgroups on the XCD
        // are streaming through.)
        __shared__ int sk_last;
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int pr = kp + KP * i, j = pr % NT, mt = pr / NT;
            const int ncol = n0 + 16 * j + nl;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + 16 * mt + 4 * g + r;
                if (mt < MT && m < p.M && ncol < p.N)
                    __hip_atomic_store(p.part + ((size_t)z * p.M + m) * p.N + ncol, vs[i][r], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0)
            sk_last = __hip_atomic_fetch_add(p.flags + mn, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                      (uint32_t)(p.splits - 1);
        __syncthreads();
        if (!sk_last) return;
        if (threadIdx.x == 0) __hip_atomic_store(p.flags + mn, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int pr = kp + KP * i, j = pr % NT, mt = pr / NT;
            const int ncol = min(n0 + 16 * j + nl, p.N - 1);
            float t[4][SK_MAX_SPLITS];   // every slice's value loaded before the in-order sum
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = min(m0 + 16 * mt + 4 * g + r, p.M - 1);
#pragma unroll
                for (int zz = 0; zz < SK_MAX_SPLITS; zz++)
                    t[r][zz] = mt < MT && zz < p.splits
                                   ? __hip_atomic_load(p.part + ((size_t)zz * p.M + m) * p.N + ncol, __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_AGENT)
                                   : 0.0f;
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float v = t[r][0];
#pragma unroll
                for (int zz = 1; zz < SK_MAX_SPLITS; zz++) v += t[r][zz];
                vs[i][r] = v;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < NP; i++) {
        const int pr = kp + KP * i, j = pr % NT, mt = pr / NT;
        if (mt >= MT) break;
        const int ncol = n0 + 16 * j + nl;
        // EPI_QKV_ROPE: destination of this column pair (per column, not per row)
        int sect = 0, hoff = 0, e = 0;
        if (rope) {
            const int D = p.head_dim;
            if (ncol < p.nq) {
                hoff = ncol / D * D;
                e = ncol - hoff;
            } else if (ncol < p.nq + p.nk) {
                sect = 1;
                hoff = (ncol - p.nq) / D * D;
                e = ncol - p.nq - hoff;
            } else {
                sect = 2;
                hoff = ncol - p.nq - p.nk;
            }
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float v = vs[i][r];
            const int m = m0 + 16 * mt + 4 * g + r;
            if (rope) {
                // the f16 projection (plus bias) of this column and of its
                // pair partner (column ^ 1, the neighbouring lane), rotated
                // and stored as the GEMV's fused epilogue does
                uint16_t x = f2h(v);
                if (p.bias) x = add_h(x, (uint16_t)bv[i]);
                const uint32_t xo = (uint32_t)__shfl_xor((int)x, 1, 64);
                if ((ncol & 1) == 0 && m < p.M && ncol + 1 < p.N) {
                    const int pos = p.pos0 + m;
                    if (sect == 2) {
                        p.vc[(size_t)pos * p.nk + hoff] = x;
                        p.vc[(size_t)pos * p.nk + hoff + 1] = (uint16_t)xo;
                        continue;
                    }
                    uint16_t* dst = sect ? p.kc + (size_t)pos * p.nk + hoff : p.q_out + (size_t)m * p.nq + hoff;
                    if (e < p.rot) {
                        const int half = p.rot >> 1, ip = e >> 1;
                        const float x0 = h2f(x), x1 = h2f((uint16_t)xo), c = rc[i][r], sn = rsn[i][r];
                        const float o0 = __fsub_rn(__fmul_rn(x0, c), __fmul_rn(x1, sn));
                        const float o1 = __fadd_rn(__fmul_rn(x0, sn), __fmul_rn(x1, c));
                        dst[p.layout ? ip : 2 * ip] = f2h(o0);
                        dst[p.layout ? ip + half : 2 * ip + 1] = f2h(o1);
                    } else {
                        dst[e] = x;
                        dst[e + 1] = (uint16_t)xo;
                    }
                }
            } else if (p.epi == EPI_SWIGLU_PAIR) {
                const float up = __shfl_down(v, 1, 64);
                if (m < p.M && ncol + 1 < p.N && (ncol & 1) == 0)
                    p.y[(size_t)m * p.ldy + ncol / 2] = swiglu_h(f2h(v), f2h(up));
            } else if (m < p.M && ncol < p.N) {
                p.y[(size_t)m * p.ldy + ncol] = epilogue_v(p.epi, v, (uint16_t)bv[i], (uint16_t)rv[i][r]);
            }
        }
    }
}

static bool gemm_skinny_ok(int M, int N, int K, int wt) {
    // byte offsets of the buffer loads are 32-bit, the padding offset
    // SK_OOB above every tensor
    const uint64_t wrow = wt == TLHIP_F16 ? 2ull * K : (wt == TLHIP_Q4_0 ? K / 2ull : (uint64_t)K);
    return M > 4 && M <= 64 && K % 64 == 0 && (wt == TLHIP_F16 || wt == TLHIP_Q8_0 || wt == TLHIP_Q4_0) &&
           (uint64_t)N * wrow < SK_OOB && 2ull * M * K < SK_OOB;
}

// The skinny GEMM's launch shape for (M, N, K, weight type): M tiles per
// workgroup (mt), 16-row weight tiles per workgroup (nt), waves (K parts)
// per workgroup (kp) and K slices.  A cost model fitted to the measured
// kernel (M = 46, cold weights): a workgroup takes its activation bytes in
// at about 50 GB/s (they are in L2: every weight tile reads them again) and
// its weight bytes at about 25 GB/s, plus 2.5 us of fixed time per round of
// workgroups (one workgroup per CU: the rings fill the LDS), plus 2.5 us
// for the exchange of a K split.  Where the weight tiles alone fill the
// device, splitting K with every row in one workgroup moves fewer bytes
// per CU (Q4_0 [2048 x 5632]: 13.8 -> 11.0 us; Q8_0: 15.7 -> 12.1 us).
// Eight waves (two per SIMD, so one's dequantisation overlaps the other's
// MFMAs and waits) wherever the LDS still holds a two-stage ring for each:
// four measured slower at every shape tried, so they are taken only when
// nothing else fits; a split leaves each wave at least two 64-k steps.
struct SkPlan {
    int mt = 1, nt = 2, kp = 4, mtiles = 1, splits = 1;
};
static int sk_stage_bytes(int wt, int mt, int nt) {
    const int wrow = wt == TLHIP_F16 ? 128 : (wt == TLHIP_Q8_0 ? 64 : 32);
    return mt * 16 * 128 + 16 * nt * wrow + (wt == TLHIP_F16 ? 0 : 256);
}
static SkPlan sk_plan(int M, int N, int K, int wt) {
    const double bpe = wt == TLHIP_F16 ? 2.0 : (wt == TLHIP_Q8_0 ? 34.0 / 32 : 18.0 / 32);
    const int mt16 = (M + 15) / 16;
    SkPlan best;
    for (int allow4 = 0; allow4 < 2; allow4++) {
        double best_us = 1e30;
        for (int nt : {2, 4})
            for (int mt = 1; mt <= mt16; mt++) {
                const int sb = sk_stage_bytes(wt, mt, nt);
                const int kp = SK_LDS / (8 * sb) >= 2 ? 8 : 4;
                if ((kp == 4 && !allow4) || SK_LDS / (kp * sb) < 2) continue;
                for (int sp = 1; sp <= SK_MAX_SPLITS; sp *= 2) {
                    const int mtiles = (mt16 + mt - 1) / mt, ntiles = (N + 16 * nt - 1) / (16 * nt);
                    if (sp > 1 && ((K / 64) / sp < 2 * kp || mtiles * ntiles > SK_MAX_TILES_SPLIT)) continue;
                    const long wgs = (long)mtiles * ntiles * sp;
                    const double rounds = (double)((wgs + 255) / 256);
                    const double bx = std::min(16 * mt, M) * 2.0 * K / sp, bw = 16 * nt * bpe * K / sp;
                    const double us = rounds * (bx / 50e3 + bw / 25e3 + 2.5) + (sp > 1 ? 2.5 : 0.0);
                    if (us < best_us - 1e-9) {
                        best_us = us;
                        best.mt = mt;
                        best.nt = nt;
                        best.kp = kp;
                        best.mtiles = mtiles;
                        best.splits = sp;
                    }
                }
            }
        if (best_us < 1e30) break;
    }
    return best;
}

// Skinny or tiled for M <= 64: tile_plan's estimate against a score of the skinny
// launch in the same us, whose constants minimise the time lost to wrong picks
// over 2980 measured shapes (M 5 - 64, N 64 - 32000, K 256 - 10240, the three
// weight types; weights in the caches and out of HBM; a decoder's shapes count
// more): 0.8 (f16), 0.6 (Q4_0) and 0.7 % (Q8_0) on average, 32 % at worst, and 1.9 /
// 0.3 / 0.2 % over a decoder's shapes.  As an estimate of the launch it is off by
// 7 - 16 % rms.  Skinny / tiled, us: f16 [256 x 2048] M = 16 6.4 / 7.9, [64 x 5632]
// M = 64 7.2 / 9.5, [16945 x 256] M = 39 16.9 / 6.8; Q4_0 [256 x 5632] M = 16 7.6 /
// 9.2, [2048 x 2048] M = 46 6.5 / 7.4, [11264 x 2048] M = 46 12.9 / 10.2; Q8_0 [2560
// x 2560] M = 46 8.0 / 8.7, [2560 x 10240] M = 64 31.5 / 16.2.
static bool skinny_wins(int M, int N, int K, int wt, const SkPlan& sk, const TilePlan& tile) {
    // us: per launch; per round of 256 workgroups, per KB of weights and of all
    // operands (busy CUs share the caches) and per 16 x 16 tile and step of a
    // wave; per split and 10^6 partials
    struct Fit {
        double launch, round, weight_kb, busy_kb, mfma, split, partials;
    };
    const Fit f = wt == TLHIP_F16    ? Fit{1.20, 2.48, 0.0091, 0.0120, 0.032, 2.31, 2.53}
                  : wt == TLHIP_Q8_0 ? Fit{0.04, 3.02, 0.0233, 0.0005, 0.224, 2.18, 2.49}
                                     : Fit{0.05, 3.27, 0.0440, 0.0022, 0.156, 2.39, 0.0};
    const double bpe = wt == TLHIP_F16 ? 2.0 : (wt == TLHIP_Q8_0 ? 34.0 / 32 : 18.0 / 32);
    const double wgs = (double)sk.mtiles * ((N + 16 * sk.nt - 1) / (16 * sk.nt)) * sk.splits, rounds = std::ceil(wgs / 256);
    const double kx = std::min(16 * sk.mt, M) * 2e-3 * K / sk.splits, kw = 16 * sk.nt * bpe * 1e-3 * K / sk.splits;
    double us = f.launch + rounds * (f.round + f.weight_kb * kw + f.busy_kb * std::min(wgs / 256, 1.0) * (kx + kw) +
                                     f.mfma * K / 64.0 / sk.splits / sk.kp * sk.mt * sk.nt);
    if (sk.splits > 1) us += f.split + f.partials * 1e-6 * sk.splits * M * N;
    return us < tile.us;
}

struct GemmPlan {
    int M = -1, N = 0, K = 0, wt = 0;
    bool skinny = false, staged = false;
    SkPlan sk;
    TilePlan tile;
    size_t ws_bytes = 0;   // split-K partials
};

// the tiled kernel's buffer ranges (128 rows of x) are below 2^31 bytes
static bool tile_ok(int K) { return K % 32 == 0 && K <= (1 << 22); }

// The plan of a shape, kept per thread for the shapes seen last (a model's
// prompt pass asks for the same few over and over; evaluating both models
// costs about a microsecond of host time).
static const GemmPlan& gemm_plan(int M, int N, int K, int wt) {
    static thread_local GemmPlan kept[64];
    GemmPlan& p = kept[((uint32_t)M * 2654435761u ^ (uint32_t)N * 40503u ^ (uint32_t)K * 9176u ^ (uint32_t)wt) >> 7 & 63];
    if (p.M == M && p.N == N && p.K == K && p.wt == wt) return p;
    p = GemmPlan();
    p.M = M;
    p.N = N;
    p.K = K;
    p.wt = wt;
    if (tile_ok(K)) p.tile = tile_plan(M, N, K, wt);
    if (gemm_skinny_ok(M, N, K, wt)) {
        p.sk = sk_plan(M, N, K, wt);
        p.skinny = !tile_ok(K) || skinny_wins(M, N, K, wt, p.sk, p.tile);
    }
    // Staged where its estimate is 5 % below the tiled kernel's, with more tiles
    // than CUs up to K = 1024 and with fewer up to 512 (f16, whose stages leave one
    // workgroup per CU, 512 and 384).  Past those bounds it is faster by 4 % at most
    // and slower by up to 45 %.  Over 380 drawn shapes that pick is 0.1 - 0.4 % off
    // the faster kernel on average, 9 % at worst.
    const bool many = (int64_t)((M + 127) / 128) * ((N + 127) / 128) > 256;
    p.staged = M > 64 && K % 64 == 0 && K <= (wt == TLHIP_F16 ? (many ? 512 : 384) : (many ? 1024 : 512)) &&
               staged_us(M, N, K, wt) < 0.95 * p.tile.us;
    p.ws_bytes = p.staged ? 0 : p.skinny ? (p.sk.splits > 1 ? (size_t)p.sk.splits * M * N * sizeof(float) : 0) : p.tile.ws_bytes;
    return p;
}

template <int WT, int MT, int NT, int KP>
static void launch_skinny_one(hipStream_t s, const GemmParams& p) {
    if constexpr (SkL<WT, MT, NT, KP>::OK) {
        const dim3 grid((unsigned)(p.mtiles * ((p.N + 16 * NT - 1) / (16 * NT)) * p.splits));
        hipLaunchKernelGGL((gemm_skinny_kernel<WT, MT, NT, KP>), grid, dim3(64 * KP), 0, s, p);
    }
}
template <int WT, int NT, int KP>
static void launch_skinny_mt(hipStream_t s, const GemmParams& p, int mt) {
    switch (mt) {
        case 1: launch_skinny_one<WT, 1, NT, KP>(s, p); break;
        case 2: launch_skinny_one<WT, 2, NT, KP>(s, p); break;
        case 3: launch_skinny_one<WT, 3, NT, KP>(s, p); break;
        default: launch_skinny_one<WT, 4, NT, KP>(s, p); break;
    }
}
template <int WT>
static void launch_skinny(hipStream_t s, const GemmParams& p, const SkPlan& pl) {
    if (pl.nt == 4) {
        if (pl.kp == 8) launch_skinny_mt<WT, 4, 8>(s, p, pl.mt);
        else launch_skinny_mt<WT, 4, 4>(s, p, pl.mt);
    } else {
        if (pl.kp == 8) launch_skinny_mt<WT, 2, 8>(s, p, pl.mt);
        else launch_skinny_mt<WT, 2, 4>(s, p, pl.mt);
    }
}

// The bounds GEMM_SPLIT_PARTIALS_MAX states (the fixed workspace of the
// no-allocation entry point is sized by it); tile_plan keeps to it itself.
static_assert((size_t)SK_MAX_SPLITS * 64 * (SK_MAX_TILES_SPLIT * 16 * 4) * sizeof(float) <= GEMM_SPLIT_PARTIALS_MAX,
              "skinny split (64 rows, N <= SK_MAX_TILES_SPLIT tiles of 16 x 4 weight rows)");

size_t gemm_ws_bytes(int M, int N, int K, int wt) {
    if (wt < 0) {
        size_t b = 0;
        for (int t : {(int)TLHIP_F16, (int)TLHIP_Q8_0, (int)TLHIP_Q4_0}) b = std::max(b, gemm_ws_bytes(M, N, K, t));
        return b;
    }
    return gemm_plan(M, N, K, wt).ws_bytes;
}

GemmRoute gemm_route(int M, int N, int K, int wt) {
    GemmRoute r;
    if (K % 32 != 0 || K == 0) {
        r.kernel = TLHIP_LINEAR_PLAIN;
        return r;
    }
    const GemmPlan& p = gemm_plan(M, N, K, wt);
    r.rope = gemm_rope_ok(M, N, K, wt);
    r.ws_bytes = p.ws_bytes;
    if (p.skinny) {
        r.kernel = TLHIP_LINEAR_SKINNY;
        r.tile_m = 16 * p.sk.mt;
        r.tile_n = 16 * p.sk.nt;
        r.splits = p.sk.splits;
    } else if (p.staged) {
        r.kernel = TLHIP_LINEAR_STAGED;
        r.tile_m = r.tile_n = 128;
    } else if (tile_ok(K)) {
        r.kernel = TLHIP_LINEAR_TILED;
        tile_dims(p.tile.shape, &r.tile_m, &r.tile_n);
        r.splits = p.tile.splits;
    } else {
        r.kernel = TLHIP_LINEAR_BASIC;
        r.tile_m = GBM;
        r.tile_n = GBN;
    }
    return r;
}

bool gemm_rope_ok(int M, int N, int K, int wt) {
    return (wt == TLHIP_F16 || wt == TLHIP_Q8_0 || wt == TLHIP_Q4_0) && tile_ok(K);
}

// Naive fp32-accumulate GEMM for f16 weights whose K is not a multiple of 32
// (reference unit-test shapes such as [50, 122]), and for K = 0 of any type.
__global__ void gemm_naive_kernel(GemmParams p) {
    int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)p.M * p.N) return;
    int m = (int)(idx / p.N), n = (int)(idx % p.N);
    const uint16_t* w = (const uint16_t*)p.wq + (size_t)n * p.K;
    const uint16_t* x = p.x + (size_t)m * p.K;
    float acc = 0.0f;
    for (int k = 0; k < p.K; k++) acc += h2f(x[k]) * h2f(w[k]);
    p.y[(size_t)m * p.ldy + n] = epilogue_h(p.epi, acc, p.bias, p.resid, (size_t)m * p.N + n, n);
}

tlhip_status launch_gemm(hipStream_t s, tlhip_dtype wt, const GemvArgs& a, int epi) {
    GemmParams p;
    p.x = a.x;
    p.wq = (const uint8_t*)a.wq;
    p.wd = a.wd;
    p.bias = a.bias;
    p.resid = a.resid;
    p.y = a.y;
    p.M = a.M;
    p.N = a.N;
    p.K = a.K;
    p.ldy = a.ldy ? a.ldy : (epi == EPI_SWIGLU_PAIR ? a.N / 2 : a.N);
    p.epi = epi;
    if (a.pro != PRO_NONE)
        return fail(TLHIP_ERR_INVALID_OPERATION, "gemm: the fused normalisation prologue is GEMV-only");
    if (epi == EPI_QKV_ROPE) {
        if (!gemm_rope_ok(p.M, p.N, p.K, wt) || a.d_pos || !a.rope_tab || !a.q_out || !a.kc || !a.vc ||
            a.head_dim <= 0 || a.head_dim % 2 || a.rot % 2 || a.rot > a.head_dim || a.nq % a.head_dim ||
            a.nk % a.head_dim || a.nq + 2 * a.nk != p.N)
            return fail(TLHIP_ERR_INVALID_OPERATION, "gemm: the RoPE epilogue needs K %% 32 == 0 and a q/k/v layout");
        p.nq = a.nq;
        p.nk = a.nk;
        p.head_dim = a.head_dim;
        p.rot = a.rot;
        p.layout = a.layout;
        p.pos0 = a.pos0;
        p.rope_tab = a.rope_tab;
        p.q_out = a.q_out;
        p.kc = a.kc;
        p.vc = a.vc;
    }
    if (wt != TLHIP_F16 && wt != TLHIP_Q4_0 && wt != TLHIP_Q8_0)
        return fail(TLHIP_ERR_DTYPE, "gemm: weight dtype %d takes the dequantised f16 path", (int)wt);
    if (p.M <= 0 || p.N <= 0) return TLHIP_OK;
    // K = 0 (an empty sum: zeros, or the bias) too: the tiled kernel always
    // computes one step of K
    if (p.K % 32 != 0 || p.K == 0) {
        if ((wt != TLHIP_F16 && p.K != 0) || epi == EPI_SWIGLU_PAIR)
            return fail(TLHIP_ERR_INVALID_OPERATION, "gemm: K=%d not a positive multiple of 32", p.K);
        int64_t n = (int64_t)p.M * p.N;
        hipLaunchKernelGGL(gemm_naive_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p);
        return TLHIP_OK;
    }
    const GemmPlan& plan = gemm_plan(p.M, p.N, p.K, wt);
    if (plan.skinny) {
        // K split over workgroups only with a workspace for the partials and
        // the per-tile counters
        const SkPlan& pl = plan.sk;
        p.mtiles = pl.mtiles;
        if (pl.splits > 1 && a.ws && a.tile_flags && (size_t)pl.splits * p.M * p.N * sizeof(float) <= a.ws_bytes) {
            p.splits = pl.splits;
            p.part = a.ws;
            p.flags = a.tile_flags;
        }
        if (wt == TLHIP_Q4_0) launch_skinny<TLHIP_Q4_0>(s, p, pl);
        else if (wt == TLHIP_Q8_0) launch_skinny<TLHIP_Q8_0>(s, p, pl);
        else launch_skinny<TLHIP_F16>(s, p, pl);
        return TLHIP_OK;
    }
    if (plan.staged && epi != EPI_QKV_ROPE) return launch_gemm_staged(s, wt, a, epi, p.ldy);
    if (tile_ok(p.K)) return launch_gemm_tile(s, wt, a, epi, p.ldy, plan.tile);
    dim3 grid((unsigned)((p.N + GBN - 1) / GBN), (unsigned)((p.M + GBM - 1) / GBM));
    if (wt == TLHIP_Q4_0) hipLaunchKernelGGL(gemm_kernel<TLHIP_Q4_0>, grid, dim3(256), 0, s, p);
    else if (wt == TLHIP_Q8_0) hipLaunchKernelGGL(gemm_kernel<TLHIP_Q8_0>, grid, dim3(256), 0, s, p);
    else hipLaunchKernelGGL(gemm_kernel<TLHIP_F16>, grid, dim3(256), 0, s, p);
    return TLHIP_OK;
}

// ---------------------------------------------------------------------------
// linear() on f32 tensors (the TensorF32 arm, builtin_math.rs:121-175:
// x.matmul_transposed_b(w), then result.add(bias)).  Every output is the
// reference kernel's sum (matmul_transposed_b_tiled_32x32_f32,
// unified.metal:4409-4461): k in order from +0, one fused multiply-add per
// term (the contraction Metal's default fast math makes of `sum += a * b`),
// the row padded with zero terms to a multiple of 32 as its tiles are; the
// bias is a separate f32 add.  A workgroup of 256 threads computes a 64 x 64
// tile, 4 x 4 outputs per thread, from 64 x 32 slices of x and w staged
// k-major in LDS.  Not on the decode path (the LLM programs are f16): plain
// VALU arithmetic, no MFMA (v_mfma_f32_*_xf32 would change the sums' order).
// ---------------------------------------------------------------------------
constexpr int LF_BM = 64, LF_BN = 64, LF_BK = 32;

__global__ __launch_bounds__(256) void linear_f32_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                         const float* __restrict__ bias, float* __restrict__ y, int M,
                                                         int N, int K) {
    __shared__ float as[LF_BK][LF_BM + 4];
    __shared__ float bs[LF_BK][LF_BN + 4];
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    const int m0 = blockIdx.y * LF_BM, n0 = blockIdx.x * LF_BN;
    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = 0.0f;
    const int kp = (K + LF_BK - 1) / LF_BK * LF_BK;   // zero terms up to a multiple of 32
    for (int k0 = 0; k0 < kp; k0 += LF_BK) {
#pragma unroll
        for (int i = 0; i < 8; i++) {   // 64 rows x 32 k of each operand, 8 per thread
            const int idx = tid + 256 * i, r = idx >> 5, c = idx & 31;
            const int k = k0 + c;
            as[c][r] = (m0 + r < M && k < K) ? x[(size_t)(m0 + r) * K + k] : 0.0f;
            bs[c][r] = (n0 + r < N && k < K) ? w[(size_t)(n0 + r) * K + k] : 0.0f;
        }
        __syncthreads();
#pragma unroll 8
        for (int kk = 0; kk < LF_BK; kk++) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; i++) a[i] = as[kk][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; j++) b[j] = bs[kk][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] = __builtin_fmaf(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int m = m0 + ty * 4 + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int n = n0 + tx * 4 + j;
            if (n < N) y[(size_t)m * N + n] = bias ? acc[i][j] + bias[n] : acc[i][j];
        }
    }
}

tlhip_status launch_linear_f32(hipStream_t s, const float* x, const float* w, const float* bias, float* y, int M, int N,
                               int K) {
    if (M <= 0 || N <= 0) return TLHIP_OK;
    const dim3 grid((unsigned)((N + LF_BN - 1) / LF_BN), (unsigned)((M + LF_BM - 1) / LF_BM));
    if (grid.y > 65535) return fail(TLHIP_ERR_INVALID_DIMENSION, "linear f32: %d rows", M);
    hipLaunchKernelGGL(linear_f32_kernel, grid, dim3(256), 0, s, x, w, bias, y, M, N, K);
    return TLHIP_OK;
}

}  // namespace tlhip
