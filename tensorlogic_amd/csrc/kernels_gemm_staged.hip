// kernels_gemm_staged.hip -- the staged MFMA dequant-GEMM: many tiles of a
// short K (more than 64 rows, K % 64 == 0), gfx950.
//
// y[M, N] = x[M, K] . W[N, K]^T in 128 x 128 x 64 tiles, 512 threads = 8 waves in
// a 2 (M) x 4 (N) grid, each wave 64 x 32 of C in 32 x 32
// v_mfma_f32_32x32x16_f16 tiles.  NS LDS stages are filled by direct
// global->LDS loads (no VGPR staging), so NS - 1 K steps are in flight while one
// is computed.  The LDS keeps the payload as stored (Q4_0 nibbles, Q8_0 int8 or
// f16) plus the block scales; each wave dequantises its B operand into registers
// right before its MFMAs, with the RNE_f16((q-8)*d) / RNE_f16(q*d) of every
// other path, and stores its accumulators itself.
//
// Beside gemm_tile_kernel, which is up to twice as fast on long rows, it has
// little to do before the first MFMA and after the last, and three packed
// stages are 60 - 74 KB: two workgroups share a CU, so that one's first loads and
// stores run under the other's MFMAs.  With a K of a few steps that decides:
// staged / tiled, us: Q4_0 [23565 x 256] M = 2000 69 / 98, [11632 x 448] M = 1720 42 /
// 56, Q8_0 [14250 x 320] M = 916 28 / 39, [17175 x 512] M = 916 42 / 55, f16 [32000 x
// 256] M = 2048 131 / 180; and with a longer one, Q8_0 [9583 x 2048] M = 1024 85 / 74.
//
// K order inside a 64-wide step: MFMA lane half h (lane / 32) carries the
// elements 32h + 8t .. 32h + 8t + 7 at sub-step t = 0..3 (quant block h of
// the step) for A and B alike, so every k is summed once in fp32.
//
// LDS rows are XOR-swizzled in 16-byte chunks so that the 32 rows a wave
// reads at one chunk index fall in distinct banks: A / f16 B rows (128 B)
// chunk c -> c ^ ((r >> 1) & 7); Q8_0 rows (64 B) c -> c ^ ((r >> 2) & 3); Q4_0 rows
// (32 B) c -> c ^ ((r >> 3) & 1).  A direct load writes lane l's 16 (4) bytes
// at LDS base + 16 l (4 l); each lane fetches the global chunk that the
// swizzle puts in its slot.
//
// Workgroups are dispatched round-robin over the 8 XCDs (workgroup id mod
// 8); the id -> tile map gives each XCD a contiguous run of tiles with the
// M tiles of one N tile adjacent, so the tiles that share weight rows run on
// one XCD and read them through one L2.
#include "gemm_tile.hpp"

namespace tlhip {

template <int WT>
struct GlRow {   // LDS bytes of one weight row per 64-wide K step
    static constexpr int B = WT == TLHIP_F16 ? 128 : (WT == TLHIP_Q8_0 ? 64 : 32);
};

// direct loads of one LDS region of R bytes by 512 threads: 16-byte loads
// when R is a multiple of 8 KB, else 4-byte loads (R multiple of 2 KB)
template <int R>
struct GlDma {
    static constexpr int SZ = R % 8192 == 0 ? 16 : 4;
    static constexpr int N = R / (512 * SZ);
    static_assert(R % 2048 == 0, "region");
};

template <int WT, int BM, int BN, int NS>
struct Gl {
    static constexpr int A_BYTES = BM * 128;
    static constexpr int B_BYTES = BN * GlRow<WT>::B;
    static constexpr int S_BYTES = WT == TLHIP_F16 ? 0 : BN * 4;
    static constexpr int STAGE = A_BYTES + B_BYTES + S_BYTES;
    static constexpr int VMC = GlDma<A_BYTES>::N + GlDma<B_BYTES>::N + (S_BYTES ? 1 : 0);
    static_assert((NS - 2) * VMC < 64, "vmcnt range");
    static_assert(BN / 8 <= 64, "scale rows per wave");
};

template <int N>
__device__ __forceinline__ void gl_wait_vm() {   // s_waitcnt vmcnt(N), gfx9 encoding
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x70 | 0xF00);
}
template <int VMC, int K>
__device__ __forceinline__ void gl_wait_stage(int ahead) {   // wait until <= ahead stages outstanding
    if constexpr (K == 0) {
        gl_wait_vm<0>();
    } else {
        if (ahead >= K) gl_wait_vm<K * VMC>();
        else gl_wait_stage<VMC, K - 1>(ahead);
    }
}

template <int SZ>
__device__ __forceinline__ void gl_dma(const void* g, uint8_t* lds) {
    if constexpr (SZ == 16) __builtin_amdgcn_global_load_lds(g, (gl_lds_t)lds, 16, 0, 0);
    else __builtin_amdgcn_global_load_lds(g, (gl_lds_t)lds, 4, 0, 0);
}

__device__ __forceinline__ void gemm_store_one(const TileParams& p, int m, int n, float v) {
    if (p.epi == EPI_SWIGLU_PAIR) {
        const float up = __shfl_down(v, 1, 64);
        if (m < p.M && n + 1 < p.N && (n & 1) == 0) p.y[(size_t)m * p.ldy + n / 2] = swiglu_h(f2h(v), f2h(up));
    } else if (m < p.M && n < p.N) {
        p.y[(size_t)m * p.ldy + n] = epilogue_h(p.epi, v, p.bias, p.resid, (size_t)m * p.N + n, n);
    }
}

template <int WT, int BM, int BN, int NS>
__global__ __launch_bounds__(512) void gemm_staged_kernel(TileParams p) {
    using L = Gl<WT, BM, BN, NS>;
    constexpr int TM = BM / 64, TN = BN / 128;   // 32x32 tiles per wave
    constexpr int WTN = BN / 4;                   // wave tile width
    static_assert(TN >= 1 && BN % 128 == 0, "BN");
    __shared__ __attribute__((aligned(1024))) uint8_t smem[NS * L::STAGE];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 2, wn = wave & 3, hh = lane >> 5, l32 = lane & 31;
    const int T = p.mT * p.nT, xcd = blockIdx.x & 7;
    const int q = xcd * (T >> 3) + min(xcd, T & 7) + ((int)blockIdx.x >> 3);
    const int m0 = (q % p.mT) * BM, n0 = (q / p.mT) * BN;
    const int nk = p.K / 64, nbr = p.K >> 5;

    using DA = GlDma<L::A_BYTES>;
    using DB = GlDma<L::B_BYTES>;
    const uint8_t* a_src[DA::N];
#pragma unroll
    for (int u = 0; u < DA::N; u++) {
        const int P = (u * 8 + wave) * 64 * DA::SZ + lane * DA::SZ;
        const int r = P >> 7, c = ((P >> 4) & 7) ^ ((r >> 1) & 7);
        const int m = min(m0 + r, p.M - 1);
        a_src[u] = (const uint8_t*)(p.x + (size_t)m * p.K + 8 * c) + (P & 15);
    }
    const uint8_t* b_src[DB::N];
#pragma unroll
    for (int u = 0; u < DB::N; u++) {
        constexpr int RB = GlRow<WT>::B;
        const int P = (u * 8 + wave) * 64 * DB::SZ + lane * DB::SZ;
        const int r = P / RB, cp = (P % RB) >> 4, byte = P & 15;
        const int n = min(n0 + r, p.N - 1);
        if (WT == TLHIP_F16) {
            b_src[u] = p.wq + ((size_t)n * p.K + 8 * (cp ^ ((r >> 1) & 7))) * 2 + byte;
        } else if (WT == TLHIP_Q8_0) {
            b_src[u] = p.wq + (size_t)n * p.K + 16 * (cp ^ ((r >> 2) & 3)) + byte;
        } else {
            b_src[u] = p.wq + (size_t)n * (p.K / 2) + 16 * (cp ^ ((r >> 3) & 1)) + byte;
        }
    }
    // scales: wave w, lanes < BN/8 -> row w*BN/8 + lane, both blocks of the step (4 bytes)
    constexpr int SR = BN / 8;
    const bool s_lane = lane < SR;
    const uint8_t* s_src = nullptr;
    if (L::S_BYTES) {
        const int n = min(n0 + wave * SR + (s_lane ? lane : 0), p.N - 1);
        s_src = (const uint8_t*)(p.wd + (size_t)n * nbr);
    }
    constexpr int B_STEP = GlRow<WT>::B == 128 ? 128 : GlRow<WT>::B;

    auto issue = [&](int step, int s) {
        uint8_t* st = smem + s * L::STAGE;
#pragma unroll
        for (int u = 0; u < DA::N; u++) gl_dma<DA::SZ>(a_src[u] + (size_t)step * 128, st + (u * 8 + wave) * 64 * DA::SZ);
#pragma unroll
        for (int u = 0; u < DB::N; u++)
            gl_dma<DB::SZ>(b_src[u] + (size_t)step * B_STEP, st + L::A_BYTES + (u * 8 + wave) * 64 * DB::SZ);
        if (L::S_BYTES && s_lane) gl_dma<4>(s_src + (size_t)step * 4, st + L::A_BYTES + L::B_BYTES + wave * SR * 4);
    };

    f16v acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = f16v{0};

#pragma unroll
    for (int s = 0; s < NS - 1; s++)
        if (s < nk) issue(s, s);

    // per-lane LDS offsets inside a stage (constant over the K loop)
    int a_off[TM][4], b_off[TN][4];
#pragma unroll
    for (int ii = 0; ii < TM; ii++) {
        const int m = wm * (BM / 2) + 32 * ii + l32;
#pragma unroll
        for (int t = 0; t < 4; t++) a_off[ii][t] = 128 * m + 16 * ((4 * hh + t) ^ ((m >> 1) & 7));
    }
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int n = wn * WTN + 32 * j + l32;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            if (WT == TLHIP_F16) b_off[j][t] = L::A_BYTES + 128 * n + 16 * ((4 * hh + t) ^ ((n >> 1) & 7));
            else if (WT == TLHIP_Q8_0) b_off[j][t] = t < 2 ? L::A_BYTES + 64 * n + 16 * ((2 * hh + t) ^ ((n >> 2) & 3))
                                                           : L::A_BYTES + L::B_BYTES + 4 * n + 2 * hh;
            else b_off[j][t] = t == 0 ? L::A_BYTES + 32 * n + 16 * (hh ^ ((n >> 3) & 1))
                                      : L::A_BYTES + L::B_BYTES + 4 * n + 2 * hh;
        }
    }

    for (int i = 0; i < nk; i++) {
        gl_wait_stage<L::VMC, NS - 2>(min(nk - 1 - i, NS - 2));
        lds_barrier();   // stage i landed for every wave; stage i-1 fully read
        if (i + NS - 1 < nk) issue(i + NS - 1, (i + NS - 1) % NS);

        const uint8_t* st = smem + (i % NS) * L::STAGE;
        // all LDS reads of the step first, then dequantise, then the MFMAs
        h8 aop[TM][4];
#pragma unroll
        for (int ii = 0; ii < TM; ii++)
#pragma unroll
            for (int t = 0; t < 4; t++) aop[ii][t] = *(const h8*)(st + a_off[ii][t]);
        h8 bop[TN][4];
        if (WT == TLHIP_F16) {
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int t = 0; t < 4; t++) bop[j][t] = *(const h8*)(st + b_off[j][t]);
        } else if (WT == TLHIP_Q8_0) {
            u4 raw[TN][2];
            h16 dh[TN];
#pragma unroll
            for (int j = 0; j < TN; j++) {
                raw[j][0] = *(const u4*)(st + b_off[j][0]);
                raw[j][1] = *(const u4*)(st + b_off[j][1]);
                dh[j] = *(const h16*)(st + b_off[j][2]);
            }
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const h2 dd = {dh[j], dh[j]};
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    uint32_t o0, o1, o2, o3;
                    q8_pairs(raw[j][t >> 1][2 * (t & 1)], dd, o0, o1);
                    q8_pairs(raw[j][t >> 1][2 * (t & 1) + 1], dd, o2, o3);
                    bop[j][t] = __builtin_bit_cast(h8, u4{o0, o1, o2, o3});
                }
            }
        } else {
            u4 raw[TN];
            h16 dh[TN];
#pragma unroll
            for (int j = 0; j < TN; j++) {
                raw[j] = *(const u4*)(st + b_off[j][0]);
                dh[j] = *(const h16*)(st + b_off[j][1]);
            }
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const h2 dd = {dh[j], dh[j]};
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    // t = 0/1: low nibbles of bytes 0-7 / 8-15; t = 2/3: high nibbles
                    const uint32_t w0 = raw[j][2 * (t & 1)], w1 = raw[j][2 * (t & 1) + 1];
                    const uint32_t n0w = t < 2 ? (w0 & 0x0F0F0F0Fu) : ((w0 >> 4) & 0x0F0F0F0Fu);
                    const uint32_t n1w = t < 2 ? (w1 & 0x0F0F0F0Fu) : ((w1 >> 4) & 0x0F0F0F0Fu);
                    uint32_t o0, o1, o2, o3;
                    q4_pairs(n0w, dd, o0, o1);
                    q4_pairs(n1w, dd, o2, o3);
                    bop[j][t] = __builtin_bit_cast(h8, u4{o0, o1, o2, o3});
                }
            }
        }
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int ii = 0; ii < TM; ii++)
#pragma unroll
                for (int j = 0; j < TN; j++)
                    acc[ii][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(aop[ii][t], bop[j][t], acc[ii][j], 0, 0, 0);
    }

    // C layout: col = lane%32 (weight row n), row = 8*(r/4) + 4*(lane/32) + r%4 (activation row m)
#pragma unroll
    for (int ii = 0; ii < TM; ii++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int n = n0 + wn * WTN + 32 * j + l32;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = m0 + wm * (BM / 2) + 32 * ii + 8 * (r >> 2) + 4 * hh + (r & 3);
                gemm_store_one(p, m, n, acc[ii][j][r]);
            }
        }
}

// The cost of a launch in us (tile_plan's is the other side), fitted to 1190
// launches of more than 64 rows, the mean of weights in the caches and out of HBM,
// most weight on shapes where the two kernels are close; 5 - 6 % rms.  Up to 256
// tiles one round, longer with more CUs in use; beyond, tiles in turn on CUs that
// hold two workgroups each (f16: one).
double staged_us(int M, int N, int K, int wt) {
    struct Cost {
        double launch, step, busy_step, more, tiles_step;
    };
    const Cost c = wt == TLHIP_F16 ? Cost{7.19, 0.397, 0.279, 5.28, 0.868}
                                   : (wt == TLHIP_Q8_0 ? Cost{7.27, 0.529, 0.227, 1.98, 0.788} : Cost{7.28, 0.561, 0.186, 0.93, 0.828});
    const double tiles = (double)((M + 127) / 128) * ((N + 127) / 128), steps = K / 64;
    if (tiles <= 256) return c.launch + steps * (c.step + c.busy_step * (tiles > 64 ? (tiles - 64) / 192 : 0.0));
    return c.launch + c.more + tiles / 256 * steps * c.tiles_step;
}

// Three stages once the tiles are more than the CUs, so that two workgroups
// share a CU; four before.
template <int WT>
static void launch_staged(hipStream_t s, TileParams& p) {
    p.mT = (p.M + 127) / 128;
    p.nT = (p.N + 127) / 128;
    const unsigned grid = (unsigned)(p.mT * p.nT);
    if (grid > 256) hipLaunchKernelGGL((gemm_staged_kernel<WT, 128, 128, 3>), dim3(grid), dim3(512), 0, s, p);
    else hipLaunchKernelGGL((gemm_staged_kernel<WT, 128, 128, 4>), dim3(grid), dim3(512), 0, s, p);
}

tlhip_status launch_gemm_staged(hipStream_t s, int wt, const GemvArgs& a, int epi, int ldy) {
    TileParams p = {};
    p.x = a.x;
    p.wq = (const uint8_t*)a.wq;
    p.wd = a.wd;
    p.bias = a.bias;
    p.resid = a.resid;
    p.y = a.y;
    p.M = a.M;
    p.N = a.N;
    p.K = a.K;
    p.ldy = ldy;
    p.epi = epi;
    if (wt == TLHIP_Q4_0) launch_staged<TLHIP_Q4_0>(s, p);
    else if (wt == TLHIP_Q8_0) launch_staged<TLHIP_Q8_0>(s, p);
    else launch_staged<TLHIP_F16>(s, p);
    return TLHIP_OK;
}

}  // namespace tlhip
