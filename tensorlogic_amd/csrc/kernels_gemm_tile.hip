// kernels_gemm_tile.hip -- launches of the tiled MFMA dequant-GEMM
// (gemm_tile.hpp): tile shape and K split by a cost model, and the sum of the
// K slices.
#include <algorithm>

#include "gemm_tile.hpp"

namespace tlhip {

// The K slices' partials summed in slice order, then the epilogue: 8
// consecutive outputs per thread.  Bound by the partials' bytes (M = 512, N =
// 2560, 3 slices: 15.7 MB, 5.5 us).
__global__ __launch_bounds__(256) void tile_reduce_kernel(TileParams p) {
    const int per_row = (p.N + 7) / 8;
    const int64_t it = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (it >= (int64_t)p.M * per_row) return;
    const int m = (int)(it / per_row), n = (int)(it % per_row) * 8;
    const size_t row = (p.N + 7) & ~7, total = (size_t)p.M * row;
    const float* s = p.part + m * row + n;
    f4 a = *(const f4*)s, b = *(const f4*)(s + 4);
    for (int z = 1; z < p.splits; z++) {
        a += *(const f4*)(s + z * total);
        b += *(const f4*)(s + z * total + 4);
    }
    float v[8];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        v[e] = a[e];
        v[4 + e] = b[e];
    }
    tile_store8(p, m, n, v);
}

namespace {

// Tile shapes.  A wave of 128 x 64 dequantises each weight once; the smaller
// ones fill more CUs.  (Measured and not built: 128 x 128 in 64 x 64 waves,
// within 4 % of the first for f16 weights and behind for packed ones; 32 x 64
// for M <= 32, never more than 3 % ahead of 64 x 32.)
struct TileShape {
    int bm, bn, bk;
};
constexpr TileShape SHAPES[5] = {{128, 128, 128}, {128, 64, 128}, {64, 128, 128}, {64, 64, 256}, {64, 32, 256}};

// The cost of a plan in us: the launch, and per round of 256 workgroups (one
// per CU: the ring fills the LDS) what does not depend on K (first loads,
// epilogue) and the steps, both longer by up to the `busy` terms as the CUs in
// use go from 64 to 256; rounds after the first cost `later` more.  A split
// adds its second launch, the partials' traffic and, per slice, the two loads
// that a thread of the sum waits for: without that term [40 x 5632] @ [2048 x
// 5632]^T took 64 x 64 tiles in 8 slices (Q8_0, 11.4 us in the caches) and not
// 64 x 32 in 4 (9.6 us), at as many workgroups.  `weights` is their one pass from
// HBM, `acts` the activations once per column of tiles, which narrow tiles pay
// more often: without it f16 [100 x 2560] @ [7680 x 2560]^T took 128 x 64 tiles
// (15.6 us in the caches, 21.7 out of HBM) and not 64 x 64 (14.3, 17.7).  All
// three per 10^6 elements.
struct TileCost {
    double launch, split, slice, partials, weights, acts;
    struct {
        double fix, step, busy_step, busy_fix, later;
    } shape[5];
};
constexpr TileCost COST_F16 = {2.63, 2.08, 0.257, 0.484, 0.1024, 0.0467,
                               {{4.47, 0.921, 0.0, 1.61, 0.0}, {2.74, 0.340, 0.070, 0.0, 1.27}, {2.44, 0.375, 0.237, 0.44, 0.67},
                                {1.77, 0.669, 0.118, 0.0, 1.19}, {1.89, 0.317, 0.0, 0.0, 1.00}}};
constexpr TileCost COST_Q8 = {2.09, 2.09, 0.277, 0.650, 0.0274, 0.0372,
                              {{6.20, 0.562, 0.242, 0.78, 0.03}, {3.20, 0.468, 0.0, 0.83, 0.27}, {3.12, 0.448, 0.098, 0.62, 0.53},
                               {2.92, 0.495, 0.006, 0.0, 0.53}, {2.57, 0.305, 0.0, 0.0, 0.0}}};
constexpr TileCost COST_Q4 = {2.29, 2.23, 0.251, 0.735, 0.0125, 0.0308,
                              {{5.82, 0.539, 0.267, 0.51, 0.0}, {3.44, 0.413, 0.038, 0.53, 0.57}, {3.18, 0.389, 0.091, 0.54, 0.71},
                               {2.75, 0.442, 0.011, 0.0, 0.63}, {2.58, 0.283, 0.0, 0.0, 0.18}}};

}  // namespace

// Tile shape and K slices for (M, N, K, weight type): the cheapest plan.  The
// costs are fitted to every shape and split of 2414 problems (M 5 - 2048, N 64 -
// 32000, K 256 - 10240, 714 of them model shapes), the mean of weights in the
// caches and out of HBM.  The pick is 0.2 % slower than the best measured plan on
// average, 14 % at worst; the estimate is off by 4 (packed) to 5 % rms.
TilePlan tile_plan(int M, int N, int K, int wt) {
    const TileCost& cost = wt == TLHIP_F16 ? COST_F16 : (wt == TLHIP_Q8_0 ? COST_Q8 : COST_Q4);
    TilePlan best;
    double best_us = 1e30;
    for (int c = 0; c < 5; c++) {
        const TileShape& t = SHAPES[c];
        const int64_t tiles = (int64_t)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
        const int steps = (K + t.bk - 1) / t.bk;
        for (int sp : {1, 2, 3, 4, 6, 8}) {
            const size_t bytes = (size_t)sp * M * ((N + 7) & ~7) * sizeof(float);
            if (sp > 1 && (tiles * sp > 320 || steps / sp < 2 || bytes > GEMM_SPLIT_PARTIALS_MAX)) break;
            const int64_t wgs = tiles * sp;
            const int64_t full = wgs / 256, last = wgs % 256;
            const double rounds = (double)(full + (last > 0));
            const double busy = (double)full + (last > 64 ? (last - 64) / 192.0 : 0.0);   // summed over the rounds
            const auto& f = cost.shape[c];
            double us = cost.launch + 1e-6 * K * (cost.weights * N + cost.acts * M * ((N + t.bn - 1) / t.bn)) +
                        rounds * f.fix + busy * f.busy_fix + (rounds - 1.0) * f.later +
                        (steps + sp - 1) / sp * (rounds * f.step + busy * f.busy_step);
            if (sp > 1) us += cost.split + cost.slice * sp + cost.partials * 1e-6 * sp * M * N;
            if (us < best_us) {
                best_us = us;
                best.shape = c;
                best.splits = sp;
                best.ws_bytes = sp > 1 ? bytes : 0;
            }
        }
    }
    best.us = best_us;
    return best;
}

void tile_dims(int shape, int* rows, int* cols) {
    *rows = SHAPES[shape].bm;
    *cols = SHAPES[shape].bn;
}

template <int WT, int TM, int TN, int WM, int WN>
static void launch_tile(hipStream_t s, TileParams& p) {
    using L = Tile<WT, TM, TN, WM, WN>;
    p.mT = (p.M + L::BM - 1) / L::BM;
    p.nT = (p.N + L::BN - 1) / L::BN;
    hipLaunchKernelGGL((gemm_tile_kernel<WT, TM, TN, WM, WN>), dim3((unsigned)(p.mT * p.nT * p.splits)), dim3(512), 0, s, p);
}
template <int WT>
static void launch_shape(hipStream_t s, TileParams& p, int shape) {
    switch (shape) {
        case 0: launch_tile<WT, 4, 2, 1, 2>(s, p); break;
        case 1: launch_tile<WT, 2, 2, 2, 1>(s, p); break;
        case 2: launch_tile<WT, 2, 2, 1, 2>(s, p); break;
        case 3: launch_tile<WT, 2, 2, 1, 1>(s, p); break;
        default: launch_tile<WT, 2, 1, 1, 1>(s, p); break;
    }
}

tlhip_status launch_gemm_tile(hipStream_t s, int wt, const GemvArgs& a, int epi, int ldy, const TilePlan& pl) {
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
    p.splits = pl.splits > 1 && a.ws && pl.ws_bytes <= a.ws_bytes && (uintptr_t)a.ws % 16 == 0 ? pl.splits : 1;
    p.part = p.splits > 1 ? a.ws : nullptr;
    if (epi == EPI_QKV_ROPE) {
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
        p.vec = a.head_dim % 8 == 0 && a.rot % 8 == 0 && ((uintptr_t)a.q_out | (uintptr_t)a.kc | (uintptr_t)a.vc) % 16 == 0;
    }
    if (wt == TLHIP_Q4_0) launch_shape<TLHIP_Q4_0>(s, p, pl.shape);
    else if (wt == TLHIP_Q8_0) launch_shape<TLHIP_Q8_0>(s, p, pl.shape);
    else launch_shape<TLHIP_F16>(s, p, pl.shape);
    if (p.splits > 1) {
        const int64_t items = (int64_t)p.M * ((p.N + 7) / 8);
        hipLaunchKernelGGL(tile_reduce_kernel, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, s, p);
    }
    return TLHIP_OK;
}

}  // namespace tlhip
