// kernels_einsum.hip -- the attention einsums of the TL program over many
// query rows ("ihd,jhd->ihj" and "ihj,jhd->ihd" as calls of their own,
// einsum.rs:653-886), on v_mfma_f32_32x32x16_f16 with fp32 accumulation.
//
// Both are bound by the [I, H, J] tensor they write or read.  Measured on
// MI355X at I = J = 400, 32 heads of 64 (10.2 MB of scores), the 8-lane
// kernels / these: scores 152 / 11.2 us, context 45 / 10.6 us.  einsum_rule.hpp
// has the sizes at which each is the faster one.
#include "device_common.hpp"
#include "einsum_rule.hpp"
#include "internal.hpp"

namespace tlhip {

namespace {

// 8 f16 of a row from column j on, zeros past its J columns.
__device__ __forceinline__ h8 load8(const uint16_t* row, int j, int J) {
    if (j + 8 <= J) return __builtin_bit_cast(h8, *(const h8_any*)(row + j));
    u4 v = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int e = 0; e < 8; e++)
        if (j + e < J) v[e / 2] |= (uint32_t)row[j + e] << (16 * (e & 1));
    return __builtin_bit_cast(h8, v);
}

// scores[i, h, j] = sum_d q[i, h, d] k[j, kvh, d]: a workgroup computes 64
// query rows x 128 keys of one head, each of its 4 waves 32 x 64.  The
// operands are whole rows (16 bytes of a row per lane and 16 dims); the
// product is formed transposed, so a lane holds 4 consecutive keys of a row,
// and goes through LDS to 16-byte stores along j.
template <int D>
__global__ __launch_bounds__(256) void scores_mfma_kernel(const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
                                                          uint16_t* __restrict__ out, int I, int J, int H, int Hkv,
                                                          int nJ, int nI) {
    constexpr int RS = 64 + 8;   // LDS row stride
    __shared__ __attribute__((aligned(16))) uint16_t tile[4][32 * RS];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, l32 = lane & 31, hh = lane >> 5;
    const int b = blockIdx.x, h = b / (nJ * nI), it = b / nJ % nI, jt = b % nJ;
    const int i0 = it * 64 + 32 * (w >> 1), j0 = jt * 128 + 64 * (w & 1);
    if (i0 >= I || j0 >= J) return;   // (no barrier below: each wave has its own LDS rows)
    const uint16_t* qr = q + ((size_t)min(i0 + l32, I - 1) * H + h) * D + 8 * hh;
    const uint16_t* kr[2];
#pragma unroll
    for (int a = 0; a < 2; a++) kr[a] = k + ((size_t)min(j0 + 32 * a + l32, J - 1) * Hkv + h / (H / Hkv)) * D + 8 * hh;
    h8 qf[D / 16], kf[2][D / 16];
#pragma unroll
    for (int t = 0; t < D / 16; t++) {
        qf[t] = *(const h8*)(qr + 16 * t);
#pragma unroll
        for (int a = 0; a < 2; a++) kf[a][t] = *(const h8*)(kr[a] + 16 * t);
    }
    f16v acc[2] = {f16v{0}, f16v{0}};
#pragma unroll
    for (int t = 0; t < D / 16; t++)
#pragma unroll
        for (int a = 0; a < 2; a++) acc[a] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[a][t], qf[t], acc[a], 0, 0, 0);
    uint16_t* mine = tile[w];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const uint32_t lo = (uint32_t)f2h(acc[a][4 * r]) | ((uint32_t)f2h(acc[a][4 * r + 1]) << 16);
            const uint32_t hi = (uint32_t)f2h(acc[a][4 * r + 2]) | ((uint32_t)f2h(acc[a][4 * r + 3]) << 16);
            *(uint2*)(mine + l32 * RS + 32 * a + 8 * r + 4 * hh) = uint2{lo, hi};
        }
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int row = 8 * u + (lane >> 3), c = lane & 7, i = i0 + row, j = j0 + 8 * c;
        if (i >= I || j >= J) continue;
        const uint16_t* src = mine + row * RS + 8 * c;
        uint16_t* dst = out + ((size_t)i * H + h) * J + j;
        if (j + 8 <= J) {
            *(h8_any*)dst = __builtin_bit_cast(h8_any, *(const u4*)src);
        } else {
            for (int e = 0; j + e < J; e++) dst[e] = src[e];
        }
    }
}

// context[i, h, d] = sum_j p[i, h, j] v[j, kvh, d]: a workgroup computes 32
// query rows of one head, its waves taking 32-key tiles in turn.  A wave
// transposes its V tile through LDS (pairs of rows, 4-byte writes) into the
// operand layout and loads the next tile while the matrix cores run; the four
// fp32 results are added in wave order.
template <int D>
__global__ __launch_bounds__(256) void context_mfma_kernel(const uint16_t* __restrict__ p, const uint16_t* __restrict__ v,
                                                           uint16_t* __restrict__ out, int I, int J, int H, int Hkv,
                                                           int nI) {
    constexpr int ND = (D + 31) / 32, C8 = D / 8, NV = (16 * C8 + 63) / 64, RS = 32 + 8;
    constexpr int VT = ND * 32 * RS;   // one wave's transposed V tile, halves
    constexpr int SMEM = 4 * VT * 2 > 4 * 32 * D * 4 ? 4 * VT * 2 : 4 * 32 * D * 4;
    __shared__ __attribute__((aligned(16))) uint8_t smem[SMEM];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, l32 = lane & 31, hh = lane >> 5;
    const int h = blockIdx.x / nI, i0 = blockIdx.x % nI * 32;
    const uint16_t* pr = p + ((size_t)min(i0 + l32, I - 1) * H + h) * J;
    const uint16_t* vb = v + (size_t)(h / (H / Hkv)) * D;
    uint16_t* vt = (uint16_t*)smem + w * VT;
    const int nt = (J + 31) / 32;

    h8 pf[2];
    u4 vr[NV][2];
    auto load = [&](int jt) {
#pragma unroll
        for (int t = 0; t < 2; t++) pf[t] = load8(pr, 32 * jt + 16 * t + 8 * hh, J);
#pragma unroll
        for (int u = 0; u < NV; u++) {
            const int x = lane + 64 * u, j = 32 * jt + 2 * (x / C8), c = x % C8;
#pragma unroll
            for (int s = 0; s < 2; s++)
                vr[u][s] = x < 16 * C8 && j + s < J ? *(const u4*)(vb + (size_t)(j + s) * Hkv * D + 8 * c) : u4{0u, 0u, 0u, 0u};
        }
    };
    f16v acc[ND];
#pragma unroll
    for (int n = 0; n < ND; n++) acc[n] = f16v{0};
    if (w < nt) load(w);
    for (int jt = w; jt < nt; jt += 4) {
#pragma unroll
        for (int u = 0; u < NV; u++) {
            const int x = lane + 64 * u, r = x / C8, c = x % C8;
            if (x < 16 * C8) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    *(uint32_t*)(vt + (8 * c + 2 * e) * RS + 2 * r) = pack_lo(vr[u][0][e], vr[u][1][e]);
                    *(uint32_t*)(vt + (8 * c + 2 * e + 1) * RS + 2 * r) = pack_hi(vr[u][0][e], vr[u][1][e]);
                }
            }
        }
        const h8 a0 = pf[0], a1 = pf[1];
        if (jt + 4 < nt) load(jt + 4);
#pragma unroll
        for (int n = 0; n < ND; n++) {
            const uint16_t* row = vt + (32 * n + l32) * RS + 8 * hh;
            acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(*(const h8*)row, a0, acc[n], 0, 0, 0);
            acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(*(const h8*)(row + 16), a1, acc[n], 0, 0, 0);
        }
    }
    __syncthreads();
    float* red = (float*)smem;   // [wave][row][D]
#pragma unroll
    for (int n = 0; n < ND; n++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int d = 32 * n + 8 * r + 4 * hh;
            if (d < D)
                *(f4*)(red + (w * 32 + l32) * D + d) =
                    f4{acc[n][4 * r], acc[n][4 * r + 1], acc[n][4 * r + 2], acc[n][4 * r + 3]};
        }
    __syncthreads();
    for (int x = threadIdx.x; x < 32 * C8; x += 256) {
        const int row = x / C8, c = x % C8;
        if (i0 + row >= I) continue;
        u4 o;
#pragma unroll
        for (int g = 0; g < 2; g++) {
            f4 s = *(const f4*)(red + row * D + 8 * c + 4 * g);
#pragma unroll
            for (int k = 1; k < 4; k++) s += *(const f4*)(red + (k * 32 + row) * D + 8 * c + 4 * g);
            o[2 * g] = (uint32_t)f2h(s[0]) | ((uint32_t)f2h(s[1]) << 16);
            o[2 * g + 1] = (uint32_t)f2h(s[2]) | ((uint32_t)f2h(s[3]) << 16);
        }
        *(u4*)(out + ((size_t)(i0 + row) * H + h) * D + 8 * c) = o;
    }
}

// Head dims the kernels are built for; rows of q, k, v and out on 16-byte
// boundaries.
bool mfma_rows_ok(int D, uintptr_t aligned) { return (D == 64 || D == 80 || D == 128) && aligned % 16 == 0; }

}  // namespace

bool launch_scores_mfma(hipStream_t s, const uint16_t* q, const uint16_t* k, uint16_t* sc, int I, int J, int H, int Hkv,
                        int D) {
    const int nJ = (J + 127) / 128, nI = (I + 63) / 64;
    const int64_t blocks = (int64_t)nJ * nI * H;
    if (!scores_mfma_wins(I, H, J) || !mfma_rows_ok(D, (uintptr_t)q | (uintptr_t)k) || blocks > 0x7fffffff) return false;
    const dim3 grid((unsigned)blocks);
    if (D == 64) hipLaunchKernelGGL(scores_mfma_kernel<64>, grid, dim3(256), 0, s, q, k, sc, I, J, H, Hkv, nJ, nI);
    else if (D == 80) hipLaunchKernelGGL(scores_mfma_kernel<80>, grid, dim3(256), 0, s, q, k, sc, I, J, H, Hkv, nJ, nI);
    else hipLaunchKernelGGL(scores_mfma_kernel<128>, grid, dim3(256), 0, s, q, k, sc, I, J, H, Hkv, nJ, nI);
    return true;
}

bool launch_context_mfma(hipStream_t s, const uint16_t* p, const uint16_t* v, uint16_t* out, int I, int J, int H, int Hkv,
                         int D) {
    const int nI = (I + 31) / 32;
    const int64_t blocks = (int64_t)nI * H;
    if (!mfma_rows_ok(D, (uintptr_t)v | (uintptr_t)out) || !context_mfma_wins(I, H, J, D) || blocks > 0x7fffffff) return false;
    const dim3 grid((unsigned)blocks);
    if (D == 64) hipLaunchKernelGGL(context_mfma_kernel<64>, grid, dim3(256), 0, s, p, v, out, I, J, H, Hkv, nI);
    else if (D == 80) hipLaunchKernelGGL(context_mfma_kernel<80>, grid, dim3(256), 0, s, p, v, out, I, J, H, Hkv, nI);
    else hipLaunchKernelGGL(context_mfma_kernel<128>, grid, dim3(256), 0, s, p, v, out, I, J, H, Hkv, nI);
    return true;
}

}  // namespace tlhip
