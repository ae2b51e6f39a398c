// k_gemm_f32.hip — fp32 FC GEMM with the fused epilogue (gfx950): the MLM head tied to the
// fp32 token embedding, and MulMat nodes whose weights are F32.
//
// Semantics: the reference's F32 MulMat (CPU src/mg-cpu/mg-cpu.cpp:48-72, GPU k_mul_mat_t
// src/mg-opencl/mg-opencl.cpp:60-94): y[m][n] = act(sum_k w[n][k] * x[m][k] + bias[n]) +
// resid[m][n], fp32 accumulation (the summation order differs from the reference's
// sequential k loop), epilogue order of mg-opencl.cpp:36-40, 485-491.
//
// gfx950 mapping: fp32 products on the bf16 matrix unit, every value split into three bf16 parts as
// it goes into LDS (k_split_bf16.h): v_mfma_f32_16x16x4_f32 runs at 1/16 of the bf16 rate, and six
// bf16 products cost 96 cycles where it costs 256. 64 x 64 output tiles per 256-thread workgroup
// (2 x 2 waves of 2 x 2 MFMA tiles), K in steps of 32. What bounds it now is the splitting (6.5 VALU
// operations per value of w and x in every tile) beside the MFMAs: at M = 4112 the VALU is busy 49% of
// the time, the matrix unit 34%. The 768 -> 2025 head against the fp32 instruction on the same tiles:
// M = 257 22.3 -> 19.9 us, M = 4112 123 -> 92 us; error against
// 64 bits 5.0e-7 -> 4.2e-7. Weights take the MFMA A role so a lane holds four consecutive output
// columns of one row; the tile leaves through LDS in whole rows (N = 2025: no aligned stores).
#include "mgh_common.h"
#include "mgh_kernels.h"
#include "k_split_bf16.h"

namespace mgh {

namespace {

constexpr int TB = 64;     // output tile (rows of w and of x)
constexpr int KS = 32;     // K step
constexpr int RS = KS;     // LDS row stride (bf16)

template <int ACT>
__device__ __forceinline__ float act_f(float v) {
    if (ACT == 1) return gelu_erf(v);
    if (ACT == 2) return v / (1.0f + expf(-v));
    return v;
}

// DB: two LDS buffers and two steps' values in registers, one barrier per step; else one of each, so
// that four workgroups share a CU and cover each other's waits
template <int ACT, int BM, int BN, bool DB>
__global__ __launch_bounds__(256, DB ? 2 : 4) void k_gemm_f32(GemmF32Args g) {
    constexpr int I = BN / 32, J = BM / 32;      // 16-row subtiles of w and x per wave (2 x 2 waves)
    constexpr int PW = BN / 64, PX = BM / 64;    // 8-value pieces per thread and step
    constexpr int WPL = BN * RS, XPL = BM * RS;  // halves per plane
    constexpr int TP = BN + 4;                   // transposed row pitch (floats)
    constexpr int HR = 32;                       // output rows per transposed pass
    constexpr int BUF = 3 * (WPL + XPL);         // values per buffer
    constexpr int OPER = (DB ? 2 : 1) * BUF * 2, TRN = HR * TP * 4;
    __shared__ __attribute__((aligned(16))) char lds[OPER > TRN ? OPER : TRN];
    const int M = g.M, N = g.N, K = g.K;
    const int tiles_n = (N + BN - 1) / BN, tiles_m = (M + BM - 1) / BM;
    const int bt = xcd_remap(blockIdx.x, tiles_n * tiles_m);
    const int n0 = (bt % tiles_n) * BN, m0 = (bt / tiles_n) * BM;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = (wave & 1) * (BN / 2), wm = (wave >> 1) * (BM / 2);
    const int l16 = lane & 15, lg = lane >> 4;

    // each thread moves 8 consecutive k of rows tid/4 + 64u; rows past the end re-read the last one
    const int r0 = tid >> 2, c8 = (tid & 3) * 8;
    const float *wp[PW], *xp[PX];
#pragma unroll
    for (int u = 0; u < PW; u++) wp[u] = g.w + (size_t)min(n0 + r0 + 64 * u, N - 1) * K + c8;
#pragma unroll
    for (int u = 0; u < PX; u++) xp[u] = g.x + (size_t)min(m0 + r0 + 64 * u, M - 1) * K + c8;
    f32x4 rg[DB ? 2 : 1][PW + PX][2];
    auto load = [&](f32x4 (&r)[PW + PX][2], int k0) {
        k0 = min(k0, K - KS);                    // past the end: the last step again, never read
#pragma unroll
        for (int u = 0; u < PW + PX; u++) {
            const float* p = (u < PW ? wp[u] : xp[u - PW]) + k0;
            r[u][0] = *(const f32x4*)p, r[u][1] = *(const f32x4*)(p + 4);
        }
    };
    auto store = [&](const f32x4 (&r)[PW + PX][2], int buf) {
        uint16_t *Ws = (uint16_t*)lds + buf * BUF, *Xs = Ws + 3 * WPL;   // [part][row][k]
#pragma unroll
        for (int u = 0; u < PW + PX; u++) {
            const bool x = u >= PW;
            const int v = x ? u - PW : u;
            u32x4 hi, mid, lo;
            split_bf16(r[u][0], r[u][1], hi, mid, lo);
            uint16_t* p = (x ? Xs : Ws) + (r0 + 64 * v) * RS + ((tid & 3) ^ swz32(r0 + 64 * v)) * 8;
            const int pl = x ? XPL : WPL;
            *(u32x4*)p = hi;
            *(u32x4*)(p + pl) = mid;
            *(u32x4*)(p + 2 * pl) = lo;
        }
    };
    auto frag = [&](const uint16_t* B, int pl, int row) {
        const uint16_t* p = B + (row + l16) * RS + (lg ^ swz32(row + l16)) * 8;
        return Frag3{*(const bf16x8*)p, *(const bf16x8*)(p + pl), *(const bf16x8*)(p + 2 * pl)};
    };

    f32x4 acc[J][I];
#pragma unroll
    for (int i = 0; i < I; i++)
#pragma unroll
        for (int j = 0; j < J; j++) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto products = [&](int buf) {
        const uint16_t *Ws = (const uint16_t*)lds + buf * BUF, *Xs = Ws + 3 * WPL;
        Frag3 a[I];
#pragma unroll
        for (int i = 0; i < I; i++) a[i] = frag(Ws, WPL, wn + 16 * i);
#pragma unroll
        for (int j = 0; j < J; j++) {
            const Frag3 b = frag(Xs, XPL, wm + 16 * j);
            mfma_split<I>(a, b, acc[j]);
        }
    };
    load(rg[0], 0);
    if constexpr (DB) {
        auto step = [&](int k0, int buf, f32x4 (&r)[PW + PX][2]) {
            products(buf);
            store(r, buf ^ 1);                   // the next step's; its registers take the third one's
            load(r, k0 + 3 * KS);
            lds_sync();
        };
        load(rg[1], KS);
        store(rg[0], 0);
        load(rg[0], 2 * KS);
        lds_sync();
        for (int k0 = 0; k0 < K; k0 += 2 * KS) {
            step(k0, 0, rg[1]);
            if (k0 + KS < K) step(k0 + KS, 1, rg[0]);
        }
    } else {
        for (int k0 = 0; k0 < K; k0 += KS) {
            lds_sync();                          // the previous step's values are read
            store(rg[0], 0);
            load(rg[0], k0 + KS);
            lds_sync();
            products(0);
        }
    }
    // A sum that is not finite comes from operands or products that are not, or not in the parts' range,
    // where a difference of parts is NaN: a wave that holds such sums takes its tile again on
    // v_mfma_f32_16x16x4_f32, operands straight from memory, 16 k at a time (lane l16, lg: k 4 lg + e
    // in MFMA e), and replaces them. (4112 rows of NaN through the head: 0.30 ms; one output after the
    // other 15.)
    float nf = 0.f;                      // 0, or NaN with a sum that is not finite
#pragma unroll
    for (int j = 0; j < J; j++)
#pragma unroll
        for (int i = 0; i < I; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                acc[j][i][e] *= kSplitUnscale;
                nf = fmaf(acc[j][i][e], 0.f, nf);
            }
    if (__any(nf != nf)) {
        f32x4 sum[J][I];
#pragma unroll
        for (int j = 0; j < J; j++)
#pragma unroll
            for (int i = 0; i < I; i++) sum[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int k0 = 0; k0 < K; k0 += KS) {
            f32x4 w[2][I], x[2][J];
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int k = k0 + 16 * u + 4 * lg;
#pragma unroll
                for (int i = 0; i < I; i++) w[u][i] = *(const f32x4*)(g.w + (size_t)min(n0 + wn + 16 * i + l16, N - 1) * K + k);
#pragma unroll
                for (int j = 0; j < J; j++) x[u][j] = *(const f32x4*)(g.x + (size_t)min(m0 + wm + 16 * j + l16, M - 1) * K + k);
            }
#pragma unroll
            for (int j = 0; j < J; j++)
#pragma unroll
                for (int i = 0; i < I; i++) {
                    f32x4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        t = __builtin_amdgcn_mfma_f32_16x16x4f32(w[e >> 2][i][e & 3], x[e >> 2][j][e & 3], t, 0, 0, 0);
                    sum[j][i] += t;
                }
        }
#pragma unroll
        for (int j = 0; j < J; j++)
#pragma unroll
            for (int i = 0; i < I; i++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (!(fabsf(acc[j][i][e]) < INFINITY)) acc[j][i][e] = sum[j][i][e];
    }
    // register r of tile (i, j) is y[m0+wm+16j+l16][n0+wn+16i+4lg+r]
    // the tile leaves through LDS as whole rows, HR rows of each wave row at a time
    float* T = (float*)lds;
    constexpr int JH = HR / 32;                  // subtiles per wave row and pass
#pragma unroll
    for (int h = 0; h < J / JH; h++) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < JH; j++)
#pragma unroll
            for (int i = 0; i < I; i++)
                *(f32x4*)&T[(16 * JH * (wave >> 1) + 16 * j + l16) * TP + wn + 16 * i + 4 * lg] = acc[h * JH + j][i];
        __syncthreads();
        // thread: column tid % BN, rows tid / BN + (256 / BN) q; consecutive lanes, consecutive columns
        const int c = tid % BN, n = n0 + c;
        const float bias = g.bias && n < N ? g.bias[n] : 0.f;
#pragma unroll
        for (int q = 0; q < HR * BN / 256; q++) {
            const int r = tid / BN + (256 / BN) * q, m = m0 + (r / (16 * JH)) * (BM / 2) + 16 * JH * h + r % (16 * JH);
            if (m >= M || n >= N) continue;
            float v = T[r * TP + c];
            if (g.bias) v += bias;
            v = act_f<ACT>(v);
            const size_t o = (size_t)m * N + n;
            if (g.resid) v += g.resid[o];
            g.y[o] = v;
        }
    }
}

template <bool DB>
hipError_t launch_t(const GemmF32Args& a, hipStream_t s) {
    const dim3 grid((unsigned)(((a.N + TB - 1) / TB) * ((a.M + TB - 1) / TB))), block(256);
    if (a.act == 1) hipLaunchKernelGGL((k_gemm_f32<1, TB, TB, DB>), grid, block, 0, s, a);
    else if (a.act == 2) hipLaunchKernelGGL((k_gemm_f32<2, TB, TB, DB>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((k_gemm_f32<0, TB, TB, DB>), grid, block, 0, s, a);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_gemm_f32(const GemmF32Args& a, hipStream_t s) {
    if (a.M == 0) return hipSuccess;
    // up to one workgroup per CU the K loop's latency counts (M = 257: 19.2 against 23.1 us), beyond
    // it the number of workgroups that share a CU (M = 514: 24.6 against 25.6; M = 4112: 90 against
    // 102). 128-row tiles in either direction: 92 us and more at M = 4112, 33 at M = 514. (All before
    // the values were scaled, which adds 3-4% to each.)
    const int64_t tiles = (int64_t)((a.N + TB - 1) / TB) * ((a.M + TB - 1) / TB);
    return tiles <= 256 ? launch_t<true>(a, s) : launch_t<false>(a, s);
}

}  // namespace mgh
