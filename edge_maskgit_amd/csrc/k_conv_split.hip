// k_conv_split.hip — fp32 convolution of the VQGAN decoder on the bf16 matrix unit: the implicit
// GEMM of k_conv2d_pk (k_vqgan.hip: output pixels x output channels, K tap-major over weights packed
// to [OC][KH][KW][IC]) with every operand split into three bf16 parts (k_split_bf16.h).
//
// What bounds it: v_mfma_f32_16x16x4_f32 runs at 1/16 of the bf16 rate, so six bf16 products cost
// 96 cycles where the fp32 instruction costs 256 (16 x 16 x 32 values). The splitting is VALU work
// (6.5 operations per value), so a tile should use each split value often: 256 pixels x 128 channels
// per workgroup of 8 waves (64 x 64 each), one workgroup per CU and two waves per SIMD. Per 32-deep
// K step a wave issues 96 MFMAs (1536 cycles) and splits 24 values per lane (156 operations, 624
// cycles) for the next step, interleaved with the MFMAs. 128-pixel tiles (32 x 64 per wave) where
// the larger ones leave CUs idle.
// Measured: 256 x 256 x 128, one image 177 -> 98 us (197 TFLOP/s of conv work; MFMA busy 47%, VALU 35%,
// the rest LDS latency that the two waves per SIMD do not cover), error against 64 bits 3.1e-7 ->
// 2.7e-7. The small products in accumulators of their own: 1.1e-7 but 3 us more (64 registers more,
// so fragments are read just before use); the six of a step summed from zero: 7e-8 but 13 us more (64
// additions per step). With K split, where a workgroup per CU and its latency set the time, the
// accumulators of their own cost nothing and are taken (128 x 128 x 128, two images: 66 us either way,
// 7.9e-8 against 1.9e-7).
//  * gather: a thread takes one pixel and 8 consecutive channels per piece as buffer loads (pixel
//    offset per lane, channel plane in the scalar offset; a tap outside the image takes an offset
//    past the range, which loads zero), one K step ahead in registers;
//  * LDS: two buffers of [part][row][32 k] with the 16-byte slots of a row XOR-swizzled
//    (swz32); one barrier per step.
#include <algorithm>

#include "k_conv_common.h"
#include "k_split_bf16.h"
#include "mgh_common.h"
#include "mgh_kernels.h"

namespace mgh {

namespace {

constexpr int KS = 32, BN = 128, NT = 512;

// blockIdx.z = image * splits + split; with SPLIT the K range [split*kps, +kps) goes into its own
// partial plane out[split][image][oc][pixel] (no bias or residual), summed in order by k_conv_reduce
template <int BM, bool SPLIT>
__global__ __launch_bounds__(NT, 2) void k_conv2d_split(ConvPkArgs a) {
    constexpr int I = BM / 64, J = 4;            // 16-row subtiles per wave: pixels, channels
    constexpr int PA = BM * 4 / NT;              // 8-value pixel pieces per thread and step
    constexpr int APL = BM * KS, BPL = BN * KS;  // values per part
    constexpr int BUF = 3 * (APL + BPL);
    __shared__ __attribute__((aligned(16))) uint16_t lds[2 * BUF];

    const int M = a.OW * a.OH, K = a.IC * a.KW * a.KH, OC = a.OC;
    const int z = blockIdx.z;
    const int n = SPLIT ? z / a.splits : z, sp = SPLIT ? z - n * a.splits : 0;
    const int kbeg = sp * a.kps, kend = min(K, kbeg + a.kps), steps = (kend - kbeg) / KS;
    const int m0 = blockIdx.x * BM, n0 = blockIdx.y * BN;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1, l16 = lane & 15, lg = lane >> 4;

    // pixel role: row pa of the tile, channels 8 (cg + (NT / BM) u) .. + 7 of the step
    const int pa = tid % BM, cg = __builtin_amdgcn_readfirstlane(tid / BM);
    const int p = m0 + pa;
    const bool pv = p < M;
    const int ow = pv ? p % a.OW : 0, oh = pv ? p / a.OW : 0;
    const int iw0 = ow * a.stride - a.pad, ih0 = oh * a.stride - a.pad;
    const uint32_t plane = (uint32_t)(a.IW * a.IH) * 4;
    const __amdgpu_buffer_rsrc_t rin = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.in + (size_t)n * a.IC * a.IW * a.IH), (short)0, (int)((uint32_t)a.IC * plane), 0x00020000);
    // weight role: channel row bo, k 8 bq .. + 7 of the step
    const int bo = tid >> 2, bq = tid & 3;
    const float* wrow = a.wpk + (size_t)min(n0 + bo, OC - 1) * K + 8 * bq;

    float ra[PA][8];
    f32x4 rb[2];
    // step state of the next load: channel, tap
    int ic = kbeg % a.IC, kw = (kbeg / a.IC) % a.KW, kh = kbeg / a.IC / a.KW, kk = kbeg;
    uint32_t voff = 0;
    auto tap = [&] {
        const int ih = ih0 + kh, iw = iw0 + kw;
        const bool in = pv && (uint32_t)ih < (uint32_t)a.IH && (uint32_t)iw < (uint32_t)a.IW;
        voff = in ? (uint32_t)(ih * a.IW + iw) * 4 : 0x80000000u;
    };
    tap();
    auto load_a = [&](int u) {
        const uint32_t so = (uint32_t)(ic + 8 * (cg + (NT / BM) * u)) * plane;
#pragma unroll
        for (int e = 0; e < 8; e++)
            ra[u][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rin, (int)voff, (int)(so + e * plane), 0));
    };
    auto load_b = [&] {
        rb[0] = *(const f32x4*)(wrow + kk);
        rb[1] = *(const f32x4*)(wrow + kk + 4);
    };
    // to the next step; past the last one the range's last step is loaded again (never read)
    auto advance = [&] {
        if (kk + KS >= kend) return;
        kk += KS;
        ic += KS;
        if (ic == a.IC) {
            ic = 0;
            if (++kw == a.KW) kw = 0, kh++;
            tap();
        }
    };
    auto put = [&](uint16_t* base, int row, int slot, int part, const f32x4 v0, const f32x4 v1) {
        u32x4 hi, mid, lo;
        split_bf16(v0, v1, hi, mid, lo);
        uint16_t* q = base + row * KS + (slot ^ swz32(row)) * 8;
        *(u32x4*)q = hi;
        *(u32x4*)(q + part) = mid;
        *(u32x4*)(q + 2 * part) = lo;
    };
    auto store_a = [&](int u, int buf) {
        put(lds + buf * BUF, pa, cg + (NT / BM) * u, APL, f32x4{ra[u][0], ra[u][1], ra[u][2], ra[u][3]},
            f32x4{ra[u][4], ra[u][5], ra[u][6], ra[u][7]});
    };
    auto store_b = [&](int buf) { put(lds + buf * BUF + 3 * APL, bo, bq, BPL, rb[0], rb[1]); };
    // fragment of 16 rows from row0: lane (row l16, k 8 lg ..)
    const int fo = l16 * KS;
    auto frag = [&](const uint16_t* base, int row0, int part) {
        const uint16_t* q = base + row0 * KS + fo + (lg ^ swz32(row0 + l16)) * 8;
        return Frag3{*(const bf16x8*)q, *(const bf16x8*)(q + part), *(const bf16x8*)(q + 2 * part)};
    };

    Frag3 fa[I], fb[2];
    f32x4 acc[J][I], rest[SPLIT ? J : 1][I];
#pragma unroll
    for (int j = 0; j < J; j++)
#pragma unroll
        for (int i = 0; i < I; i++) acc[j][i] = rest[SPLIT ? j : 0][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto prod = [&](int i, int j, const Frag3& b) {
        if constexpr (SPLIT) mfma_split1(fa[i], b, acc[j][i], rest[j][i]);
        else mfma_split1(fa[i], b, acc[j][i]);
    };

#pragma unroll
    for (int u = 0; u < PA; u++) load_a(u);
    load_b();
#pragma unroll
    for (int u = 0; u < PA; u++) store_a(u, 0);
    store_b(0);
    advance();
#pragma unroll
    for (int u = 0; u < PA; u++) load_a(u);
    load_b();
    lds_sync();
    auto rows_a = [&](int buf, int i) { return frag(lds + buf * BUF, (BM / 4) * wm + 16 * i, APL); };
    auto rows_b = [&](int buf, int j) { return frag(lds + buf * BUF + 3 * APL, 64 * wn + 16 * j, BPL); };
#pragma unroll
    for (int i = 0; i < I; i++) fa[i] = rows_a(0, i);
    fb[0] = rows_b(0, 0);
    for (int s = 0; s < steps; s++) {
        const int cur = s & 1, nxt = cur ^ 1;
        advance();
#pragma unroll
        for (int j = 0; j < J - 1; j++) {
            fb[(j + 1) & 1] = rows_b(cur, j + 1);
            if (j == 0) {                // (fragment by fragment: the last ones are still arriving)
#pragma unroll
                for (int i = 0; i < I; i++) prod(i, 0, fb[0]);
            } else if constexpr (SPLIT) {
                mfma_split<I>(fa, fb[j & 1], acc[j], rest[j]);
            } else {
                mfma_split<I>(fa, fb[j & 1], acc[j]);
            }
            // the next step's values: split and stored, then the one after requested
            if (j < PA) store_a(j, nxt), load_a(j);
            else if (j == PA) store_b(nxt), load_b();
            __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
            for (int q = 0; q < 6 * I; q++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, I == 4 ? 2 : 4, 0);
            }
        }
        // hand-over: this buffer is read, the next one filled; its first fragments replace the
        // current ones as the last channel subtile's products are done with them
        lds_sync();
        fb[0] = rows_b(nxt, 0);
#pragma unroll
        for (int i = 0; i < I; i++) {
            prod(i, J - 1, fb[1]);
            fa[i] = rows_a(nxt, i);
        }
    }

    if constexpr (SPLIT) {
#pragma unroll
        for (int j = 0; j < J; j++)
#pragma unroll
            for (int i = 0; i < I; i++) acc[j][i] += rest[j][i];
    }
    // A sum that is not finite comes from operands or products that are not, or not in the parts' range,
    // where a difference of parts is NaN: a wave that holds such sums takes its tile again on
    // v_mfma_f32_16x16x4_f32, operands straight from memory, 16 k at a time (lane l16, lg: k 4 lg + e
    // in MFMA e), and replaces them. A tap outside the image is no product (an infinite weight there
    // counts nothing): each slab, one tap, is summed from zero and added where the pixel's tap is
    // inside. (An image of NaN through 256 x 256 x 128: 0.31 ms; one output after the other 27.6.)
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
        int rw0[I], rh0[I];
#pragma unroll
        for (int i = 0; i < I; i++) {
            const int q = min(m0 + (BM / 4) * wm + 16 * i + l16, M - 1);
            rw0[i] = q % a.OW * a.stride - a.pad, rh0[i] = q / a.OW * a.stride - a.pad;
#pragma unroll
            for (int j = 0; j < J; j++) sum[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll 1
        for (int k = kbeg; k < kend; k += 16) {
            const int c = k % a.IC, kx = (k / a.IC) % a.KW, ky = k / a.IC / a.KW;
            f32x4 w[J];
            float x[I][4];
            uint64_t in[I];
#pragma unroll
            for (int j = 0; j < J; j++)
                w[j] = *(const f32x4*)(a.wpk + (size_t)min(n0 + 64 * wn + 16 * j + l16, OC - 1) * K + k + 4 * lg);
#pragma unroll
            for (int i = 0; i < I; i++) {
                const int ih = rh0[i] + ky, iw = rw0[i] + kx;
                const bool inside = (uint32_t)ih < (uint32_t)a.IH && (uint32_t)iw < (uint32_t)a.IW;
                in[i] = __ballot(inside);            // bits 0 .. 15: the pixels of subtile i
                const uint32_t o = inside ? (uint32_t)(ih * a.IW + iw) * 4 + 4 * lg * plane : 0x80000000u;
#pragma unroll
                for (int e = 0; e < 4; e++)
                    x[i][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rin, (int)o, (int)((c + e) * plane), 0));
            }
#pragma unroll
            for (int i = 0; i < I; i++)
#pragma unroll
                for (int j = 0; j < J; j++) {
                    f32x4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int e = 0; e < 4; e++) t = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i][e], w[j][e], t, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 4; e++) sum[j][i][e] += (in[i] >> (4 * lg + e)) & 1 ? t[e] : 0.f;
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
    // register e of tile (i, j): pixel m0 + (BM/4) wm + 16i + 4lg + e, channel n0 + 64wn + 16j + l16
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int oc = n0 + 64 * wn + 16 * j + l16;
        if (oc >= OC) continue;
        const size_t row = ((size_t)(SPLIT ? sp * a.N + n : n) * OC + oc) * M;
#pragma unroll
        for (int i = 0; i < I; i++)
            conv_store<!SPLIT>(a.out, SPLIT ? nullptr : a.bias, SPLIT ? nullptr : a.resid, row, oc,
                               m0 + (BM / 4) * wm + 16 * i + 4 * lg, M, acc[j][i]);
    }
}

}  // namespace

bool conv_split_ok(const ConvPkArgs& a) {
    return a.IC % KS == 0 && a.OC > 16 && (int64_t)a.IC * a.IW * a.IH * 4 < (1ll << 31);
}

template <int BM>
static void launch_split_t(const ConvPkArgs& a, hipStream_t s) {
    const dim3 grid((unsigned)((a.OW * a.OH + BM - 1) / BM), (unsigned)((a.OC + BN - 1) / BN), (unsigned)(a.N * a.splits));
    if (a.splits > 1) hipLaunchKernelGGL((k_conv2d_split<BM, true>), grid, dim3(NT), 0, s, a);
    else hipLaunchKernelGGL((k_conv2d_split<BM, false>), grid, dim3(NT), 0, s, a);
}

void launch_conv_split(const ConvPkArgs& a, hipStream_t s) {
    // 256-pixel tiles while they give most CUs a workgroup, else 128-pixel ones (3 x 3, us, 256 / 128
    // pixels: 256 x 256 x 128 95 / 110, 64 x 64 x 256 40 / 45, 16 x 16 x 512 in 32 splits with two
    // images 32 / 35; with one image, 128 large workgroups, 33 / 25; 32 x 32 x 256 27 / 24; the 1 x 1
    // 128 x 128 x 128, 64 large workgroups, 22 / 14; all before the values were scaled, at most 3%
    // each). Both add each output's K range in the same order, so the choice, which depends on the
    // batch, does not change a result.
    const int64_t wgs = (int64_t)((a.OW * a.OH + 255) / 256) * ((a.OC + BN - 1) / BN) * a.N * a.splits;
    if (wgs >= 200) launch_split_t<256>(a, s);
    else launch_split_t<128>(a, s);
}

}  // namespace mgh
