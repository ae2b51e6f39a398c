// k_flash_attn.hip — fused self-attention with fp16 K/V (gfx950).
//
// Semantics: the reference's k_flash_attention_h (src/mg-opencl/mg-opencl.cpp:859-937) with
// the CPU oracle k_flash_attention (src/mg-cpu/mg-cpu.cpp:211-239) for the math:
//   per (batch b, head h, query s): q, k, v rounded to fp16; score_t = (q . k_t) * scale in
//   fp32; softmax over keys in fp32 (online, max-subtracted); o = sum_t p_t v_t / sum_t p_t.
// Inputs are strided {D, S, H, B} views (element strides st[0..3]); the reference passes
// the q/k/v FC outputs [S*B][H*D] with st = {1, H*D, D, H*D*S} (mg-opencl.cpp:1493-1496).
// The output strides are a parameter too, so the head merge that follows in the reference
// graph (permute + cont, mg-transformer.cpp:84-85) is written directly.
//
// Three kernels: k_attn_head (S <= 272: a head's K and V resident in LDS), k_attn_long (longer
// sequences; both need unit feature strides and aligned rows) and k_flash_attn_f16kv (any strides).
// gfx950 mapping of the last (one workgroup = 4 waves = 64 queries of one (b, h); keys in chunks of
// 64 staged once per workgroup in LDS as fp16):
//  * Scores as S^T = K . Q^T on v_mfma_f32_16x16x32_f16 (two 16-wide d chunks per
//    instruction, an odd last chunk paired with zeros): fp16 products are exact in fp32, so
//    only the summation order differs from the reference. The S^T accumulator layout (lane
//    = query, registers = 4 consecutive keys) is exactly the A-operand layout of the next
//    product, so P . V needs no data exchange between lanes.
//  * Softmax statistics per query in fp32 (max, running sum), cross-lane over the 4 lane
//    groups; exp is the fp32 expf.
//  * P . V on the same MFMA with P split into fp16 hi + lo parts (two instructions), so the
//    fp32 probabilities are applied to ~2^-22 — the reference multiplies them in fp32.
// LDS rows are padded (K: D+8 halves, V^T: 72 halves) so the fragment reads are
// bank-conflict free.
#include <algorithm>
#include <type_traits>

#include "mgh_common.h"
#include "mgh_kernels.h"

namespace mgh {

namespace {

typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f16x8 cat8(f16x4 a, f16x4 b) {
    return f16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
}

// -1.0f as a value the compiler cannot fold: with it, fmaf((float)h, -1, p) for an fp16 h
// is selected as v_fma_mix_f32 (h read as an fp16 half of its register, no conversion), where
// the constant form becomes a conversion and a subtraction. A scalar move, read by VALU
// instructions only.
__device__ __forceinline__ float opaque_neg_one() {
    float m;
    asm("s_mov_b32 %0, 0xbf800000" : "=s"(m));
    return m;
}

constexpr int KT = 64;             // keys per LDS chunk
constexpr int VLD = KT + 8;        // V^T row stride (halves)

template <int DC>
__global__ __launch_bounds__(256) void k_flash_attn_f16kv(FaArgs a) {
    constexpr int D = 16 * DC;
    constexpr int KLD = D + 8;     // K row stride (halves)
    __shared__ __attribute__((aligned(16))) _Float16 Ks[KT * KLD];
    __shared__ __attribute__((aligned(16))) _Float16 Vt[D * VLD];

    const int S = a.S;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int l16 = lane & 15, lg = lane >> 4;
    const int h = blockIdx.y, b = blockIdx.z;
    const int q0w = blockIdx.x * 64 + wave * 16;
    const bool active = q0w < S;
    const int64_t base = (int64_t)b * a.st[3] + (int64_t)h * a.st[2];

    // Q as the B operand: lane = query q0w + l16, k = d = 16c + 4lg + j
    f16x4 qf[DC];
    {
        const int qi = min(q0w + l16, S - 1);
#pragma unroll
        for (int c = 0; c < DC; c++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                qf[c][j] = (_Float16)a.q[base + (int64_t)qi * a.st[1] + (int64_t)(16 * c + 4 * lg + j) * a.st[0]];
    }

    f32x4 O[DC];
#pragma unroll
    for (int c = 0; c < DC; c++) O[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;          // statistics of query q0w + l16

    for (int k0 = 0; k0 < S; k0 += KT) {
        __syncthreads();                   // the previous chunk is consumed
        for (int idx = tid; idx < KT * D; idx += 256) {
            const int key = idx / D, d = idx - key * D, t = k0 + key;
            float kv = 0.f, vv = 0.f;
            if (t < S) {
                const int64_t off = base + (int64_t)t * a.st[1] + (int64_t)d * a.st[0];
                kv = a.k[off];
                vv = a.v[off];
            }
            Ks[key * KLD + d] = (_Float16)kv;
            Vt[d * VLD + key] = (_Float16)vv;
        }
        __syncthreads();
        if (!active) continue;

        // scores: register r of subtile t holds key k0 + 16t + 4lg + r for query l16
        f32x4 sc[KT / 16];
#pragma unroll
        for (int t = 0; t < KT / 16; t++) {
            // pairs of 16-wide d chunks on the 32-deep MFMA (k = 8lg + j: d = 16(c + j/4) + 4lg +
            // j%4 in both operands); an odd last chunk is paired with zeros (the 16-deep MFMA
            // takes as long, and a 16-deep MFMA accumulating right after a 32-deep one into
            // the same registers gave wrong sums)
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
            const _Float16* krow = &Ks[(16 * t + l16) * KLD + 4 * lg];
#pragma unroll
            for (int c = 0; c < DC; c += 2) {
                const f16x4 k1 = c + 1 < DC ? *(const f16x4*)(krow + 16 * c + 16) : f16x4{0, 0, 0, 0};
                const f16x4 q1 = c + 1 < DC ? qf[c + 1] : f16x4{0, 0, 0, 0};
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(cat8(*(const f16x4*)(krow + 16 * c), k1),
                                                             cat8(qf[c], q1), acc, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int key = k0 + 16 * t + 4 * lg + r;
                sc[t][r] = key < S ? acc[r] * a.scale : -INFINITY;
            }
        }
        float mx = -INFINITY;
#pragma unroll
        for (int t = 0; t < KT / 16; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) mx = fmaxf(mx, sc[t][r]);
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float mn = fmaxf(m, mx);
        const float alpha = expf(m - mn);
        float ps = 0.f;
#pragma unroll
        for (int t = 0; t < KT / 16; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float p = sc[t][r] == -INFINITY ? 0.f : expf(sc[t][r] - mn);
                sc[t][r] = p;
                ps += p;
            }
        ps += __shfl_xor(ps, 16);
        ps += __shfl_xor(ps, 32);
        l = alpha * l + ps;
        m = mn;

        // O rows are queries 4lg + r: rescale by that query's alpha (held by lane 4lg + r)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float ar = __shfl(alpha, 4 * lg + r);
#pragma unroll
            for (int c = 0; c < DC; c++) O[c][r] *= ar;
        }
        // O += P . V with P = hi + lo in fp16 (A operand: query l16, keys 16t + 4lg + j)
#pragma unroll
        for (int t = 0; t < KT / 16; t++) {
            f16x4 ph, pl;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                ph[j] = (_Float16)sc[t][j];
                pl[j] = (_Float16)(sc[t][j] - (float)ph[j]);
            }
#pragma unroll
            for (int c = 0; c < DC; c++) {
                const f16x4 vf = *(const f16x4*)&Vt[(16 * c + l16) * VLD + 16 * t + 4 * lg];
                O[c] = __builtin_amdgcn_mfma_f32_16x16x16f16(ph, vf, O[c], 0, 0, 0);
                O[c] = __builtin_amdgcn_mfma_f32_16x16x16f16(pl, vf, O[c], 0, 0, 0);
            }
        }
    }
    if (!active) return;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const float inv = 1.f / __shfl(l, 4 * lg + r);
        const int qi = q0w + 4 * lg + r;
        if (qi >= S) continue;
        const int64_t ro = (int64_t)b * a.os[3] + (int64_t)h * a.os[2] + (int64_t)qi * a.os[1];
#pragma unroll
        for (int c = 0; c < DC; c++) {
            const int64_t e = ro + (int64_t)(16 * c + l16) * a.os[0];
            if (a.o16) a.o16[e] = (_Float16)(O[c][r] * inv);
            else a.o[e] = O[c][r] * inv;
        }
    }
}


// Whole-head variant for S <= 16*KT: one workgroup per (h, b) stages the head's K (row-major)
// and V (transposed) once in LDS as fp16, then each wave takes 16-query tiles and computes all
// scores of a tile in registers, a plain (not online) max-subtracted softmax over the row —
// the order of the reference CPU kernel — and P . V. K/V are read once per head instead of
// once per query tile (needs unit d stride and 16-byte aligned rows; q/k/v either fp32,
// rounded to fp16 on load, or already fp16). The exponentials use the hardware exp2 on
// log2(e)-scaled scores (relative error ~1e-7, far inside the attention tolerance), with the
// scale folded into one fma. Both products run on v_mfma_f32_16x16x32_f16 (the 16-deep
// instruction takes as many cycles on gfx950): scores over pairs of d chunks, P . V over pairs
// of key tiles (k = 8lg + j maps to key 16(t + j/4) + 4lg + j%4 in both operands, so the score
// registers are the P operand as they stand). The work per tile is VALU-bound (exp, the
// hi/lo split of P), so the VALU is kept to what the math needs: P . V is computed transposed
// (each lane ends with consecutive features of one query: one division, 8/16-byte stores),
// the row sums come from the MFMA on an all-ones operand, the lo part of P takes one
// v_fma_mix_f32 per element, and LDS fragments are read ahead of their MFMAs.
// At most NW waves (a workgroup takes min(NW, ~half the query tiles) waves), so the score
// registers (4 * KT per lane) fit without spilling: 17 key tiles take 9 waves (3 per SIMD,
// 168 registers) only for fp16 q/k/v at D <= 48 with a 17th, partial tile (S = 257 .. 272);
// at D = 64, with fp32 q/k/v (the next tile's Q held as fp32) or for S <= 256 (16 query
// tiles, two per wave) 8 (256 registers per wave, two waves per SIMD); 32 key tiles with
// D >= 48 need more than 256, so there one wave per SIMD
template <int DC, int KT, bool I16, bool TAIL>
constexpr int kHeadWaves = KT <= 17 ? std::min((KT + 1) / 2, DC >= 4 || !I16 || !TAIL ? 8 : 9)
                                    : (KT == 32 && DC >= 3 ? 4 : 8);

// 4 consecutive elements of q/k/v as fp16: rounded from fp32 (RNE) or, with I16, loaded as
// stored (the producer rounded them the same way)
template <bool I16>
__device__ __forceinline__ f16x4 load_h4(const float* p32, const _Float16* p16, int64_t e) {
    if (I16) return *(const f16x4*)(p16 + e);
    const f32x4 v = *(const f32x4*)(p32 + e);
    return f16x4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
}
// 8 consecutive elements (e % 8 == 0): one 16-byte load of fp16 rows when they are 16-byte
// aligned (A16), two 8-byte loads otherwise; fp32 rows as two 16-byte loads, rounded
template <bool I16, bool A16>
__device__ __forceinline__ f16x8 load_h8(const float* p32, const _Float16* p16, int64_t e) {
    if (I16 && A16) return *(const f16x8*)(p16 + e);
    return cat8(load_h4<I16>(p32, p16, e), load_h4<I16>(p32, p16, e + 4));
}

// TAIL: S > 16 (KT - 1), so every key tile but the last is full (no masking there).
// A16: fp16 inputs whose rows start on 16-byte boundaries (element strides multiples of 8).
template <int DC, int KT, bool I16, bool TAIL, bool A16>
__global__ __launch_bounds__(64 * (kHeadWaves<DC, KT, I16, TAIL>)) void k_attn_head(FaArgs a) {
    constexpr int D = 16 * DC;
    // K row stride (halves): an odd number of 16-wide d chunks is padded with one chunk of
    // zeros, the upper half of the last score MFMA's K operand, so it is read, not zeroed
    constexpr int KLD = D + 8;
    constexpr int SP = 16 * KT;        // keys, padded
    constexpr int VT = SP + 8;         // V^T row stride (halves)
    __shared__ __attribute__((aligned(16))) _Float16 Ks[SP * KLD];
    __shared__ __attribute__((aligned(16))) _Float16 Vt[D * VT];

    const int S = a.S;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, nw = blockDim.x >> 6;
    const int l16 = lane & 15, lg = lane >> 4;
    // XCD-aware placement: workgroup i runs on XCD i % 8, so the logical (query split, head,
    // image) order is remapped into contiguous runs per XCD — each XCD takes whole images, whose
    // q/k/v rows (all heads interleaved in one row) its L2 then fetches once
    const int QS = gridDim.z;
    const int lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    const int lid = xcd_remap(lin, gridDim.x * gridDim.y * QS);
    const int zq = lid % QS, hb = lid / QS;
    const int h = hb % gridDim.x, b = hb / gridDim.x;
    const int64_t base = (int64_t)b * a.st[3] + (int64_t)h * a.st[2];

    // The staging is latency-bound (one workgroup per CU at typical shapes), so each round
    // issues all of a thread's K and V loads before it stores any, and the first query tile's
    // Q is requested with them: at the usual shapes one round trip fills LDS.
    // K row-major: a task moves 8 elements of a key row. V transposed: a task loads an
    // 8-key x 8-d block and stores it as eight 16-byte rows of V^T.
    constexpr int DW = D / 8;
    constexpr int KTASK = SP * DW, VTASK = (SP / 8) * DW;
    constexpr int UK = 8;              // K tasks per thread and round (one V task: 8 loads)
    static_assert(KTASK == UK * VTASK, "one V task per UK K tasks");

    const int nqt = (S + 15) / 16;
    const int qstep = nw * gridDim.z;
    int qt = zq * nw + wave;           // query split z takes query tiles z*nw + wave, + qstep, ...
    // Q as the B operand: lane = query 16t + l16, k = d = 16c + 4lg + j
    f16x4 qf[DC];
    auto load_q = [&](int t) {
        const int qi = min(16 * t + l16, S - 1);
        const int64_t qrow = base + (int64_t)qi * a.st[1];
#pragma unroll
        for (int c = 0; c < DC; c++) qf[c] = load_h4<I16>(a.q, a.q16, qrow + 16 * c + 4 * lg);
    };
    if (qt < nqt) load_q(qt);

    // rounds are workgroup-uniform: round r0 takes K tasks UK*r0 .. UK*(r0 + nth) - 1 and V
    // tasks r0 .. r0 + nth - 1
    for (int r0 = 0; r0 < VTASK; r0 += blockDim.x) {
        f16x8 kv[UK], vv[8];
        const f16x8 z8 = {0, 0, 0, 0, 0, 0, 0, 0};
        const int iv = r0 + tid, kg = iv / DW, dv = 8 * (iv - kg * DW);
#pragma unroll
        for (int u = 0; u < UK; u++) {
            const int idx = UK * r0 + u * blockDim.x + tid;
            const int t = idx / DW, d = 8 * (idx - t * DW);
            kv[u] = z8;
            if (idx < KTASK && t < S) kv[u] = load_h8<I16, A16>(a.k, a.k16, base + (int64_t)t * a.st[1] + d);
        }
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int t = 8 * kg + i;
            vv[i] = z8;
            if (iv < VTASK && t < S) vv[i] = load_h8<I16, A16>(a.v, a.v16, base + (int64_t)t * a.st[1] + dv);
        }
#pragma unroll
        for (int u = 0; u < UK; u++) {
            const int idx = UK * r0 + u * blockDim.x + tid;
            const int t = idx / DW, d = 8 * (idx - t * DW);
            if (idx < KTASK) *(f16x8*)&Ks[t * KLD + d] = kv[u];
        }
        if (iv < VTASK) {
#pragma unroll
            for (int j = 0; j < 8; j++)
                *(f16x8*)&Vt[(dv + j) * VT + 8 * kg] = f16x8{vv[0][j], vv[1][j], vv[2][j], vv[3][j],
                                                            vv[4][j], vv[5][j], vv[6][j], vv[7][j]};
        }
    }
    __syncthreads();

    // scores in log2 units: exp(s*scale - max) = exp2(s*scale*log2(e) - max'), evaluated with
    // the hardware exp2 (v_exp_f32, ~1 ulp)
    const float scale2 = a.scale * 1.4426950408889634f;
    // Output rows are written with 8-byte (fp16) or 16-byte (fp32) stores when the features are
    // unit-stride and every row starts 16-byte aligned, element by element otherwise.
    const bool vec = a.os[0] == 1 && ((a.os[1] | a.os[2] | a.os[3]) & 3) == 0 &&
                     ((uintptr_t)(a.o16 ? (const void*)a.o16 : (const void*)a.o) & 15) == 0;
    constexpr int KC = (DC + 1) / 2;   // 32-deep MFMAs per score tile
    constexpr int NPT = (KT + 1) / 2;  // key-tile pairs of P . V (an odd last tile with zeros)
    // LDS fragment prefetch distances (key tiles for K, key-tile pairs for V), as far as the
    // registers allow
    constexpr int PF = KT <= 17 ? (DC <= 3 ? 2 : 0) : (DC <= 2 ? 1 : 0);
    constexpr int PFV = KT <= 17 && DC <= 3 ? 1 : 0;
    // P . V is computed transposed, O^T = V^T . P^T, with row i of the chunk-c V^T fragment
    // holding feature d = 4 DC (i / 4) + 4c + i % 4: O^T register r of chunk c in lane (l16,
    // lg) is then feature 4 DC lg + 4c + r of query q0 + l16, so each lane ends with 4 DC
    // consecutive features of one query and that query's softmax sum.
    const int vrow0 = 4 * DC * (l16 >> 2) + (l16 & 3);
    const float m1 = opaque_neg_one();
    for (; qt < nqt; qt += qstep) {
        const int q0 = 16 * qt;
        // Q as the B operand of the score MFMAs, d chunks in pairs
        f16x8 qb[KC];
#pragma unroll
        for (int i = 0; i < KC; i++)
            qb[i] = cat8(qf[2 * i], 2 * i + 1 < DC ? qf[2 * i + 1] : f16x4{0, 0, 0, 0});
        // scores: register r of key tile t holds key 16t + 4lg + r of query q0 + l16
        f32x4 sc[KT];
        float mx = -INFINITY;
        // pairs of 16-wide d chunks on the 32-deep MFMA (k = 8lg + j: d = 16(c + j/4) + 4lg + j%4
        // in both operands); an odd last chunk is paired with zeros (the 16-deep MFMA takes as
        // long, and a 16-deep MFMA accumulating right after a 32-deep one into the same
        // registers gave wrong sums). Fragments are read PF key tiles ahead.
        f16x8 kf[PF + 1][KC];
        auto kfrag = [&](int t, int i) {
            const _Float16* krow = &Ks[(16 * t + l16) * KLD + 4 * lg + 32 * i];
            return cat8(*(const f16x4*)krow, 2 * i + 1 < DC ? *(const f16x4*)(krow + 16) : f16x4{0, 0, 0, 0});
        };
        auto load_k = [&](int t, f16x8 (&f)[KC]) {
#pragma unroll
            for (int i = 0; i < KC; i++) f[i] = kfrag(t, i);
        };
#pragma unroll
        for (int t = 0; t < PF && t < KT; t++) load_k(t, kf[t]);
#pragma unroll
        for (int t = 0; t < KT; t++) {
            if (PF && t + PF < KT) load_k(t + PF, kf[(t + PF) % (PF + 1)]);
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < KC; i++)   // without prefetch, one fragment at a time
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(PF ? kf[t % (PF + 1)][i] : kfrag(t, i), qb[i], acc, 0, 0, 0);
            // raw scores; keys past S are -inf (with TAIL only the last tile holds such keys;
            // otherwise the tiles from key S on, a uniform branch)
            if ((TAIL && t < KT - 1) || 16 * t + 16 <= S) {
                sc[t] = acc;
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++) sc[t][r] = 16 * t + 4 * lg + r < S ? acc[r] : -INFINITY;
            }
            // the running max takes the previous tile, whose MFMAs have completed by now
            if (t > 0) {
                mx = fmaxf(fmaxf(mx, sc[t - 1][0]), sc[t - 1][1]);
                mx = fmaxf(fmaxf(mx, sc[t - 1][2]), sc[t - 1][3]);
            }
            __builtin_amdgcn_sched_barrier(0);  // the fragment reads stay PF tiles ahead
        }
        mx = fmaxf(fmaxf(mx, sc[KT - 1][0]), sc[KT - 1][1]);
        mx = fmaxf(fmaxf(mx, sc[KT - 1][2]), sc[KT - 1][3]);
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        // the scores are done with Q: request the next tile's while this one's P . V runs
        if (qt + qstep < nqt) load_q(qt + qstep);
        // scale2 > 0 (checked at launch), so the max of the scaled scores is the scaled max;
        // p = exp2(s * scale2 - max) as one fma, and exp2(-inf) = 0 for the masked keys
        const float mxs = mx * scale2;
#pragma unroll
        for (int t = 0; t < KT; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) sc[t][r] = __builtin_amdgcn_exp2f(fmaf(sc[t][r], scale2, -mxs));
        // O^T += V^T . P^T, P = hi + lo in fp16 (B operand: query l16, keys 16t + 4lg + j): hi
        // is P rounded toward zero, lo the exact remainder P - hi rounded toward zero
        // (|P - hi - lo| <= 2^-20 P, or 2^-24 where lo is an fp16 subnormal). The row sums
        // come from the same MFMAs on an all-ones V^T chunk (S1 = 1 . P^T: every register of
        // lane (l16, lg) holds the sum of query l16), so they add exactly the hi + lo that
        // the numerators use.
        f32x4 O[DC], S1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < DC; c++) O[c] = f32x4{0.f, 0.f, 0.f, 0.f};
        const f16x4 z4 = {0, 0, 0, 0};
        const f16x8 ones = {1, 1, 1, 1, 1, 1, 1, 1};
        // hi and lo operands of key tiles t, t + 1 (t + 1 = KT: zeros); p - hi is exact in fp32
        // and taken as one v_fma_mix_f32 (m1 = -1) per element
        auto split = [&](int t, f16x8& ph, f16x8& pl) {
            const f32x4 zf = {0.f, 0.f, 0.f, 0.f};
            const f32x4 a = sc[t], b = t + 1 < KT ? sc[t + 1] : zf;
            const auto h0 = __builtin_amdgcn_cvt_pkrtz(a[0], a[1]), h1 = __builtin_amdgcn_cvt_pkrtz(a[2], a[3]);
            const auto h2 = __builtin_amdgcn_cvt_pkrtz(b[0], b[1]), h3 = __builtin_amdgcn_cvt_pkrtz(b[2], b[3]);
            const auto l0 = __builtin_amdgcn_cvt_pkrtz(fmaf((float)h0[0], m1, a[0]), fmaf((float)h0[1], m1, a[1]));
            const auto l1 = __builtin_amdgcn_cvt_pkrtz(fmaf((float)h1[0], m1, a[2]), fmaf((float)h1[1], m1, a[3]));
            const auto l2 = __builtin_amdgcn_cvt_pkrtz(fmaf((float)h2[0], m1, b[0]), fmaf((float)h2[1], m1, b[1]));
            const auto l3 = __builtin_amdgcn_cvt_pkrtz(fmaf((float)h3[0], m1, b[2]), fmaf((float)h3[1], m1, b[3]));
            auto u = [](auto v) { return __builtin_bit_cast(uint32_t, v); };
            ph = __builtin_bit_cast(f16x8, u32x4{u(h0), u(h1), u(h2), u(h3)});
            pl = __builtin_bit_cast(f16x8, u32x4{u(l0), u(l1), u(l2), u(l3)});
        };
        // pairs of key tiles on the 32-deep MFMA (k = 8lg + j: key 16(t + j/4) + 4lg + j%4 in
        // both operands); an odd last tile is paired with zeros. V^T fragments are read PF
        // pairs ahead.
        f16x8 vf[PFV + 1][DC];
        auto vfrag = [&](int p, int c) {
            const _Float16* vrow = &Vt[(vrow0 + 4 * c) * VT + 32 * p + 4 * lg];
            return cat8(*(const f16x4*)vrow, 2 * p + 1 < KT ? *(const f16x4*)(vrow + 16) : z4);
        };
        auto load_v = [&](int p, f16x8 (&f)[DC]) {
#pragma unroll
            for (int c = 0; c < DC; c++) f[c] = vfrag(p, c);
        };
#pragma unroll
        for (int p = 0; p < PFV && p < NPT; p++) load_v(p, vf[p]);
#pragma unroll
        for (int p = 0; p < NPT; p++) {
            if (PFV && p + PFV < NPT) load_v(p + PFV, vf[(p + PFV) % (PFV + 1)]);
            f16x8 ph, pl;
            split(2 * p, ph, pl);
#pragma unroll
            for (int c = 0; c < DC; c++) {
                const f16x8 v = PFV ? vf[p % (PFV + 1)][c] : vfrag(p, c);   // without prefetch, one chunk at a time
                O[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v, ph, O[c], 0, 0, 0);
                O[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v, pl, O[c], 0, 0, 0);
            }
            S1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, ph, S1, 0, 0, 0);
            S1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, pl, S1, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);  // the fragment reads stay PFV pairs ahead
        }
        // features 4 DC lg .. 4 DC lg + 4 DC - 1 of query q0 + l16, divided by its row sum
        const float inv = 1.f / S1[0];
        const int qi = q0 + l16;
        if (qi < S) {
            const int64_t ro = (int64_t)b * a.os[3] + (int64_t)h * a.os[2] + (int64_t)qi * a.os[1];
            const int d0 = 4 * DC * lg;
            if (vec) {
#pragma unroll
                for (int c = 0; c < DC; c++) {
                    const f32x4 v = O[c] * inv;
                    if (a.o16)
                        *(f16x4*)(a.o16 + ro + d0 + 4 * c) = f16x4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
                    else
                        *(f32x4*)(a.o + ro + d0 + 4 * c) = v;
                }
            } else {
#pragma unroll
                for (int c = 0; c < DC; c++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int64_t e = ro + (int64_t)(d0 + 4 * c + r) * a.os[0];
                        if (a.o16) a.o16[e] = (_Float16)(O[c][r] * inv);
                        else a.o[e] = O[c][r] * inv;
                    }
            }
        }
    }
}

template <int DC, int KT>
void launch_head_t(const FaArgs& a, hipStream_t s) {
    const int nqt = (a.S + 15) / 16;
    const int64_t heads = (int64_t)a.H * a.B;
    // A head's query tiles spread over qs workgroups (each restaging the head's K/V) while the
    // heads alone give fewer than ~256 workgroups, keeping >= 6 waves per workgroup (staging
    // with fewer threads costs more than the finer split gains); every query's arithmetic is
    // the same either way. Measured at S = 257, 16 heads (cfg4 shapes, fp32 q/k/v): one image
    // 10.8 us (3 workgroups per head) against ~15 us with 2 waves in 9 and 18 us unsplit;
    // 8 images 14.2 against 18.0 us unsplit (2 per head, 9 waves); at 16 images (256 heads)
    // splitting costs (29.4 against 21.4 us), so qs = 1 there, ~2 query tiles per wave.
    // With the staging down to one round trip, four waves per workgroup (one per SIMD) win
    // where that finer split still gives every workgroup its own CU: S = 257, one image 7.4
    // against 8.5 us (3 workgroups of 6 waves), two images 7.6 against 8.7; 3, 5, 6 or 9 waves
    // 8.4-9.8 us at one image.
    int qs = (int)std::max<int64_t>(1, std::min<int64_t>(256 / std::max<int64_t>(heads, 1), (nqt + 5) / 6));
    const bool tail = a.S > 16 * (KT - 1);
    const int maxw = a.q16 ? (tail ? kHeadWaves<DC, KT, true, true> : kHeadWaves<DC, KT, true, false>)
                           : (tail ? kHeadWaves<DC, KT, false, true> : kHeadWaves<DC, KT, false, false>);
    int nw = std::min(maxw, std::max(1, qs > 1 ? (nqt + qs - 1) / qs : (nqt + 1) / 2));
    if (qs > 1 && maxw >= 4 && heads * ((nqt + 3) / 4) <= 256) nw = 4;
    if (qs > 1) qs = (nqt + nw - 1) / nw;
    const dim3 grid((unsigned)a.H, (unsigned)a.B, (unsigned)qs), block((unsigned)(64 * nw));
    // fp16 rows 16-byte aligned (the pointers are, head_ok): one load per 8 elements
    const bool a16 = a.st[1] % 8 == 0 && a.st[2] % 8 == 0 && a.st[3] % 8 == 0;
    if (a.q16 && a16) {
        if (tail) hipLaunchKernelGGL((k_attn_head<DC, KT, true, true, true>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((k_attn_head<DC, KT, true, false, true>), grid, block, 0, s, a);
    } else if (a.q16) {
        if (tail) hipLaunchKernelGGL((k_attn_head<DC, KT, true, true, false>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((k_attn_head<DC, KT, true, false, false>), grid, block, 0, s, a);
    } else {
        if (tail) hipLaunchKernelGGL((k_attn_head<DC, KT, false, true, false>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((k_attn_head<DC, KT, false, false, false>), grid, block, 0, s, a);
    }
}

template <int DC>
hipError_t launch_head(const FaArgs& a, hipStream_t s) {
    const int kt = (a.S + 15) / 16;
    if (kt <= 4) launch_head_t<DC, 4>(a, s);
    else if (kt <= 8) launch_head_t<DC, 8>(a, s);
    else if (kt <= 17) launch_head_t<DC, 17>(a, s);
    else if (kt <= 24) launch_head_t<DC, 24>(a, s);
    else launch_head_t<DC, 32>(a, s);
    return hipGetLastError();
}

// Long sequences (S > 272): online softmax over 64-key chunks, a wave holding QT 16-query tiles
// (each K / V fragment read from LDS serves QT tiles) and QG waves side by side along the queries.
// The keys go to KS * SEQ groups, group g taking every KS * SEQ-th chunk from the g-th on: KS groups of
// QG waves side by side, or SEQ groups one after the other in the same waves; the groups' (max,
// sum, O) are merged through LDS, in both cases alike. The VALU is the busiest unit (4.5 operations per
// score, one of them a quarter-rate exp2), so:
//  * the products, the row sums from the matrix unit and the transposed P . V are k_attn_head's,
//    as is P = hi + lo but for the rounding: both parts to nearest (v_cvt_pk_f16_f32, as fast as the
//    truncating form), at most 1.2e-7 of P lost against 3.6e-7; one 32-deep MFMA covers 32 features /
//    keys, whose order inside a fragment is free as long as both operands share it, so K rows
//    (padded with zeros to 32) and V^T rows (keys permuted within 32: position 8 lg + 4 (t % 2) + r
//    holds key 16 (t % 2) + 4 lg + r) are read with one conflict-free 16-byte read per fragment;
//  * the softmax reference of a query only has to be near its maximum: it starts 7 below the
//    first chunk's (log2 units), so p = 2^7 there, and moves (and O is rescaled) only when a score
//    of the wave exceeds it by more than 15, a wave-uniform branch almost never taken after the
//    first chunk. p <= 2^15 is inside fp16, and the larger p keeps the lo parts of the small ones
//    above the fp16 subnormals: with p <= 1, a row whose maximum stands 8 above its other scores
//    lost 4.5e-6 of its weights' sum to them;
//  * P . V and the row sums of a chunk start from zero and are added to O in fp32: the matrix
//    unit's own accumulation over the whole sequence had twice the error against 64 bits
//    (6.4e-7 against 3.3e-7 at S = 4097) for 6% less time;
//  * keys past S are masked in the last chunk only.
// K and V arrive as fp32: each workgroup loads the next chunk into registers (16-byte loads)
// while it computes the current one, rounds once and stores fp16 to the other LDS buffer, V as
// 4 x 4 blocks transposed in registers: one barrier per chunk.
// A sequence of 2^k + 1 tokens (the class token) leaves one query past the whole blocks: a last
// block with a single wave's queries is split over the keys instead (NV parts, each wave reading its
// own fragments from memory without the staging or its barriers).
// Measured (16 heads, D = 48, one image) against the kernel for any strides: S = 1025 114 -> 18 us,
// S = 4097 549 -> 122 us (VALU busy 62 us of it, the matrix unit 42), error against
// 64 bits 3.8e-7 -> 2.1e-7 and 6.6e-7 -> 2.8e-7.
constexpr int LKT = 64;                  // keys per chunk
constexpr int LVLD = LKT + 8;            // V^T row stride (halves): 9 16-byte slots
template <int DC>
constexpr int kLongKLD = DC <= 2 ? 40 : 72;   // K row stride (halves): 32 or 64 features + 8

// queries [body, S) are a split block's: at most `tail` of them, past a multiple of `gran`
struct LongCut {
    int gran, tail;
};
template <int QG, int QT, int KS, int SEQ>
constexpr LongCut kLongCut = KS * SEQ == 1 ? LongCut{16 * QT * QG, 16 * QT} : LongCut{64, 16};

template <int DC, int QG, int QT, int KS, int SEQ, bool I16>
__global__ __launch_bounds__(64 * QG * KS) void k_attn_long(FaArgs a, int nblk, int body, int heads) {
    constexpr int D = 16 * DC, KLD = kLongKLD<DC>, KC = (DC + 1) / 2, NW = QG * KS;
    constexpr int G = KS * SEQ;          // key groups
    constexpr int NV = G == 1 ? NW : 8;  // parts a split block's keys are taken in
    static_assert((KS == 1 || SEQ == 1) && NV % NW == 0, "");
    constexpr int GT = 64 * QG;          // threads per key group
    constexpr int KV4 = LKT * D / 4;     // 16-byte pieces of a chunk's K
    constexpr int UK = (KV4 + GT - 1) / GT, VB = LKT / 4 * (D / 4), UV = (VB + GT - 1) / GT;
    constexpr int CH = LKT * KLD + D * LVLD;     // halves per chunk buffer
    constexpr int MR = QT * (4 * DC + 2);   // floats a lane hands over in the merge
    constexpr int STAGE = 2 * KS * CH * 2, MERGE = NV * 64 * MR * 4, STASH = SEQ > 1 ? NW * 64 * MR * 4 : 0;
    __shared__ __attribute__((aligned(16))) char lds[STAGE + STASH > MERGE ? STAGE + STASH : MERGE];

    const int S = a.S;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wave / QG, qg = wave - kg * QG, gt = tid - kg * GT;
    const int l16 = lane & 15, lg = lane >> 4;
    // each XCD takes contiguous runs of (head, block), so that its L2 holds few heads' K and V; then
    // the heads' split blocks
    const int nf = nblk * heads;
    const bool split = (int)blockIdx.x >= nf;
    const int lid = split ? (int)blockIdx.x - nf : xcd_remap(blockIdx.x, nf);
    const int hb = split ? lid : lid / nblk, qb = lid - hb * nblk;
    const int h = hb % a.H, b = hb / a.H;
    const int64_t base = (int64_t)b * a.st[3] + (int64_t)h * a.st[2];
    const int q0 = split ? body : (qb * QG + qg) * 16 * QT;
    const bool active = q0 < (split ? S : body);

    // staging: this key group's chunk c, K pieces (key, 4 features) and V blocks (4 keys x 4
    // features; lanes run over 4 feature blocks, then key blocks: 64-byte row segments). Buffer
    // loads over the head's rows: loop-invariant lane offsets, the chunk in the scalar offset,
    // rows past S outside the range (zeros; the check takes lane and scalar offset together, also
    // where the scalar one alone is past the range: measured), so the loop spends no vector
    // instruction on addresses or bounds.
    constexpr int EB = I16 ? 2 : 4;      // bytes per element
    typedef std::conditional_t<I16, f16x4, f32x4> E4;
    const uint32_t ext = (uint32_t)(((int64_t)(S - 1) * a.st[1] + D) * EB);
    auto rsrc = [&](const float* p, const _Float16* p16) {
        void* q = I16 ? (void*)(p16 + base) : (void*)(p + base);
        return __builtin_amdgcn_make_buffer_rsrc(q, (short)0, (int)ext, 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t rsk = rsrc(a.k, a.k16), rsv = rsrc(a.v, a.v16);
    auto ld4 = [](__amdgpu_buffer_rsrc_t r, uint32_t vo, uint32_t so) -> E4 {
        if constexpr (I16) return __builtin_bit_cast(E4, __builtin_amdgcn_raw_buffer_load_b64(r, (int)vo, (int)so, 0));
        else return __builtin_bit_cast(E4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)vo, (int)so, 0));
    };
    auto h4 = [](E4 v) { return f16x4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]}; };
    const uint32_t rowb = (uint32_t)a.st[1] * EB;
    uint32_t ok[UK], ov[UV], sk[UK], sv[UV];     // byte offsets in the source, half offsets in LDS
#pragma unroll
    for (int u = 0; u < UK; u++) {
        const int i = gt + GT * u, key = i / (D / 4), d = 4 * (i - key * (D / 4));
        ok[u] = key * rowb + EB * d;
        sk[u] = key * KLD + d;
    }
#pragma unroll
    for (int u = 0; u < UV; u++) {
        const int i = gt + GT * u, kb = (i >> 2) & 15, db = (i & 3) + 4 * (i >> 6);
        ov[u] = 4 * kb * rowb + EB * 4 * db;
        sv[u] = LKT * KLD + 4 * db * LVLD + 32 * (kb >> 3) + 8 * (kb & 3) + 4 * ((kb >> 2) & 1);
    }
    E4 rk[UK], rv[UV][4];
    auto load = [&](int c) {
        const uint32_t so = (uint32_t)c * LKT * rowb;
#pragma unroll
        for (int u = 0; u < UK; u++)
            if (KV4 % GT == 0 || gt + GT * u < KV4)
                rk[u] = ld4(rsk, ok[u], so);
#pragma unroll
        for (int u = 0; u < UV; u++)
            if (VB % GT == 0 || gt + GT * u < VB)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    rv[u][j] = ld4(rsv, ov[u], so + j * rowb);
    };
    auto store = [&](int buf) {
        _Float16* B = (_Float16*)lds + (buf * KS + kg) * CH;
#pragma unroll
        for (int u = 0; u < UK; u++)
            if (KV4 % GT == 0 || gt + GT * u < KV4)
                *(f16x4*)(B + sk[u]) = h4(rk[u]);
#pragma unroll
        for (int u = 0; u < UV; u++)
            if (VB % GT == 0 || gt + GT * u < VB)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    *(f16x4*)(B + sv[u] + e * LVLD) =
                        f16x4{(_Float16)rv[u][0][e], (_Float16)rv[u][1][e], (_Float16)rv[u][2][e], (_Float16)rv[u][3][e]};
    };

    // Q as the B operand: lane = query 16 qt + l16, features 32 c + 8 lg + j (zeros past D)
    f16x8 qf[QT][KC];
#pragma unroll
    for (int qt = 0; qt < QT; qt++) {
        const int qi = min(q0 + 16 * qt + l16, S - 1);
        const int64_t qrow = base + (int64_t)qi * a.st[1];
#pragma unroll
        for (int c = 0; c < KC; c++) {
            const int d = 32 * c + 8 * lg;
            qf[qt][c] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
            if (d < D) qf[qt][c] = load_h8<I16, false>(a.q, a.q16, qrow + d);
        }
    }
    // the features between D and the padded width meet zeros of Q: they only have to be finite (a split
    // block keeps its parts' states there instead)
    if (D % 32 && !split) {
        for (int i = tid; i < 2 * KS * LKT; i += 64 * NW)
#pragma unroll
            for (int e = 0; e < 2; e++)
                *(f16x8*)((_Float16*)lds + (i / LKT) * CH + (i % LKT) * KLD + D + 8 * e) = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }

    const float scale2 = a.scale * 1.4426950408889634f;
    const float m1 = opaque_neg_one();
    const f16x8 ones = {1, 1, 1, 1, 1, 1, 1, 1};
    // softmax reference (scaled, log2 units), O^T (register r of chunk c: feature 16 c + 4 lg + r of
    // query l16) and the row sums (every register of S1)
    float mref[QT], S1[QT];
    f32x4 O[QT][DC];
    auto reset = [&] {
#pragma unroll
        for (int qt = 0; qt < QT; qt++) {
            mref[qt] = -1e30f;
            S1[qt] = 0.f;
#pragma unroll
            for (int c = 0; c < DC; c++) O[qt][c] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    };
    reset();
    // this state in LDS ([MR][64 lanes] per part), and two parts' merged: the earlier part's is this
    // one (LATER: the one in LDS)
    constexpr int MQ = 4 * DC + 2;
    auto put = [&](float* w) {
        w += lane;
#pragma unroll
        for (int qt = 0; qt < QT; qt++) {
            w[qt * MQ * 64] = mref[qt];
            w[(qt * MQ + 1) * 64] = S1[qt];
#pragma unroll
            for (int c = 0; c < DC; c++)
#pragma unroll
                for (int r = 0; r < 4; r++) w[(qt * MQ + 2 + 4 * c + r) * 64] = O[qt][c][r];
        }
    };
    auto merge = [&](const float* w, auto later) {
        w += lane;
#pragma unroll
        for (int qt = 0; qt < QT; qt++) {
            const float mo = w[qt * MQ * 64], mn = fmaxf(mref[qt], mo);
            const float al = __builtin_amdgcn_exp2f(mref[qt] - mn), be = __builtin_amdgcn_exp2f(mo - mn);
            auto add = [&](float x, float y) { return decltype(later)::value ? fmaf(x, al, y * be) : fmaf(y, be, x * al); };
            mref[qt] = mn;
            S1[qt] = add(S1[qt], w[(qt * MQ + 1) * 64]);
#pragma unroll
            for (int c = 0; c < DC; c++)
#pragma unroll
                for (int r = 0; r < 4; r++) O[qt][c][r] = add(O[qt][c][r], w[(qt * MQ + 2 + 4 * c + r) * 64]);
        }
    };

    // NT key tiles from key0 on: kfrag(t, i) is the K fragment of tile t, features 32 i + 8 lg + j;
    // vfrag(p, c) the V^T fragment of tiles 2p, 2p + 1, feature 16 c + l16. (MASK is a property
    // of the call, not a branch between the score MFMAs and their use: around such a branch the
    // compiler left out the wait for the MFMA results.)
    auto compute = [&](auto ntc, auto mask, int key0, auto kfrag, auto vfrag) {
        constexpr int NT = decltype(ntc)::value;
        f32x4 sc[QT][NT];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            f16x8 kf[KC];
#pragma unroll
            for (int i = 0; i < KC; i++) kf[i] = kfrag(t, i);
#pragma unroll
            for (int qt = 0; qt < QT; qt++) {
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < KC; i++) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[i], qf[qt][i], acc, 0, 0, 0);
                sc[qt][t] = acc;
            }
        }
        if (decltype(mask)::value) {             // keys past S
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (key0 + 16 * t + 4 * lg + r >= S)
#pragma unroll
                        for (int qt = 0; qt < QT; qt++) sc[qt][t][r] = -INFINITY;
        }
        float mx[QT];
        bool up[QT], any = false;        // (per query tile: a tile's sums do not depend on the wave's other one)
#pragma unroll
        for (int qt = 0; qt < QT; qt++) {
            float v = -INFINITY;
#pragma unroll
            for (int t = 0; t < NT; t++) {
                v = fmaxf(fmaxf(v, sc[qt][t][0]), sc[qt][t][1]);
                v = fmaxf(fmaxf(v, sc[qt][t][2]), sc[qt][t][3]);
            }
            mx[qt] = v * scale2;
            up[qt] = __any(mx[qt] > mref[qt] + 15.f);
            any = any || up[qt];
        }
        if (any) {
#pragma unroll
            for (int qt = 0; qt < QT; qt++) {
                float v = up[qt] ? fmaxf(mx[qt] - 7.f, mref[qt]) : mref[qt];
                v = fmaxf(v, __shfl_xor(v, 16));
                v = fmaxf(v, __shfl_xor(v, 32));
                const float al = __builtin_amdgcn_exp2f(mref[qt] - v);
                mref[qt] = v;
                S1[qt] *= al;
#pragma unroll
                for (int cc = 0; cc < DC; cc++) O[qt][cc] *= al;
            }
        }
        f32x4 sc1[QT], oc[QT][DC];
#pragma unroll
        for (int qt = 0; qt < QT; qt++) {
            sc1[qt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int cc = 0; cc < DC; cc++) oc[qt][cc] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int p = 0; p < NT / 2; p++) {
            f16x8 vf[DC];
#pragma unroll
            for (int cc = 0; cc < DC; cc++) vf[cc] = vfrag(p, cc);
#pragma unroll
            for (int qt = 0; qt < QT; qt++) {
                float e[8];
#pragma unroll
                for (int j = 0; j < 8; j++)
                    e[j] = __builtin_amdgcn_exp2f(fmaf(sc[qt][2 * p + j / 4][j % 4], scale2, -mref[qt]));
                u32x4 hi, lo;
                auto u = [](auto v) { return __builtin_bit_cast(uint32_t, v); };
                auto rne = [](float a, float b) { return __builtin_convertvector(f32x2{a, b}, f16x2); };
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const f16x2 hh = rne(e[2 * j], e[2 * j + 1]);
                    hi[j] = u(hh);
                    lo[j] = u(rne(fmaf((float)hh[0], m1, e[2 * j]), fmaf((float)hh[1], m1, e[2 * j + 1])));
                }
                const f16x8 ph = __builtin_bit_cast(f16x8, hi), pl = __builtin_bit_cast(f16x8, lo);
#pragma unroll
                for (int cc = 0; cc < DC; cc++) {
                    oc[qt][cc] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[cc], pl, oc[qt][cc], 0, 0, 0);
                    oc[qt][cc] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[cc], ph, oc[qt][cc], 0, 0, 0);
                }
                sc1[qt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, pl, sc1[qt], 0, 0, 0);
                sc1[qt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, ph, sc1[qt], 0, 0, 0);
            }
        }
#pragma unroll
        for (int qt = 0; qt < QT; qt++) {
            S1[qt] += sc1[qt][0];
#pragma unroll
            for (int cc = 0; cc < DC; cc++) O[qt][cc] += oc[qt][cc];
        }
    };

    if (!split) {
        // chunks it * KS + kg; the last round, which holds the sequence's last chunk, masks
        const int nch = (S + LKT - 1) / LKT, nit = (nch + KS - 1) / KS;
        auto step = [&](auto mask, int buf, int c) {
            const _Float16* Ks = (const _Float16*)lds + (buf * KS + kg) * CH;
            const _Float16* Vt = Ks + LKT * KLD;
            compute(std::integral_constant<int, LKT / 16>{}, mask, c * LKT,
                    [&](int t, int i) { return *(const f16x8*)&Ks[(16 * t + l16) * KLD + 32 * i + 8 * lg]; },
                    [&](int p, int cc) { return *(const f16x8*)&Vt[(16 * cc + l16) * LVLD + 32 * p + 8 * lg]; });
        };
        load(kg);
        store(0);
        if constexpr (SEQ == 1) {
            for (int it = 0; it + 1 < nit; it++) {
                __syncthreads();         // this buffer is filled, the other one no longer read
                // (past the last chunk its values are stored again, never read)
                if (KS == 1 || (it + 1) * KS + kg < nch) load((it + 1) * KS + kg);
                if (active) step(std::false_type{}, it & 1, it * KS + kg);
                store((it + 1) & 1);
            }
            __syncthreads();
            const int c = (nit - 1) * KS + kg;
            if (active && c < nch) step(std::true_type{}, (nit - 1) & 1, c);
        } else {
            // the key groups one after the other, the first one's state kept in LDS meanwhile
            float* stash = (float*)(lds + STAGE) + wave * MR * 64;
            int buf = 0;
#pragma unroll 1
            for (int g = 0; g < SEQ; g++) {
                int c = g;
                for (; c + SEQ < nch; c += SEQ) {
                    __syncthreads();
                    load(c + SEQ);
                    if (active) step(std::false_type{}, buf, c);
                    buf ^= 1;
                    store(buf);
                }
                __syncthreads();
                if (g + 1 < SEQ) load(g + 1);
                if (active) step(std::true_type{}, buf, c);
                if (g + 1 < SEQ) {
                    buf ^= 1;
                    store(buf);
                    put(stash);
                    reset();
                }
            }
            merge(stash, std::true_type{});
        }
    } else {
        // part v takes 32-key groups v, v + NV, ..., each wave's fragments straight from memory (rows
        // past S and features past D outside the buffer range: zeros). Holding the next group's
        // values as well would cost the registers that let this block share a CU with two whole
        // ones
        const int ng = (S + 31) / 32;
        E4 kr[2][KC][2];
        std::conditional_t<I16, _Float16, float> vr[DC][8];
        auto fetch = [&](int g) {
            const uint32_t so = 32u * g * rowb;
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int i = 0; i < KC; i++) {
                    const int d = 32 * i + 8 * lg;
                    const uint32_t o = d < D ? (16 * t + l16) * rowb + EB * d : 0x80000000u;
                    kr[t][i][0] = ld4(rsk, o, so);
                    kr[t][i][1] = ld4(rsk, o + 4 * EB, so);
                }
#pragma unroll
            for (int cc = 0; cc < DC; cc++)
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const int o = (int)((16 * (j >> 2) + 4 * lg + (j & 3)) * rowb + EB * (16 * cc + l16));
                    if constexpr (I16)
                        vr[cc][j] = __builtin_bit_cast(_Float16, __builtin_amdgcn_raw_buffer_load_b16(rsv, o, (int)so, 0));
                    else
                        vr[cc][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsv, o, (int)so, 0));
                }
        };
#pragma unroll 1
        for (int v = wave; v < NV; v += NW) {
            for (int g = v; g < ng; g += NV) {
                fetch(g);
                f16x8 kf[2][KC], vf[DC];
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int i = 0; i < KC; i++)
#pragma unroll
                        for (int j = 0; j < 8; j++) kf[t][i][j] = (_Float16)kr[t][i][j >> 2][j & 3];
#pragma unroll
                for (int cc = 0; cc < DC; cc++)
#pragma unroll
                    for (int j = 0; j < 8; j++) vf[cc][j] = (_Float16)vr[cc][j];
                compute(std::integral_constant<int, 2>{}, std::true_type{}, 32 * g, [&](int t, int i) { return kf[t][i]; },
                        [&](int, int cc) { return vf[cc]; });
            }
            if (NV > NW) {
                put((float*)lds + v * MR * 64);
                reset();
            }
        }
    }

    // merge, in the order of the parts: the waves that share queries (the key groups; in a split block
    // all of them) hand their state to the first of them
    if (KS > 1 || split) {
        __syncthreads();
        float* mg = (float*)lds;         // [part][MR][64 lanes]
        const bool first = kg == 0 && (!split || qg == 0);
        if (!first && active && !(split && NV > NW)) put(mg + wave * MR * 64);
        __syncthreads();
        if (!first) return;
        // (NV > NW: part 0 merged into the empty state is itself: its scale is exp2(0), the other's exp2(-inf))
        const int step = split ? 1 : QG;
        for (int o = split && NV > NW ? 0 : wave + step; o < (split ? NV : NW); o += step) merge(mg + o * MR * 64, std::false_type{});
    }
    if (!active) return;
    const bool vec = a.os[0] == 1 && ((a.os[1] | a.os[2] | a.os[3]) & 3) == 0 &&
                     ((uintptr_t)(a.o16 ? (const void*)a.o16 : (const void*)a.o) & 15) == 0;
#pragma unroll
    for (int qt = 0; qt < QT; qt++) {
        const float inv = 1.f / S1[qt];
        const int qi = q0 + 16 * qt + l16;
        if (qi >= S) continue;
        const int64_t ro = (int64_t)b * a.os[3] + (int64_t)h * a.os[2] + (int64_t)qi * a.os[1];
#pragma unroll
        for (int c = 0; c < DC; c++) {
            const int d = 16 * c + 4 * lg;
            f32x4 v = O[qt][c] * inv;
            // (rounded to fp32 before the fp16 store rounds again: kept from fusing into one step)
            asm volatile("" : "+v"(v));
            if (vec) {
                if (a.o16)
                    *(f16x4*)(a.o16 + ro + d) = f16x4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
                else
                    *(f32x4*)(a.o + ro + d) = v;
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int64_t e = ro + (int64_t)(d + r) * a.os[0];
                    if (a.o16) a.o16[e] = (_Float16)v[r];
                    else a.o[e] = v[r];
                }
            }
        }
    }
}

template <int DC, int QG, int QT, int KS, int SEQ>
void launch_long_t(const FaArgs& a, hipStream_t s) {
    constexpr LongCut cut = kLongCut<QG, QT, KS, SEQ>;
    const int r = a.S % cut.gran, body = r && r <= cut.tail ? a.S - r : a.S;
    const int qb = 16 * QT * QG, nblk = (body + qb - 1) / qb, heads = a.H * a.B;
    const dim3 grid((unsigned)(heads * (nblk + (body < a.S ? 1 : 0)))), block(64 * QG * KS);
    if (a.q16) hipLaunchKernelGGL((k_attn_long<DC, QG, QT, KS, SEQ, true>), grid, block, 0, s, a, nblk, body, heads);
    else hipLaunchKernelGGL((k_attn_long<DC, QG, QT, KS, SEQ, false>), grid, block, 0, s, a, nblk, body, heads);
}

// From 200 128-query blocks per image (120 at D = 64, whose 64-query form holds 150 registers) 128
// queries per workgroup, each K / V fragment serving two query tiles, one key group. An image with fewer
// (up to ~1500 tokens) takes its keys in two groups, so that one image gives every CU a workgroup of
// eight waves: 64 queries and the groups side by side, or, in a call with many blocks, 128 queries and
// the groups one after the other, the same sums: an image's result does not depend on its batch.
// Measured, 16 heads, D = 48, fp32 q/k/v:
//  * one image, two groups side by side against 128 queries and one group: S = 600 10.0 / 15.4 us, 1025
//    18.0 / 23.3, 2049 48.9 / 45.3, 4097 156 / 124 (D = 64: S = 1500, 12 heads 36.9 / 33.3);
//  * a batch, side by side against one after the other: S = 600 x 3 16.7 / 17.6, 801 x 2 18.4 / 20.9, 1025 x
//    4 46.9 / 44.0, 1025 x 16 186 / 149; D = 64: 513 x 8 44.7 / 33.2. Side by side while its 64-query
//    blocks run in one round (two per CU; D = 64: one), or while the 128-query blocks' last round is so
//    empty that they take longer (a CU's round of two waves per SIMD: 1.5 times as long; 1300 x 3: 50 /
//    62). With one group instead, whose sums are others, a batch took up to 20% less (1025 x 4: 38.8): the
//    first group's state costs LDS and so one of three workgroups per CU.
template <int DC>
hipError_t launch_long(const FaArgs& a, hipStream_t s) {
    constexpr LongCut cut = kLongCut<4, 1, 2, 1>;
    const int64_t heads = (int64_t)a.H * a.B;
    const bool tail = a.S % cut.gran && a.S % cut.gran <= cut.tail;
    const int body = a.S - (tail ? cut.tail : 0);        // (rounded up to blocks: the queries of whole ones)
    const int64_t n64 = heads * ((body + 63) / 64), n128 = heads * ((body + 127) / 128);
    if ((int64_t)a.H * ((a.S + 127) / 128) >= (DC <= 3 ? 200 : 120))
        launch_long_t<DC, 4, 2, 1, 1>(a, s);
    else if (n64 + (tail ? heads : 0) <= (DC <= 3 ? 512 : 256) || 2 * ((n64 + 255) / 256) < 3 * ((n128 + 255) / 256))
        launch_long_t<DC, 4, 1, 2, 1>(a, s);
    else
        launch_long_t<DC, 4, 2, 1, 2>(a, s);
    return hipGetLastError();
}

// q/k/v whose rows are features in order, spaced at least a head apart, that the staging's 8- or
// 16-byte loads and 31-bit byte offsets can take; the launch's threads fit 32 bits
bool long_ok(const FaArgs& a, int D) {
    auto al = [](const void* p) { return ((uintptr_t)p & 15u) == 0; };
    const bool ptrs = a.q16 ? al(a.q16) && al(a.k16) && al(a.v16) : al(a.q) && al(a.k) && al(a.v);
    return D % 16 == 0 && ptrs && a.st[0] == 1 && a.st[1] >= D && ((int64_t)a.S + 512) * a.st[1] * 4 < (1ll << 31) &&
           a.st[1] % 4 == 0 && a.st[2] % 4 == 0 && a.st[3] % 4 == 0 && a.scale > 0.f &&
           (int64_t)a.H * a.B * (a.S / 64 + 2) * 512 < (1ll << 32);
}

bool head_ok(const FaArgs& a, int D) {
    auto al = [](const void* p) { return ((uintptr_t)p & 15u) == 0; };
    const bool ptrs = a.q16 ? al(a.q16) && al(a.k16) && al(a.v16) : al(a.q) && al(a.k) && al(a.v);
    return a.S <= 512 && a.st[0] == 1 && a.st[1] % 4 == 0 && a.st[2] % 4 == 0 && a.st[3] % 4 == 0 &&
           D % 16 == 0 && ptrs && a.H <= 65535 && a.B <= 65535 && a.scale > 0.f;
}

}  // namespace

hipError_t launch_flash_attn_f16kv(const FaArgs& a, int D, hipStream_t s) {
    if (a.S <= 0 || a.H <= 0 || a.B <= 0) return hipSuccess;
    const bool head = head_ok(a, D);
    if (a.q16 && !head) return hipErrorInvalidValue;   // fp16 inputs: S <= 512 with aligned rows only
    // The whole-head kernel up to 17 key tiles (S = 272, one 256-token image and its class token:
    // 16 images 13.0 against 14.6 us for the long kernel, one image 6.3 against 6.6, fp16 q/k/v);
    // beyond, its score registers leave one or two waves per SIMD and the long kernel wins (one
    // image, S = 512: 10.2 against 8.0 us; 4 images, S = 400: 26.2 against 11.8). Both input
    // types take the same kernel, so their results stay equal.
    if ((!head || a.S > 272) && long_ok(a, D)) {
        switch (D) {
            case 16: return launch_long<1>(a, s);
            case 32: return launch_long<2>(a, s);
            case 48: return launch_long<3>(a, s);
            case 64: return launch_long<4>(a, s);
            default: break;
        }
    }
    if (head) {
        switch (D) {
            case 16: return launch_head<1>(a, s);
            case 32: return launch_head<2>(a, s);
            case 48: return launch_head<3>(a, s);
            case 64: return launch_head<4>(a, s);
            default: break;
        }
    }
    // any strides
    const dim3 grid((unsigned)((a.S + 63) / 64), (unsigned)a.H, (unsigned)a.B), block(256);
    switch (D) {
        case 16: hipLaunchKernelGGL(k_flash_attn_f16kv<1>, grid, block, 0, s, a); break;
        case 32: hipLaunchKernelGGL(k_flash_attn_f16kv<2>, grid, block, 0, s, a); break;
        case 48: hipLaunchKernelGGL(k_flash_attn_f16kv<3>, grid, block, 0, s, a); break;
        case 64: hipLaunchKernelGGL(k_flash_attn_f16kv<4>, grid, block, 0, s, a); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace mgh
