// k_split_bf16.h — fp32 products on the bf16 matrix unit: a value is split into three bf16 parts,
// x = hi + mid + lo, each rounded to nearest, which hold all 24 bits of its significand. Six of
// the nine partial products are summed; the other three (mid * lo twice, lo * lo) come to at most
// 2^-24 of |x w| (|mid| <= 2^-8, |lo| <= 2^-17 of |x|; reached near x = w = 1 + 2^-8), half an ulp of
// the product, and to far less on average. The running sum is rounded six times per 32 values of k,
// where v_mfma_f32_16x16x4_f32 rounds it eight times: the result is as close to the exact sum
// (measured: closer), at 6 x 16 against 8 x 32 cycles per 16 x 16 x 32 tile. (Splitting a number into
// parts of fewer bits so that their products are exact: T. J. Dekker, A floating-point technique for
// extending the available precision, Numer. Math. 18, 1971.)
//
// Range: bf16 has fp32's exponents, so the low parts of values under 2^-110 would be subnormal and lose
// bits (6e-5 of a value of 2^-120). Values are split times 2^16 and sums taken times 2^-32, which keeps
// every fp32 value's bits at one multiplication each (256 x 256 x 128 convolution 100 -> 101 us, 4112 x
// 768 -> 2025 head 89 -> 92); values from 2^112 and sums from 2^96 on become infinities instead, and
// their users redo sums that are not finite on the fp32 instruction.
#pragma once
#include "mgh_common.h"

namespace mgh {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32v2 __attribute__((ext_vector_type(2)));

constexpr float kSplitScale = 0x1p16f, kSplitUnscale = 0x1p-32f;

// eight values -> their three parts (packed pairs, element order kept)
__device__ __forceinline__ void split_bf16(const f32x4 a, const f32x4 b, u32x4& hi, u32x4& mid, u32x4& lo) {
    const float x[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
#pragma unroll
    for (int p = 0; p < 4; p++) {
        float u = x[2 * p] * kSplitScale, v = x[2 * p + 1] * kSplitScale;
        auto part = [&] {
            const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32v2{u, v}, bf16x2));
            u -= __builtin_bit_cast(float, h << 16);            // exact
            v -= __builtin_bit_cast(float, h & 0xFFFF0000u);
            return h;
        };
        hi[p] = part();
        mid[p] = part();
        lo[p] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32v2{u, v}, bf16x2));
    }
}

// LDS rows of 32 values of one part (64 bytes, four 16-byte slots): value slot s of row r sits in
// slot s ^ swz32(r). A 16-byte LDS access is served in groups of lanes 0-3, 12-15, 20-23, 24-27
// (then 4-7, 8-11, 16-19, 28-31, and the same from 32), so that distinct slots for 16 consecutive
// lanes do not suffice: this form is conflict-free for fragment reads (16 rows x 4 slots), for writes
// of one slot of consecutive rows and for writes of whole consecutive rows. ((r >> 2) & 3 was not:
// two-way conflicts on every fragment read, 42K of 218K cycles of the 256 x 256 x 128 convolution.)
__device__ __forceinline__ int swz32(int r) { return ((r >> 2) & 2) ^ ((r >> 4) & 1); }

// parts of a fragment (16 rows x 32 k: lane = row, 8 k)
struct Frag3 {
    bf16x8 h, m, l;
};

// acc[i] += the six products of I a-fragments with one b-fragment, smallest first; each product for
// all i in turn, so that consecutive MFMAs are independent
template <int I>
__device__ __forceinline__ void mfma_split(const Frag3 (&a)[I], const Frag3& b, f32x4 (&acc)[I]) {
    auto go = [&](bf16x8 Frag3::*pa, const bf16x8& vb) {
#pragma unroll
        for (int i = 0; i < I; i++) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i].*pa, vb, acc[i], 0, 0, 0);
    };
    go(&Frag3::l, b.h);
    go(&Frag3::h, b.l);
    go(&Frag3::m, b.m);
    go(&Frag3::m, b.h);
    go(&Frag3::h, b.m);
    go(&Frag3::h, b.h);
}
// the same for one a-fragment
__device__ __forceinline__ void mfma_split1(const Frag3& a, const Frag3& b, f32x4& acc) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.l, b.h, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, b.l, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.m, b.m, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.m, b.h, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, b.m, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, b.h, acc, 0, 0, 0);
}
// both with the five small products in accumulators of their own: the large ones are rounded
// once per 32 k
template <int I>
__device__ __forceinline__ void mfma_split(const Frag3 (&a)[I], const Frag3& b, f32x4 (&acc)[I], f32x4 (&rest)[I]) {
    auto go = [&](bf16x8 Frag3::*pa, const bf16x8& vb, f32x4(&s)[I]) {
#pragma unroll
        for (int i = 0; i < I; i++) s[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i].*pa, vb, s[i], 0, 0, 0);
    };
    go(&Frag3::h, b.h, acc);
    go(&Frag3::l, b.h, rest);
    go(&Frag3::h, b.l, rest);
    go(&Frag3::m, b.m, rest);
    go(&Frag3::m, b.h, rest);
    go(&Frag3::h, b.m, rest);
}
__device__ __forceinline__ void mfma_split1(const Frag3& a, const Frag3& b, f32x4& acc, f32x4& rest) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, b.h, acc, 0, 0, 0);
    rest = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.l, b.h, rest, 0, 0, 0);
    rest = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, b.l, rest, 0, 0, 0);
    rest = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.m, b.m, rest, 0, 0, 0);
    rest = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.m, b.h, rest, 0, 0, 0);
    rest = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, b.m, rest, 0, 0, 0);
}

// LDS hand-over inside a K step: this wave's LDS accesses are done, then the workgroup barrier; the
// global loads in flight (into registers) stay in flight, which __syncthreads() would wait for
__device__ __forceinline__ void lds_sync() {
    __builtin_amdgcn_s_waitcnt(0xC07F);          // lgkmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

}  // namespace mgh
