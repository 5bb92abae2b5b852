// f32 products on the bf16 matrix cores (gfx950).
//
// An f32 value is the exact sum of three bf16 pieces, v = p0 + p1 + p2 (8 significant bits each,
// rounded to nearest, so |p1| <= 2^-8 |v| and |p2| <= 2^-17 |v|). Of the nine piece products of
// a * b the six largest are summed; the others are at most 2^-24 of the product, 2^-27.5 in the mean
// square (Henry, Tang, Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations", ARITH 2019). A sum of products takes six bf16 multiply-adds per f32
// one, at sixteen times the rate: v_mfma_f32_16x16x32_bf16 runs 1.95 PFLOP/s on registers (random
// operands, eight chains, one wave per SIMD), i.e. 325 TFLOP/s of f32 products, against 137-142 for
// v_mfma_f32_16x16x4_f32, and unlike the f32 form it runs beside vector work.
//
// A lane holds four channels of an operand as six registers [p1 x4 | p0 x4 | p2 x4]: its first
// four (`lo`) are the pieces (p1, p0), its last four (`hi`) the pieces (p0, p2), each the eight K
// slots of one 16x16x32 MFMA. With A = (a1, a0, a2) and B = (b1, b0, b2) the six products are
//   lo . lo = a1 b1 + a0 b0,   lo . hi = a1 b0 + a0 b2,   hi . lo = a0 b1 + a2 b0,
// so one MFMA triple covers 16 channels of K and the packing stays 16 channels per chunk.
//
// The first goes to one accumulator, the two small ones to another, added once at the end: the
// matrix core rounds its accumulator once per 8 products, so the full-size sum is rounded K / 4
// times where the f32 MFMA rounds it K times (K = 1152, against 64-bit sums: 3e-7 relative
// instead of 4-6e-7).
//
// From 2^15 on p0 is cut off instead of rounded, so that p1 has the value's sign: where a0 b0 overflows,
// a1 b1, which shares its accumulator, can then only overflow to the same infinity (it overflows only if
// both operands are that large). FLT_MAX's p0 is finite for the same reason. An infinity or NaN is p0,
// with p1 = 0 and p2 NaN: a0 b0 goes to infinity or NaN as the f32 product does, and the full-size sum
// with it, while the small products, which zero pieces turn into NaN, no longer count (split_sum).
// Values below 2^-110 lose low bits (the pieces become subnormal). A product within 2^-7 of overflow may
// overflow: its a0 b0 can be that much larger.
#pragma once

#include <cfloat>

#include "mfma.h"

namespace zjai {

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// From here on a value's p0 is cut off instead of rounded.
constexpr float SPLIT_CUT = 0x1p15f;

struct SplitFrag {
    u32x4 lo;  // p1 of channels 0..3, p0 of channels 0..3
    u32x2 hi;  // p2 of channels 0..3
};

__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
    bf16x2 r;
    r[0] = (__bf16)a;
    r[1] = (__bf16)b;
    return __builtin_bit_cast(unsigned, r);
}

// What rounds to v's p0 (`fin`: v is finite).
__device__ __forceinline__ float split_p0(float v, bool fin) {
    const float cut = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, v) & 0xffff0000u);
    return __builtin_fabsf(v) < SPLIT_CUT ? v : fin ? cut : v;
}

// ORDINARY: all four values are finite and below SPLIT_CUT (the same pieces without a test).
template <bool ORDINARY = false>
__device__ __forceinline__ SplitFrag split_f32(f32x4 v) {
    SplitFrag f;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const float x = v[2 * h], y = v[2 * h + 1];
        const bool fx = ORDINARY || __builtin_fabsf(x) <= FLT_MAX, fy = ORDINARY || __builtin_fabsf(y) <= FLT_MAX;
        const unsigned p0 = ORDINARY ? pack_bf16(x, y) : pack_bf16(split_p0(x, fx), split_p0(y, fy));
        const float rx = x - __builtin_bit_cast(float, p0 << 16);
        const float ry = y - __builtin_bit_cast(float, p0 & 0xffff0000u);
        const unsigned p1 = pack_bf16(fx ? rx : 0.0f, fy ? ry : 0.0f);
        f.lo[h] = p1;
        f.lo[2 + h] = p0;
        f.hi[h] = pack_bf16(rx - __builtin_bit_cast(float, p1 << 16), ry - __builtin_bit_cast(float, p1 & 0xffff0000u));
    }
    return f;
}

// store(i, split_f32(v[i])) for each of a lane's N vectors: the maximum over them (NaN if one is) costs
// half an instruction a value, the tests that it spares a wave of ordinary values five of their eleven.
template <int N, typename F>
__device__ __forceinline__ void split_each(const f32x4 (&v)[N], F store) {
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) m = __builtin_elementwise_maximum(m, __builtin_fabsf(v[i][k]));
    if (__builtin_amdgcn_ballot_w64(!(m < SPLIT_CUT)) == 0) {
#pragma unroll
        for (int i = 0; i < N; ++i) store(i, split_f32<true>(v[i]));
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) store(i, split_f32(v[i]));
    }
}

// big += lo . lo, small += the other two MFMAs (16 channels of K).
__device__ __forceinline__ f32x4 mfma_bf16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ u32x4 split_hi(const SplitFrag& f) { return u32x4{f.lo[2], f.lo[3], f.hi[0], f.hi[1]}; }
__device__ __forceinline__ void mma_split(f32x4& big, f32x4& small, const SplitFrag& a, const SplitFrag& b) {
    small = mfma_bf16(a.lo, split_hi(b), small);
    big = mfma_bf16(a.lo, b.lo, big);
    small = mfma_bf16(split_hi(a), b.lo, small);
}

// mma_split for N accumulator pairs sharing A, one MFMA of the triple at a time over all of them.
template <int N>
__device__ __forceinline__ void mma_split_rows(f32x4 (&big)[N], f32x4 (&small)[N], const SplitFrag& a, const SplitFrag (&b)[N]) {
    const u32x4 ahi = split_hi(a);
#pragma unroll
    for (int r = 0; r < N; ++r) small[r] = mfma_bf16(a.lo, split_hi(b[r]), small[r]);
#pragma unroll
    for (int r = 0; r < N; ++r) big[r] = mfma_bf16(a.lo, b[r].lo, big[r]);
#pragma unroll
    for (int r = 0; r < N; ++r) small[r] = mfma_bf16(ahi, b[r].lo, small[r]);
}

// The sum of a pair of accumulators, the small one made finite: where the full-size sum is infinite or
// NaN, which it then stays, the small products may be NaN or have overflowed to the other sign. (The
// median of a NaN and two numbers is the smaller number.)
__device__ __forceinline__ f32x4 split_sum(f32x4 big, f32x4 small) {
#pragma unroll
    for (int i = 0; i < 4; ++i) small[i] = __builtin_amdgcn_fmed3f(small[i], -FLT_MAX, FLT_MAX);
    return big + small;
}

// 1x1 layers keep one accumulator: the small products of every two K chunks (32 channels; the last
// chunk of an odd number by itself) are summed from zero and then added to it, which leaves
// registers for the fused transformer blocks and rounds the full-size sum 9 times per 32 products.
//
// The MFMAs are inline assembly, accumulators in place: with a fresh small sum every 32 channels
// the compiler renames the chains a few instructions apart. It does not know what the block holds,
// so the block carries its own wait states: two before (an operand written by vector code just
// before) and eight after (results read or overwritten by vector code), as the compiler puts them
// around the builtin.
#define ZJAI_MF "v_mfma_f32_16x16x32_bf16 "
#define ZJAI_WAIT "s_nop 7"
__device__ __forceinline__ void mma_split32_2(f32x4& c0, f32x4& c1, const SplitFrag& a0, const SplitFrag& a1,
                                              const SplitFrag& b00, const SplitFrag& b01, const SplitFrag& b10,
                                              const SplitFrag& b11) {
    f32x4 s0, s1;
    asm("s_nop 1\n\t"
        ZJAI_MF "%2, %4, %9, 0\n\t" ZJAI_MF "%0, %4, %8, %0\n\t" ZJAI_MF "%2, %5, %8, %2\n\t"
        ZJAI_MF "%3, %4, %13, 0\n\t" ZJAI_MF "%1, %4, %12, %1\n\t" ZJAI_MF "%3, %5, %12, %3\n\t"
        ZJAI_MF "%2, %6, %11, %2\n\t" ZJAI_MF "%0, %6, %10, %0\n\t" ZJAI_MF "%2, %7, %10, %2\n\t"
        ZJAI_MF "%3, %6, %15, %3\n\t" ZJAI_MF "%1, %6, %14, %1\n\t" ZJAI_MF "%3, %7, %14, %3\n\t" ZJAI_WAIT
        : "+v"(c0), "+v"(c1), "=&v"(s0), "=&v"(s1)
        : "v"(a0.lo), "v"(split_hi(a0)), "v"(a1.lo), "v"(split_hi(a1)), "v"(b00.lo), "v"(split_hi(b00)), "v"(b01.lo),
          "v"(split_hi(b01)), "v"(b10.lo), "v"(split_hi(b10)), "v"(b11.lo), "v"(split_hi(b11)));
    c0 = split_sum(c0, s0);
    c1 = split_sum(c1, s1);
}
__device__ __forceinline__ void mma_split32_1(f32x4& c0, const SplitFrag& a0, const SplitFrag& a1, const SplitFrag& b0,
                                              const SplitFrag& b1) {
    f32x4 s0;
    asm("s_nop 1\n\t"
        ZJAI_MF "%1, %2, %7, 0\n\t" ZJAI_MF "%0, %2, %6, %0\n\t" ZJAI_MF "%1, %3, %6, %1\n\t"
        ZJAI_MF "%1, %4, %9, %1\n\t" ZJAI_MF "%0, %4, %8, %0\n\t" ZJAI_MF "%1, %5, %8, %1\n\t" ZJAI_WAIT
        : "+v"(c0), "=&v"(s0)
        : "v"(a0.lo), "v"(split_hi(a0)), "v"(a1.lo), "v"(split_hi(a1)), "v"(b0.lo), "v"(split_hi(b0)), "v"(b1.lo),
          "v"(split_hi(b1)));
    c0 = split_sum(c0, s0);
}
__device__ __forceinline__ void mma_split16_1(f32x4& c0, const SplitFrag& a0, const SplitFrag& b0) {
    f32x4 s0;
    asm("s_nop 1\n\t"
        ZJAI_MF "%1, %2, %5, 0\n\t" ZJAI_MF "%0, %2, %4, %0\n\t" ZJAI_MF "%1, %3, %4, %1\n\t" ZJAI_WAIT
        : "+v"(c0), "=&v"(s0)
        : "v"(a0.lo), "v"(split_hi(a0)), "v"(b0.lo), "v"(split_hi(b0)));
    c0 = split_sum(c0, s0);
}
// N accumulators sharing A; chunk 1 is there only if `two` (uniform).
template <int N>
__device__ __forceinline__ void mma_split32(f32x4 (&acc)[N], const SplitFrag& a0, const SplitFrag& a1,
                                            const SplitFrag (&b0)[N], const SplitFrag (&b1)[N], bool two) {
    if (two) {
#pragma unroll
        for (int r = 0; r + 1 < N; r += 2) mma_split32_2(acc[r], acc[r + 1], a0, a1, b0[r], b1[r], b0[r + 1], b1[r + 1]);
        if (N % 2) mma_split32_1(acc[N - 1], a0, a1, b0[N - 1], b1[N - 1]);
    } else {
#pragma unroll
        for (int r = 0; r < N; ++r) mma_split16_1(acc[r], a0, b0[r]);
    }
}

// A packed 16 x 16 weight block (16 outputs x 16 input channels) in split form: 96 16-byte
// units, the `lo` of the 64 lanes of an A fragment (lane = 16 * (channel / 4) + output), then
// their `hi`s.
constexpr int SPLIT_BLOCK_U = 96;

}  // namespace zjai
