// ResAU as one kernel (src/model/synthesis.rs:24-74, `ResAu::forward`):
//   t = conv3x3_grouped(relu6(x)), 16 channels per group, no bias;
//   y = x * (1 + conv1x1(t)), no bias (the gate of src/nn/fast/layers.rs:195-201).
// Unfused, t makes a round trip to HBM and the two convolutions are separate launches; for the
// 32- and 64-channel ResAUs of the SOP / BOP luma nets and the HOP chroma net both are small
// (K = 144 and K = C) and launch- and latency-bound on small maps.
//
// One workgroup (4 waves) owns a TR x 16 tile of positions and all C channels:
//   1. relu6(x) over the (TR + 2) x 18 halo -> LDS (storage type; 16-byte units of a pixel XORed
//      with the pixel index so that 16 consecutive pixels' same unit hits different banks);
//   2. wave w computes t for group w % G (G = C / 16) and rows (w / G) * NPW .. : per output,
//      bias-free, the 9 taps in (ky, kx) order, one K chunk of 16 channels (f32:
//      the piece products of mma_split; f16 / bf16: one 16x16x32 MFMA whose upper 16 K lanes are the
//      zero padding the unfused kernel also multiplies) -- conv_igemm's instruction sequence for
//      this layer; t is rounded to the storage type into LDS, as the unfused kernel stores it;
//   3. the 1x1 over t for output block w % G on the same rows: K chunks in ascending order, the
//      sequence of conv_igemm / conv1x1_ring for a 1x1 layer; then y = x * (1 + a) as two IEEE
//      operations on the raw x, stored in the storage type.
// The A fragments of both convolutions (9 + C / CK per wave) come straight from global memory
// (the same few KB for every workgroup, L2-resident), so LDS holds only the halo and t and
// several workgroups share a CU. Results equal the two unfused launches bit for bit.

#include "ops.h"
#include "split.h"

namespace zjai {

// acc[r] += a . b[r] for N accumulators sharing one A fragment (16-bit types).
template <typename T, int N>
__device__ __forceinline__ void mma_rows(f32x4 (&acc)[N], u32x4 a, const u32x4 (&b)[N]) {
#pragma unroll
    for (int r = 0; r < N; ++r) Mma16<T>::run(acc[r], a, b[r]);
}

template <typename T, int C, int TR>
__global__ void __launch_bounds__(256, sizeof(T) == 4 ? 2 : 1) k_resau(const ResauArgs p) {
    constexpr int VEC = 16 / (int)sizeof(T);  // channels per 16-byte unit
    constexpr int CK = 4 * VEC;               // channels per K chunk (64 bytes)
    constexpr int G = C / 16;                 // groups of 16 channels
    constexpr int UPP = C / VEC;              // 16-byte units per pixel
    constexpr int UG = 16 / VEC;              // units per group
    constexpr int HY = TR + 2, HX = 18, HP = HY * HX;
    constexpr int WPG = 4 / G;                // waves per group
    constexpr int NPW = TR / WPG;             // rows (16-position blocks) per wave
    constexpr int NC2 = C / CK;               // K chunks of the 1x1
    constexpr int HU = HP * UPP, HIT = (HU + 255) / 256;
    static_assert(G == 2 || G == 4, "32 or 64 channels in groups of 16");
    static_assert(TR % WPG == 0 && NPW >= 1, "rows per wave");
    // f32: the halo in split form (split.h) as planes [channel quad][NPX] of (p1, p0) units, then
    // of p2 units; t takes its place once the 3x3 is done.
    constexpr bool F32 = sizeof(T) == 4;
    constexpr int NPX = (HP + 15) / 32 * 32 + 16;
    constexpr int TU = TR * 16 * UPP;
    __shared__ u32x4 s_h[F32 ? UPP * NPX * 3 / 2 : HU];
    __shared__ u32x4 s_tb[F32 ? 1 : TU];
    u32x4* const s_t = F32 ? s_h : s_tb;
    u32x2* const s_hhi = (u32x2*)(s_h + (F32 ? UPP * NPX : 0));

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 15, grp = lane >> 4;
    const int bid = (int)blockIdx.x;
    const int tx = bid % p.gx, ty = (bid / p.gx) % p.gy, b = bid / (p.gx * p.gy);
    const int y0 = ty * TR, x0 = tx * 16;
    const T* xb = (const T*)p.x.p + (long long)b * p.x.bstride + p.x.c_off;
    const int gi = wave % G;           // group (phase 2) and output block (phase 3)
    const int r0 = (wave / G) * NPW;   // first row of this wave

    // A fragments: grouped 3x3 packing [group][tap][16 out][CK], 1x1 packing [chunk][nblk][16][CK]
    // (16-byte units; lane (col, grp) holds row col, K group grp).
    const u32x4* w1 = (const u32x4*)p.w1 + (long long)gi * 9 * (F32 ? SPLIT_BLOCK_U : 64);
    const u32x4* w2 = (const u32x4*)p.w2;
    u32x4 a1[F32 ? 1 : 9], a2[F32 ? 1 : NC2];
    SplitFrag an;  // f32: one tap at a time, the next one's loaded ahead
    auto load_tap = [&](int t) __attribute__((always_inline)) {
        const u32x4* w = w1 + t * SPLIT_BLOCK_U;
        an = SplitFrag{w[lane], ((const u32x2*)(w + 64))[lane]};
    };
    if constexpr (F32) {
        load_tap(0);
    } else {
#pragma unroll
        for (int t = 0; t < 9; ++t) a1[t] = w1[(t * 16 + col) * 4 + grp];
    }
#pragma unroll
    for (int c = 0; c < (F32 ? 0 : NC2); ++c) a2[F32 ? 0 : c] = w2[((c * p.nblk2 + gi) * 16 + col) * 4 + grp];

    // 1. relu6(x) halo. Every load reads a clamped (in-picture) pixel and off-picture ones take
    // zeros afterwards, so all of a thread's loads are in flight together.
    u32x4 hv[HIT];
#pragma unroll
    for (int i = 0; i < HIT; ++i) {
        const int u = min(tid + i * 256, HU - 1), pix = u / UPP, q = u - pix * UPP;
        const int hy = pix / HX, hx = pix - hy * HX;
        const int cy = min(max(y0 - 1 + hy, 0), p.h - 1), cx = min(max(x0 - 1 + hx, 0), p.w - 1);
        hv[i] = *(const u32x4*)(xb + (long long)cy * p.x.row + (long long)cx * p.x.cs + q * VEC);
    }
#pragma unroll
    for (int i = 0; i < HIT; ++i) {
        const int u = tid + i * 256, pix = u / UPP, q = u - pix * UPP;
        const int hy = pix / HX, hx = pix - hy * HX;
        const int iy = y0 - 1 + hy, ix = x0 - 1 + hx;
        const bool in = iy >= 0 && iy < p.h && ix >= 0 && ix < p.w;
        hv[i] = in ? relu6_vec<T>(hv[i]) : u32x4{0u, 0u, 0u, 0u};
        if (!F32 && u < HU) s_h[pix * UPP + (q ^ (pix & (UPP - 1)))] = hv[i];
    }
    if constexpr (F32) {
        f32x4 v[HIT];
#pragma unroll
        for (int i = 0; i < HIT; ++i) v[i] = __builtin_bit_cast(f32x4, hv[i]);
        split_each<HIT>(v, [&](int i, const SplitFrag& f) __attribute__((always_inline)) {
            const int u = tid + i * 256, pix = u / UPP, q = u - pix * UPP;
            if (u >= HU) return;
            s_h[q * NPX + pix] = f.lo;
            s_hhi[q * NPX + pix] = f.hi;
        });
    }
    __syncthreads();

    // 2. t for group gi, rows r0 .. r0 + NPW - 1: bias-free, taps (ky, kx) ascending.
    f32x4 acc[NPW];
#pragma unroll
    for (int r = 0; r < NPW; ++r) acc[r] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const int qb = gi * UG + (grp & (UG - 1));  // this lane's unit of the group
    if constexpr (F32) {
        f32x4 small[NPW];
#pragma unroll
        for (int r = 0; r < NPW; ++r) small[r] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
        for (int t = 0; t < 9; ++t) {
            const SplitFrag a = an;
            load_tap(min(t + 1, 8));
            const int i0 = qb * NPX + (r0 + t / 3) * HX + col + t % 3;
            SplitFrag bv[NPW];
#pragma unroll
            for (int r = 0; r < NPW; ++r) bv[r] = SplitFrag{s_h[i0 + r * HX], s_hhi[i0 + r * HX]};
            mma_split_rows<NPW>(acc, small, a, bv);
        }
#pragma unroll
        for (int r = 0; r < NPW; ++r) acc[r] = split_sum(acc[r], small[r]);
        __syncthreads();  // the halo is no longer read: t takes its place
    } else {
#pragma unroll
        for (int t = 0; t < 9; ++t) {
            const int ky = t / 3, kx = t - 3 * (t / 3);
            u32x4 bv[NPW];
#pragma unroll
            for (int r = 0; r < NPW; ++r) {
                const int pix = (r0 + r + ky) * HX + col + kx;
                bv[r] = s_h[pix * UPP + (qb ^ (pix & (UPP - 1)))];
                if (grp >= UG) bv[r] = u32x4{0u, 0u, 0u, 0u};  // 16-bit: K lanes 16..31 are padding
            }
            mma_rows<T, NPW>(acc, a1[t], bv);
        }
    }
    // f32: t in split form, planes [channel quad][TPX positions] as the halo's.
    constexpr int TPX = (TR * 16 + 15) / 32 * 32 + 16;
    static_assert(!F32 || UPP * TPX <= UPP * NPX, "t fits the halo's place");
    u32x2* const s_thi = (u32x2*)(s_h + (F32 ? UPP * TPX : 0));
    // t (channel gi * 16 + 4 grp + k at position (r0 + r) * 16 + col) rounded to the storage type.
    if constexpr (F32)
        split_each<NPW>(acc, [&](int r, const SplitFrag& f) __attribute__((always_inline)) {
            const int i = (gi * 4 + grp) * TPX + (r0 + r) * 16 + col;
            s_h[i] = f.lo;
            s_thi[i] = f.hi;
        });
#pragma unroll
    for (int r = 0; r < (F32 ? 0 : NPW); ++r) {
        const int pos = (r0 + r) * 16 + col;
        const int ch = gi * 16 + 4 * grp, unit = ch / VEC;
        T* dst = reinterpret_cast<T*>(s_t + pos * UPP + (unit ^ (pos & (UPP - 1)))) + (ch - unit * VEC);
        typedef T t4 __attribute__((ext_vector_type(4)));
        t4 v;
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = (T)acc[r][k];
        *reinterpret_cast<t4*>(dst) = v;
    }
    __syncthreads();

    // 3. a = W2 . t (output block gi), K chunks ascending; y = x * (1 + a).
    f32x4 acc2[NPW];
#pragma unroll
    for (int r = 0; r < NPW; ++r) acc2[r] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (F32) {
        // Two chunks at a time (mma_split32); the weights are L2-resident.
#pragma unroll 1
        for (int c = 0; c < NC2; c += 2) {
            SplitFrag a[2], bv[2][NPW];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const u32x4* w = w2 + ((c + k) * p.nblk2 + gi) * SPLIT_BLOCK_U;
                a[k] = SplitFrag{w[lane], ((const u32x2*)(w + 64))[lane]};
#pragma unroll
                for (int r = 0; r < NPW; ++r) {
                    const int i = ((c + k) * 4 + grp) * TPX + (r0 + r) * 16 + col;
                    bv[k][r] = SplitFrag{s_h[i], s_thi[i]};
                }
            }
            mma_split32<NPW>(acc2, a[0], a[1], bv[0], bv[1], true);
        }
    } else {
#pragma unroll
        for (int c = 0; c < NC2; ++c) {
            u32x4 bv[NPW];
#pragma unroll
            for (int r = 0; r < NPW; ++r) {
                const int pos = (r0 + r) * 16 + col;
                bv[r] = s_t[pos * UPP + ((c * 4 + grp) ^ (pos & (UPP - 1)))];
            }
            mma_rows<T, NPW>(acc2, a2[c], bv);
        }
    }
    T* yb = (T*)p.y.p + (long long)b * p.y.bstride + p.y.c_off;
    const int ch = gi * 16 + 4 * grp;
#pragma unroll
    for (int r = 0; r < NPW; ++r) {
        const int oy = y0 + r0 + r, ox = x0 + col;
        if (oy >= p.h || ox >= p.w) continue;
        const f32x4 xv = load4<T>(xb + (long long)oy * p.x.row + (long long)ox * p.x.cs + ch);
        f32x4 v;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float g = 1.0f + acc2[r][k];
            v[k] = xv[k] * g;
        }
        store4<T>(yb + (long long)oy * p.y.row + (long long)ox * p.y.cs + ch, v);
    }
}

namespace {

template <typename T, int C, int TR>
hipError_t go_resau(ResauArgs p, hipStream_t s) {
    p.gx = (p.w + 15) / 16;
    p.gy = (p.h + TR - 1) / TR;
    const long long total = (long long)p.gx * p.gy * p.N;
    if (total <= 0 || total > (1ll << 30)) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_resau<T, C, TR>), dim3((unsigned)total), dim3(256), 0, s, p);
    return hipGetLastError();
}

template <typename T>
hipError_t go_resau_t(int C, int tr, const ResauArgs& p, hipStream_t s) {
    if (C == 32) return tr == 8 ? go_resau<T, 32, 8>(p, s) : go_resau<T, 32, 4>(p, s);
    if (C == 64) return tr == 8 ? go_resau<T, 64, 8>(p, s) : go_resau<T, 64, 4>(p, s);
    return hipErrorInvalidValue;
}

}  // namespace

bool resau_fused_supported(int C, int groups) { return (C == 32 || C == 64) && groups * 16 == C; }

int resau_rows(int N, int h, int w) {
    // 8-row tiles unless that leaves fewer than 256 workgroups (one per CU).
    const long long t8 = (long long)((w + 15) / 16) * ((h + 7) / 8) * N;
    return t8 >= 256 ? 8 : 4;
}

hipError_t launch_resau(int dtype, int C, const ResauArgs& p, hipStream_t s) {
    const int vec = dtype == DT_F32 ? 4 : 8;
    if (p.N < 1 || p.N > MAXB || p.h < 1 || p.w < 1 || p.x.cs % vec || p.x.c_off % vec || p.x.row % vec ||
        p.x.bstride % vec || p.y.cs % vec || p.y.c_off % vec || (uintptr_t)p.x.p % 16 || (uintptr_t)p.y.p % 16)
        return hipErrorInvalidValue;
    const int tr = resau_rows(p.N, p.h, p.w);
    switch (dtype) {
        case DT_F32: return go_resau_t<float>(C, tr, p, s);
        case DT_F16: return go_resau_t<_Float16>(C, tr, p, s);
        case DT_BF16: return go_resau_t<__bf16>(C, tr, p, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace zjai
