// f32 implicit-GEMM convolution on the bf16 matrix cores (see split.h for the arithmetic).
//
// GEMM roles and tiling as conv_igemm (conv.hip): one workgroup computes TY = WP * PF output rows
// x 16 columns x NB = WC * CF blocks of 16 output channels, K = input channels (16 per chunk) x
// taps. Per chunk the input halo is loaded into registers one chunk ahead, split into its bf16
// pieces and stored to LDS once (each staged value feeds 9 taps x NB * 16 outputs, so the split's
// ~9 vector instructions per value disappear beside the MFMAs they allow); the weights are packed
// already split and stream through a two-slot LDS ring by direct loads, TS taps per slot.
//
// LDS layout of a halo: planes [4 channel quads][NPX pixels] of 16-byte (p1, p0) units, then of
// 8-byte p2 units, NPX = 16 (mod 32): a fragment read's 16 consecutive pixels x 4 quads then fall
// on distinct banks for any first pixel (ds_read_b128 takes 16 lanes of two quads per pass,
// ds_read_b64 32 lanes). Weight blocks are stored in lane order.
//
// The sum of an output is, for every tile shape: bias, then per chunk and tap the three MFMAs of
// mma_split -- so the choice of tile never changes a bit.

#include "conv.h"
#include "epilogue.h"
#include "split.h"

#include <type_traits>

namespace zjai {

__device__ u32x4 g_zero_split[1];  // 16 zero bytes: the source of padding units

template <int KH, int KW, int S, bool TR, int WC, int WP, int CF, int PF, int TS, int NHB, int RW>
__global__ void __launch_bounds__(WC * WP * 64, S == 1 && CF * PF == 4 ? 4 : 2)  // 4: as LDS allows, in 128 registers
conv_igemm_split(const ConvParams p) {
    constexpr int NT = WC * WP * 64;
    constexpr int TY = WP * PF;
    constexpr int HY = (TY - 1) * S + KH, HX = 15 * S + KW, HP = HY * HX;
    constexpr int NTAP = TR ? 4 : KH * KW, NST = NTAP / TS;
    static_assert(!TR || (KH == 3 && KW == 3 && S == 1 && TS == 4), "a phase's taps in one stage");
    static_assert(NTAP % TS == 0, "whole stages");
    constexpr int NB = WC * CF;
    constexpr int NPX = (HP + 15) / 32 * 32 + 16;
    static_assert(NPX >= HP, "plane size");
    constexpr int HALO_U = 6 * NPX;                  // 16-byte units of one halo buffer
    constexpr int W_U = NB * TS * SPLIT_BLOCK_U;     // of one weight slot
    constexpr int OUT_LD = NB * 16 + 4;              // f32 output tile [positions][channels + 4]
    constexpr int OUT_U = (TY * 16 * OUT_LD + 3) / 4;
    constexpr int RUN_U = NHB * HALO_U + RW * W_U;
    constexpr int LDS_U = RUN_U > OUT_U ? RUN_U : OUT_U;
    constexpr int HN = (HP * 4 + NT - 1) / NT, WN = (W_U + NT - 1) / NT;
    __shared__ u32x4 s_lds[LDS_U];
    u32x4* const s_w = s_lds + NHB * HALO_U;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wc = wave % WC, wp = wave / WC;
    const int col = lane & 15, grp = lane >> 4;

    // Workgroup -> tile: the XCD-aware order of conv_igemm.
    const int nz = p.ntiles * (TR ? 4 : 1);
    const int total = p.gx * p.gy * p.N * nz;
    const int bid = (int)blockIdx.x, xj = bid & 7, xk = bid >> 3;
    const int q8 = total >> 3, r8 = total & 7;
    const int lid = xj < r8 ? xj * (q8 + 1) + xk : r8 * (q8 + 1) + (xj - r8) * q8 + xk;
    int rest = lid / nz;
    const int zl = lid - rest * nz, phase = TR ? (zl & 3) : 0, nt = TR ? (zl >> 2) : zl;
    const int tx = rest % p.gx;
    rest /= p.gx;
    const int ty = rest % p.gy, bi = rest / p.gy;
    const int gb = nt * NB;
    const int g = gb / p.nblk_g, nb0 = gb - g * p.nblk_g;
    const int ox0 = tx * 16, oy0 = ty * TY;
    if (nb0 * 16 >= p.cout_g) return;  // padding blocks only (uniform)

    f32x4 big[CF][PF], small[CF][PF];
#pragma unroll
    for (int cf = 0; cf < CF; ++cf) {
        const int ocl = (nb0 + wc * CF + cf) * 16 + grp * 4;
        f32x4 b;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            b[i] = (p.bias && ocl + i < p.cout_g) ? p.bias[g * p.cout_g + ocl + i] : 0.0f;
#pragma unroll
        for (int pf = 0; pf < PF; ++pf) {
            big[cf][pf] = b;
            small[cf][pf] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }

    const int iy0 = TR ? oy0 - 1 : oy0 * S - p.pad_t, ix0 = TR ? ox0 - 1 : ox0 * S - p.pad_l;
    const float* xg = (const float*)p.x.p + (long long)bi * p.x.bstride;
    const long long xbase = (long long)p.x.c_off + (long long)g * p.cin_g;

    // LDS slot of halo pixel (hy, hx): stride-2 halos keep each row's even columns, then its odd
    // ones, so that a fragment's every-other-column reads are consecutive slots.
    constexpr int HXE = (HX + 1) / 2;
    auto hslot = [](int hy, int hx) __attribute__((always_inline)) {
        return S == 2 ? hy * HX + ((hx & 1) ? HXE + (hx >> 1) : (hx >> 1)) : hy * HX + hx;
    };
    // This thread's halo units (channel quad q of a pixel): where the next chunk's is read from and
    // how far that moves per chunk (padding reads 16 zero bytes and stays there), and its LDS slot.
    const float* hp[HN];
    int hstep[HN], hdst[HN];
#pragma unroll
    for (int i = 0; i < HN; ++i) {
        const int u = tid + i * NT, pix = u >> 2, q = u & 3;
        const int hy = pix / HX, hx = pix - hy * HX;
        const int iy = iy0 + hy, ix = ix0 + hx;
        const bool in = u < HP * 4 && iy >= 0 && iy < p.H && ix >= 0 && ix < p.W;
        hp[i] = in ? xg + (long long)iy * p.x.row + (long long)ix * p.x.cs + xbase + q * 4 : (const float*)g_zero_split;
        hstep[i] = in ? 16 : 0;
        hdst[i] = q * NPX + hslot(hy, hx);
    }
    const int qv = (tid & 3) * 4;
    u32x4 rh[HN];
    auto load_halo = [&](int chunk) __attribute__((always_inline)) {
        if (chunk * 16 + 16 <= p.cin_g) {
#pragma unroll
            for (int i = 0; i < HN; ++i) {
                rh[i] = *(const u32x4*)hp[i];
                hp[i] += hstep[i];
            }
        } else {  // the last chunk of a cin_g off 16
#pragma unroll
            for (int i = 0; i < HN; ++i)
                rh[i] = *(chunk * 16 + qv < p.cin_g ? (const u32x4*)hp[i] : g_zero_split);
        }
    };
    auto store_halo = [&](int chunk) __attribute__((always_inline)) {
        u32x4* dst = s_lds + (NHB == 2 ? (chunk & 1) * HALO_U : 0);
        u32x2* hi = (u32x2*)(dst + 4 * NPX);
        f32x4 v[HN];
#pragma unroll
        for (int i = 0; i < HN; ++i) v[i] = __builtin_bit_cast(f32x4, p.relu6_in ? relu6_vec<float>(rh[i]) : rh[i]);
        split_each<HN>(v, [&](int i, const SplitFrag& f) __attribute__((always_inline)) {
            if (tid + i * NT < HP * 4) {
                dst[hdst[i]] = f.lo;
                hi[hdst[i]] = f.hi;
            }
        });
    };
    // Weight slot of stage (chunk, j): taps j * TS .. of blocks nb0 .. nb0 + NB - 1, loaded RW - 1
    // stages ahead (the slot was last read that many stages ago). The lanes' offsets stay, the
    // uniform base moves.
    const char* const wg = (const char*)((const u32x4*)((const float*)p.w + phase * p.phase_stride + bi * p.w_bstride) + ((long long)g * p.nchunks * p.nblk_g + nb0) * (NTAP * SPLIT_BLOCK_U));
    const long long wchunk = (long long)p.nblk_g * (NTAP * SPLIT_BLOCK_U * 16);
    unsigned woff[WN];
#pragma unroll
    for (int i = 0; i < WN; ++i) {
        const int u = tid + i * NT, nb = u / (TS * SPLIT_BLOCK_U);
        woff[i] = (unsigned)(nb * (NTAP * SPLIT_BLOCK_U) + (u - nb * (TS * SPLIT_BLOCK_U))) * 16;
    }
    auto issue_stage = [&](int st, int slot) __attribute__((always_inline)) {
        const int c = NST == 1 ? st : st / NST;
        const char* src = wg + c * wchunk + (st - c * NST) * (TS * SPLIT_BLOCK_U * 16);
        u32x4* dst = s_w + slot * W_U;
#pragma unroll
        for (int i = 0; i < WN; ++i) {
            const int ub = wave * 64 + i * NT;
            if (ub >= W_U) break;
            if (ub + lane < W_U) lds_dma16_at(src, woff[i], dst + ub);
        }
    };

    constexpr int CW = W_U / NT;  // direct loads per stage that every wave issues at least
    const int nchunks = p.nchunks, nst = nchunks * NST;
    load_halo(0);
    for (int k = 0; k < RW - 1 && k < nst; ++k) issue_stage(k, k);
    int slot = 0, nslot = RW - 1;  // ring slots of stage st and of stage st + RW - 1
#pragma unroll 1
    for (int chunk = 0, st = 0; chunk < nchunks; ++chunk) {
        const u32x4* s_halo = s_lds + (NHB == 2 ? (chunk & 1) * HALO_U : 0);
        const u32x2* s_hhi = (const u32x2*)(s_halo + 4 * NPX);
#pragma unroll 1
        for (int j = 0; j < NST; ++j, ++st) {
            if (j == 0) {
                if (NHB == 1 && chunk > 0) __syncthreads();  // every wave is done with the last halo
                store_halo(chunk);
            }
            // This wave's weight loads of the stage are in LDS; those of the next RW - 2 stages and
            // the halo loads of the next chunk (issued after them) may still fly.
            const bool more = RW == 3 && st + 1 < nst, halo = j >= 1 && j < RW && chunk + 1 < nchunks;
            if (more && halo) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(CW + HN) : "memory");
            else if (more) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(CW) : "memory");
            else if (halo && RW == 2) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(HN) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
            __syncthreads();  // ... and every other wave's, and the split halo
            if (st + RW - 1 < nst) issue_stage(st + RW - 1, nslot);
            if (j == 0 && chunk + 1 < nchunks) load_halo(chunk + 1);
            const u32x4* sw = s_w + slot * W_U;
            slot = slot + 1 == RW ? 0 : slot + 1;
            nslot = nslot + 1 == RW ? 0 : nslot + 1;
#pragma unroll
            for (int t = 0; t < TS; ++t) {
                const int tap = j * TS + t;
                if (TR && t >= p.ntaps[phase]) break;
                const int ky = TR ? p.tap_dy[phase][t] : tap / KW, kx = TR ? p.tap_dx[phase][t] : tap - tap / KW * KW;
                SplitFrag a[CF], b[PF];
#pragma unroll
                for (int cf = 0; cf < CF; ++cf) {
                    const u32x4* w = sw + ((wc * CF + cf) * TS + t) * SPLIT_BLOCK_U;
                    a[cf].lo = w[lane];
                    a[cf].hi = ((const u32x2*)(w + 64))[lane];
                }
#pragma unroll
                for (int pf = 0; pf < PF; ++pf) {
                    const int s = grp * NPX + hslot((wp * PF + pf) * S + ky, col * S + kx);
                    b[pf].lo = s_halo[s];
                    b[pf].hi = s_hhi[s];
                }
#pragma unroll
                for (int cf = 0; cf < CF; ++cf)
#pragma unroll
                    for (int pf = 0; pf < PF; ++pf) mma_split(big[cf][pf], small[cf][pf], a[cf], b[pf]);
            }
            if (NTAP == 1 && ((chunk & 1) || chunk + 1 == nchunks)) {  // mma_split32's order
#pragma unroll
                for (int cf = 0; cf < CF; ++cf)
#pragma unroll
                    for (int pf = 0; pf < PF; ++pf) {
                        big[cf][pf] = split_sum(big[cf][pf], small[cf][pf]);
                        small[cf][pf] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                    }
            }
        }
    }

    // Transposed through LDS: every position's NB * 16 channels leave as one contiguous run.
    __syncthreads();
    float* so = reinterpret_cast<float*>(s_lds);
#pragma unroll
    for (int cf = 0; cf < CF; ++cf)
#pragma unroll
        for (int pf = 0; pf < PF; ++pf)
            *reinterpret_cast<f32x4*>(so + ((wp * PF + pf) * 16 + col) * OUT_LD + (wc * CF + cf) * 16 + grp * 4) =
                NTAP == 1 ? big[cf][pf] : split_sum(big[cf][pf], small[cf][pf]);
    __syncthreads();
    // Output row / column of position pos (a phase's are every other one).
    auto oy_of = [&](int pos) { return TR ? 2 * (oy0 + (pos >> 4)) + (phase >> 1) : oy0 + (pos >> 4); };
    auto ox_of = [&](int pos) { return TR ? 2 * (ox0 + (pos & 15)) + (phase & 1) : ox0 + (pos & 15); };
    const bool full = nb0 * 16 + NB * 16 <= p.cout_g;  // all of the tile's channels are real
    if (full && epilogue_simple(p)) {
        constexpr int QP8 = NB * 2;  // 8 channels per thread and step
#pragma unroll 4
        for (int u = tid; u < TY * 16 * QP8; u += NT) {
            const int pos = u / QP8, c8 = u - pos * QP8;
            const int oy = oy_of(pos), ox = ox_of(pos);
            const f32x4 v0 = *reinterpret_cast<const f32x4*>(so + pos * OUT_LD + c8 * 8);
            const f32x4 v1 = *reinterpret_cast<const f32x4*>(so + pos * OUT_LD + c8 * 8 + 4);
            if (oy < p.OH && ox < p.OW) epilogue_store8<float>(p, bi, oy, ox, g * p.cout_g + nb0 * 16 + c8 * 8, v0, v1);
        }
        return;
    }
    if (full && epilogue_ps2(p)) {
        // Pixel shuffle by 2: conv channels 4 c + s of 4 consecutive output channels c, one
        // sub-position s, as one vector store.
        constexpr int QP = NB * 4;
        for (int u = tid; u < TY * 16 * QP; u += NT) {
            const int pos = u / QP, q = u - pos * QP, cq = q % NB, sub = q / NB;
            const int oy = oy_of(pos), ox = ox_of(pos);
            if (oy >= p.OH || ox >= p.OW) continue;
            const float* v = so + pos * OUT_LD + cq * 16 + sub;
            epilogue_store_ps2<float>(p, bi, oy, ox, sub, (g * p.cout_g + nb0 * 16) / 4 + cq * 4,
                                      f32x4{v[0], v[4], v[8], v[12]});
        }
        return;
    }
    constexpr int QP = NB * 4;
    for (int u = tid; u < TY * 16 * QP; u += NT) {
        const int pos = u / QP, cq = u - pos * QP;
        const int oy = oy_of(pos), ox = ox_of(pos);
        const int ocl = nb0 * 16 + cq * 4;
        if (oy >= p.OH || ox >= p.OW || ocl >= p.cout_g) continue;
        const f32x4 v = *reinterpret_cast<const f32x4*>(so + pos * OUT_LD + cq * 4);
        epilogue_store<float>(p, bi, oy, ox, g * p.cout_g + ocl, min(4, p.cout_g - ocl), v);
    }
}

// ---------------------------------------------------------------------------------------------
// Stride-2 transposed 3x3 convolution, padding 1, the four output phases of a tile in one
// workgroup (conv_tr_merged's plan, conv.hip): four blocks of 16 channels x four rows x 16 columns of
// input positions; each wave accumulates two blocks x two rows for all four phases. A
// phase reads the 2 x 2 input neighbourhood of a position, so the halo is one row and one column
// and a chunk's nine taps share its few fragments. Weights (split, phase by phase) go through an
// LDS ring three taps at a time. Per output the sums are conv_igemm_split's: bias, then per chunk
// its phase's taps in table order.
// ---------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256, 2)
conv_tr_merged_split(const ConvParams p) {
    constexpr int WC = 2, WP = 2, CF = 2, PF = 2, NT = WC * WP * 64;
    constexpr int TY = WP * PF, HY = TY + 1, HX = 17, HP = HY * HX;
    constexpr int NB = WC * CF, TS = 3, NST = 3;
    constexpr int NPX = (HP + 15) / 32 * 32 + 16;
    constexpr int HALO_U = 6 * NPX, W_U = NB * TS * SPLIT_BLOCK_U;
    constexpr int OUT_LD = NB * 16 + 4, OUT_U = (TY * 16 * OUT_LD + 3) / 4;
    constexpr int RUN_U = HALO_U + 2 * W_U;
    constexpr int LDS_U = RUN_U > OUT_U ? RUN_U : OUT_U;
    constexpr int HN = (HP * 4 + NT - 1) / NT, WN = (W_U + NT - 1) / NT;
    // Taps in packing order: phase (py * 2 + px) and input offset (dy, dx) of each.
    constexpr int PH[9] = {0, 1, 1, 2, 2, 3, 3, 3, 3};
    constexpr int DY[9] = {0, 0, 0, 1, 0, 1, 1, 0, 0}, DX[9] = {0, 1, 0, 0, 0, 1, 0, 1, 0};
    __shared__ u32x4 s_lds[LDS_U];
    u32x2* const s_hhi = (u32x2*)(s_lds + 4 * NPX);
    u32x4* const s_w = s_lds + HALO_U;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wc = wave % WC, wp = wave / WC;
    const int col = lane & 15, grp = lane >> 4;

    const int nz = p.ntiles;
    const int total = p.gx * p.gy * p.N * nz;
    const int bid = (int)blockIdx.x, xj = bid & 7, xk = bid >> 3;
    const int q8 = total >> 3, r8 = total & 7;
    const int lid = xj < r8 ? xj * (q8 + 1) + xk : r8 * (q8 + 1) + (xj - r8) * q8 + xk;
    int rest = lid / nz;
    const int nb0 = (lid - rest * nz) * NB;
    const int tx = rest % p.gx;
    rest /= p.gx;
    const int ty = rest % p.gy, bi = rest / p.gy;
    const int ox0 = tx * 16, oy0 = ty * TY;
    if (nb0 * 16 >= p.cout_g) return;  // padding blocks only (uniform)

    f32x4 big[4][CF][PF], small[4][CF][PF];
#pragma unroll
    for (int cf = 0; cf < CF; ++cf) {
        const int ocl = (nb0 + wc * CF + cf) * 16 + grp * 4;
        f32x4 b;
#pragma unroll
        for (int i = 0; i < 4; ++i) b[i] = (p.bias && ocl + i < p.cout_g) ? p.bias[ocl + i] : 0.0f;
#pragma unroll
        for (int ph = 0; ph < 4; ++ph)
#pragma unroll
            for (int pf = 0; pf < PF; ++pf) {
                big[ph][cf][pf] = b;
                small[ph][cf][pf] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
    }

    const float* xg = (const float*)p.x.p + (long long)bi * p.x.bstride + p.x.c_off;
    const float* hp[HN];
    int hstep[HN], hdst[HN];
#pragma unroll
    for (int i = 0; i < HN; ++i) {
        const int u = tid + i * NT, pix = u >> 2, q = u & 3;
        const int hy = pix / HX, hx = pix - hy * HX;
        const int iy = oy0 + hy, ix = ox0 + hx;
        const bool in = u < HP * 4 && iy < p.H && ix < p.W;
        hp[i] = in ? xg + (long long)iy * p.x.row + (long long)ix * p.x.cs + q * 4 : (const float*)g_zero_split;
        hstep[i] = in ? 16 : 0;
        hdst[i] = q * NPX + pix;
    }
    const int qv = (tid & 3) * 4;
    u32x4 rh[HN];
    auto load_halo = [&](int chunk) __attribute__((always_inline)) {
        if (chunk * 16 + 16 <= p.cin_g) {
#pragma unroll
            for (int i = 0; i < HN; ++i) {
                rh[i] = *(const u32x4*)hp[i];
                hp[i] += hstep[i];
            }
        } else {
#pragma unroll
            for (int i = 0; i < HN; ++i)
                rh[i] = *(chunk * 16 + qv < p.cin_g ? (const u32x4*)hp[i] : g_zero_split);
        }
    };
    const char* const wg = (const char*)((const u32x4*)p.w + (long long)nb0 * (TR_MERGED_TAPS * SPLIT_BLOCK_U));
    const long long wchunk = (long long)p.nblk_g * (TR_MERGED_TAPS * SPLIT_BLOCK_U * 16);
    unsigned woff[WN];
#pragma unroll
    for (int i = 0; i < WN; ++i) {
        const int u = tid + i * NT, nb = u / (TS * SPLIT_BLOCK_U);
        woff[i] = (unsigned)(nb * (TR_MERGED_TAPS * SPLIT_BLOCK_U) + (u - nb * (TS * SPLIT_BLOCK_U))) * 16;
    }
    auto issue_stage = [&](int st, int slot) __attribute__((always_inline)) {
        const int c = st / NST;
        const char* src = wg + c * wchunk + (st - c * NST) * (TS * SPLIT_BLOCK_U * 16);
        u32x4* dst = s_w + slot * W_U;
#pragma unroll
        for (int i = 0; i < WN; ++i) {
            const int ub = wave * 64 + i * NT;
            if (ub >= W_U) break;
            if (ub + lane < W_U) lds_dma16_at(src, woff[i], dst + ub);
        }
    };

    const int nchunks = p.nchunks, nst = nchunks * NST;
    load_halo(0);
    issue_stage(0, 0);
#pragma unroll 1
    for (int chunk = 0, st = 0; chunk < nchunks; ++chunk) {
        auto stage = [&](auto jc) __attribute__((always_inline)) {
            constexpr int j = decltype(jc)::value;
            if (j == 0) {
                if (chunk > 0) __syncthreads();  // every wave is done with the last halo
                f32x4 v[HN];
#pragma unroll
                for (int i = 0; i < HN; ++i) v[i] = __builtin_bit_cast(f32x4, rh[i]);
                split_each<HN>(v, [&](int i, const SplitFrag& f) __attribute__((always_inline)) {
                    if (tid + i * NT < HP * 4) {
                        s_lds[hdst[i]] = f.lo;
                        s_hhi[hdst[i]] = f.hi;
                    }
                });
            }
            // This stage's weights have landed; the next chunk's halo loads, issued after them, may
            // still fly.
            if (j == 1 && chunk + 1 < nchunks) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(HN) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
            __syncthreads();
            if (st + 1 < nst) issue_stage(st + 1, (st + 1) & 1);
            if (j == 0 && chunk + 1 < nchunks) load_halo(chunk + 1);
            const u32x4* sw = s_w + (st & 1) * W_U;
            ++st;
#pragma unroll
            for (int t = 0; t < TS; ++t) {
                constexpr int E = j * TS;
                SplitFrag a[CF], b[PF];
#pragma unroll
                for (int cf = 0; cf < CF; ++cf) {
                    const u32x4* w = sw + ((wc * CF + cf) * TS + t) * SPLIT_BLOCK_U;
                    a[cf] = SplitFrag{w[lane], ((const u32x2*)(w + 64))[lane]};
                }
#pragma unroll
                for (int pf = 0; pf < PF; ++pf) {
                    const int i = grp * NPX + (wp * PF + pf + DY[E + t]) * HX + col + DX[E + t];
                    b[pf] = SplitFrag{s_lds[i], s_hhi[i]};
                }
#pragma unroll
                for (int cf = 0; cf < CF; ++cf)
#pragma unroll
                    for (int pf = 0; pf < PF; ++pf)
                        mma_split(big[PH[E + t]][cf][pf], small[PH[E + t]][cf][pf], a[cf], b[pf]);
            }
        };
        stage(std::integral_constant<int, 0>{});
        stage(std::integral_constant<int, 1>{});
        stage(std::integral_constant<int, 2>{});
    }

    // One phase at a time through the LDS transpose (NHWC output without pixel shuffle).
    float* so = reinterpret_cast<float*>(s_lds);
#pragma unroll
    for (int ph = 0; ph < 4; ++ph) {
        __syncthreads();
#pragma unroll
        for (int cf = 0; cf < CF; ++cf)
#pragma unroll
            for (int pf = 0; pf < PF; ++pf)
                *reinterpret_cast<f32x4*>(so + ((wp * PF + pf) * 16 + col) * OUT_LD + (wc * CF + cf) * 16 + grp * 4) =
                    split_sum(big[ph][cf][pf], small[ph][cf][pf]);
        __syncthreads();
        if (nb0 * 16 + NB * 16 <= p.cout_g) {
            constexpr int QP8 = NB * 2;
#pragma unroll 4
            for (int u = tid; u < TY * 16 * QP8; u += NT) {
                const int pos = u / QP8, c8 = u - pos * QP8;
                const int oy = 2 * (oy0 + (pos >> 4)) + (ph >> 1), ox = 2 * (ox0 + (pos & 15)) + (ph & 1);
                const f32x4 v0 = *reinterpret_cast<const f32x4*>(so + pos * OUT_LD + c8 * 8);
                const f32x4 v1 = *reinterpret_cast<const f32x4*>(so + pos * OUT_LD + c8 * 8 + 4);
                if (oy < p.OH && ox < p.OW) epilogue_store8<float>(p, bi, oy, ox, nb0 * 16 + c8 * 8, v0, v1);
            }
        } else {
            constexpr int QP = NB * 4;
            for (int u = tid; u < TY * 16 * QP; u += NT) {
                const int pos = u / QP, cq = u - pos * QP, ocl = nb0 * 16 + cq * 4;
                const int oy = 2 * (oy0 + (pos >> 4)) + (ph >> 1), ox = 2 * (ox0 + (pos & 15)) + (ph & 1);
                if (oy >= p.OH || ox >= p.OW || ocl >= p.cout_g) continue;
                const f32x4 v = *reinterpret_cast<const f32x4*>(so + pos * OUT_LD + cq * 4);
                epilogue_store<float>(p, bi, oy, ox, ocl, min(4, p.cout_g - ocl), v);
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// 1x1 layers as a GEMM over row-major positions: WC * CF blocks of 16 channels x MP = WP * PF * 16
// consecutive positions of one batch item per workgroup, K in stages of 32 channels. A stage's
// positions are loaded into registers one stage ahead (8 lanes read a position's 128 bytes), split
// and stored to planes [8 channel quads][positions], position p of quad q at p ^ q: the eight
// quads a store pass holds of one position, and the 16 positions x 2 quads of a fragment read
// pass, fall on distinct banks. The weights stream through a two-slot ring of direct loads. Sums
// are mma_split32's, so a layer gives the same bits here and in conv_igemm_split.
//
// Bound by what surrounds the products: 128 -> 512 at 431^2 takes 255 us (317 on the f32 MFMA), 95
// TFLOP/s and 1.9 TB/s of its 0.48 GB. In a 4K picture the matrix cores work 24 % of the kernel's CU
// time, beside nine vector instructions per MFMA (splits, folds, addresses, the epilogue).
// ---------------------------------------------------------------------------------------------
template <int WC, int WP, int CF, int PF>
__global__ void __launch_bounds__(WC * WP * 64, 3)  // three workgroups per CU, as LDS allows, in 168 registers
conv1x1_ring_split(const ConvParams p) {
    constexpr int NT = WC * WP * 64;
    constexpr int NB = WC * CF, MP = WP * PF * 16;
    constexpr int PXS = (MP + 15) / 32 * 32 + 16;
    constexpr int X_U = 8 * PXS * 3 / 2, W_U = NB * SPLIT_BLOCK_U;  // W_U: one chunk's blocks
    constexpr int OUT_LD = NB * 16 + 4, OUT_U = (MP * OUT_LD + 3) / 4;
    constexpr int RUN_U = X_U + 4 * W_U;
    constexpr int LDS_U = RUN_U > OUT_U ? RUN_U : OUT_U;
    constexpr int XN = MP * 8 / NT, WN = (W_U + NT - 1) / NT;
    static_assert(MP * 8 % NT == 0, "whole loads");
    __shared__ u32x4 s_lds[LDS_U];
    u32x2* const s_xhi = (u32x2*)(s_lds + 8 * PXS);
    u32x4* const s_w = s_lds + X_U;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wc = wave % WC, wp = wave / WC;
    const int col = lane & 15, grp = lane >> 4;

    // XCD-aware order (conv_igemm's): the channel tiles of one position tile share an L2.
    const int P = p.OH * p.OW;
    const int ptiles = (P + MP - 1) / MP;
    const int nct = p.ntiles;
    const int total = p.N * ptiles * nct;
    const int bid = (int)blockIdx.x, xj = bid & 7, xk = bid >> 3;
    const int q8 = total >> 3, r8 = total & 7;
    const int lid = xj < r8 ? xj * (q8 + 1) + xk : r8 * (q8 + 1) + (xj - r8) * q8 + xk;
    int rest = lid / nct;
    const int ct = lid - rest * nct;
    const int pt = rest % ptiles, bi = rest / ptiles;
    const int pos0 = pt * MP, nb0 = ct * NB;
    if (nb0 * 16 >= p.cout_g) return;  // padding blocks only (uniform)

    f32x4 acc[CF][PF];
#pragma unroll
    for (int cf = 0; cf < CF; ++cf) {
        const int oc = (nb0 + wc * CF + cf) * 16 + grp * 4;
        f32x4 b;
#pragma unroll
        for (int i = 0; i < 4; ++i) b[i] = (p.bias && oc + i < p.cout_g) ? p.bias[oc + i] : 0.0f;
#pragma unroll
        for (int pf = 0; pf < PF; ++pf) acc[cf][pf] = b;
    }

    // This thread's position units (quad q of a stage's 32 channels): source, step per stage (0 for
    // positions past the map, which read zeros) and LDS slot.
    const float* xg = (const float*)p.x.p + (long long)bi * p.x.bstride + p.x.c_off;
    const int q = tid & 7;
    const float* xp[XN];
    int xstep[XN], xdst[XN];
#pragma unroll
    for (int i = 0; i < XN; ++i) {
        const int pos = (tid + i * NT) >> 3, pg = pos0 + pos;
        const int oy = pg / p.OW, ox = pg - oy * p.OW;
        xp[i] = pg < P ? xg + (long long)oy * p.x.row + (long long)ox * p.x.cs + q * 4 : (const float*)g_zero_split;
        xstep[i] = pg < P ? 32 : 0;
        xdst[i] = q * PXS + (pos ^ q);
    }
    u32x4 rx[XN];
    auto load_x = [&](int st) __attribute__((always_inline)) {
        if (st * 32 + 32 <= p.cin_g) {
#pragma unroll
            for (int i = 0; i < XN; ++i) {
                rx[i] = *(const u32x4*)xp[i];
                xp[i] += xstep[i];
            }
        } else {  // the last stage of a cin off 32
#pragma unroll
            for (int i = 0; i < XN; ++i)
                rx[i] = *(st * 32 + q * 4 < p.cin_g ? (const u32x4*)xp[i] : g_zero_split);
        }
    };
    const char* const wg = (const char*)((const u32x4*)((const float*)p.w + bi * p.w_bstride) + (long long)nb0 * SPLIT_BLOCK_U);
    const long long wchunk = (long long)p.nblk_g * (SPLIT_BLOCK_U * 16);
    const int nchunks = p.nchunks, nst = (nchunks + 1) / 2;
    auto issue_w = [&](int st) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            if (2 * st + k >= nchunks) break;
            u32x4* dst = s_w + ((st & 1) * 2 + k) * W_U;
#pragma unroll
            for (int i = 0; i < WN; ++i) {
                const int ub = wave * 64 + i * NT;
                if (ub >= W_U) break;
                if (ub + lane < W_U) lds_dma16_at(wg + (2 * st + k) * wchunk, (ub + lane) * 16, dst + ub);
            }
        }
    };

    load_x(0);
    issue_w(0);
#pragma unroll 1
    for (int st = 0; st < nst; ++st) {
        if (st > 0) __syncthreads();  // every wave is done with the last stage's positions
        f32x4 v[XN];
#pragma unroll
        for (int i = 0; i < XN; ++i) v[i] = __builtin_bit_cast(f32x4, rx[i]);
        split_each<XN>(v, [&](int i, const SplitFrag& f) __attribute__((always_inline)) {
            s_lds[xdst[i]] = f.lo;
            s_xhi[xdst[i]] = f.hi;
        });
        asm volatile("s_waitcnt vmcnt(0)" : : : "memory");  // this wave's weights of the stage
        __syncthreads();
        if (st + 1 < nst) {
            issue_w(st + 1);
            load_x(st + 1);
        }
        const u32x4* sw = s_w + (st & 1) * 2 * W_U;
        SplitFrag b[2][PF];
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int pf = 0; pf < PF; ++pf) {
                const int qq = 4 * k + grp, i = qq * PXS + (((wp * PF + pf) * 16 + col) ^ qq);
                b[k][pf] = SplitFrag{s_lds[i], s_xhi[i]};
            }
        const bool two = 2 * st + 1 < nchunks;
#pragma unroll
        for (int cf = 0; cf < CF; ++cf) {
            SplitFrag a[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const u32x4* w = sw + k * W_U + (wc * CF + cf) * SPLIT_BLOCK_U;
                a[k] = SplitFrag{w[lane], ((const u32x2*)(w + 64))[lane]};
            }
            mma_split32<PF>(acc[cf], a[0], a[1], b[0], b[1], two);
        }
    }

    // Transposed through LDS: every position's NB * 16 channels leave as one contiguous run.
    __syncthreads();
    float* so = reinterpret_cast<float*>(s_lds);
#pragma unroll
    for (int cf = 0; cf < CF; ++cf)
#pragma unroll
        for (int pf = 0; pf < PF; ++pf)
            *reinterpret_cast<f32x4*>(so + ((wp * PF + pf) * 16 + col) * OUT_LD + (wc * CF + cf) * 16 + grp * 4) = acc[cf][pf];
    __syncthreads();
    const bool full = nb0 * 16 + NB * 16 <= p.cout_g;
    if (full && epilogue_simple(p)) {
        constexpr int QP8 = NB * 2;
#pragma unroll 4
        for (int u = tid; u < MP * QP8; u += NT) {
            const int pos = u / QP8, c8 = u - pos * QP8, pg = pos0 + pos;
            const f32x4 v0 = *reinterpret_cast<const f32x4*>(so + pos * OUT_LD + c8 * 8);
            const f32x4 v1 = *reinterpret_cast<const f32x4*>(so + pos * OUT_LD + c8 * 8 + 4);
            if (pg < P) {
                const int oy = pg / p.OW, ox = pg - oy * p.OW;
                epilogue_store8<float>(p, bi, oy, ox, nb0 * 16 + c8 * 8, v0, v1);
            }
        }
    } else if (full && epilogue_ps2(p)) {
        constexpr int QP = NB * 4;
#pragma unroll 2
        for (int u = tid; u < MP * QP; u += NT) {
            const int pos = u / QP, r = u - pos * QP, sub = r / NB, cq = r - sub * NB, pg = pos0 + pos;
            if (pg >= P) continue;
            const int oy = pg / p.OW, ox = pg - oy * p.OW;
            const float* v = so + pos * OUT_LD + cq * 16 + sub;
            epilogue_store_ps2<float>(p, bi, oy, ox, sub, nb0 * 4 + cq * 4, f32x4{v[0], v[4], v[8], v[12]});
        }
    } else {
        constexpr int QP = NB * 4;
        for (int u = tid; u < MP * QP; u += NT) {
            const int pos = u / QP, cq = u - pos * QP, pg = pos0 + pos, oc = nb0 * 16 + cq * 4;
            if (pg >= P || oc >= p.cout_g) continue;
            const int oy = pg / p.OW, ox = pg - oy * p.OW;
            epilogue_store<float>(p, bi, oy, ox, oc, min(4, p.cout_g - oc), *reinterpret_cast<const f32x4*>(so + pos * OUT_LD + cq * 4));
        }
    }
}

// Weight blocks [16 outputs][16 channels] to split blocks (split.h), a lane's four channels per
// thread.
__global__ void __launch_bounds__(256) k_split_weights(const float* src, u32x4* dst, long long nblk) {
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x, b = t >> 6;
    if (b >= nblk) return;
    const int lane = (int)t & 63;
    const SplitFrag f = split_f32(*(const f32x4*)(src + b * 256 + (lane & 15) * 16 + (lane >> 4) * 4));
    dst[b * SPLIT_BLOCK_U + lane] = f.lo;
    ((u32x2*)(dst + b * SPLIT_BLOCK_U + 64))[lane] = f.hi;
}

hipError_t launch_split_weights(const float* src, void* dst, long long nblk, hipStream_t s) {
    if (nblk <= 0 || nblk > (1ll << 28)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_split_weights, dim3((unsigned)((nblk + 3) / 4)), dim3(256), 0, s, src, (u32x4*)dst, nblk);
    return hipGetLastError();
}

namespace {

template <int WC, int WP, int CF, int PF>
hipError_t go_1x1_split(const ConvParams& p0, hipStream_t s) {
    constexpr int NB = WC * CF, MP = WP * PF * 16;
    ConvParams p = p0;
    p.ntiles = p.nblk_g / NB;
    const long long total = ((long long)p.OH * p.OW + MP - 1) / MP * p.N * p.ntiles;
    if (p.nblk_g % NB || total <= 0 || total > (1ll << 30)) return hipErrorInvalidValue;
    hipLaunchKernelGGL((conv1x1_ring_split<WC, WP, CF, PF>), dim3((unsigned)total), dim3(WC * WP * 64), 0, s, p);
    return hipGetLastError();
}

template <int KH, int KW, int S, bool TR, int WC, int WP, int CF, int PF, int TS, int NHB, int RW>
hipError_t go_split(const ConvParams& p0, hipStream_t s) {
    constexpr int TY = WP * PF;
    ConvParams p = p0;
    if (p.ntiles != p.groups * p.nblk_g / (WC * CF) || p.nblk_g % (WC * CF) || p.N < 1 || p.N > MAXB)
        return hipErrorInvalidValue;
    p.gx = ((TR ? (p.OW + 1) / 2 : p.OW) + 15) / 16;
    p.gy = ((TR ? (p.OH + 1) / 2 : p.OH) + TY - 1) / TY;
    const long long total = (long long)p.gx * p.gy * p.N * p.ntiles * (TR ? 4 : 1);
    if (total <= 0 || total > (1ll << 30)) return hipErrorInvalidValue;
    hipLaunchKernelGGL((conv_igemm_split<KH, KW, S, TR, WC, WP, CF, PF, TS, NHB, RW>), dim3((unsigned)total),
                       dim3(WC * WP * 64), 0, s, p);
    return hipGetLastError();
}

}  // namespace

// Instantiated shapes per kind: (wc, wp, cf, pf), taps per weight slot, halo buffers, slots.
#define ZJAI_SPLIT(KIND, KH, KW, S, A, B, C, D, TS, NHB, RW) \
    if (kind == KIND && c.wc == A && c.wp == B && c.cf == C && c.pf == D) return go_split<KH, KW, S, KIND == CK_T3, A, B, C, D, TS, NHB, RW>(p, s);

hipError_t launch_conv_split(int kind, TileCfg c, const ConvParams& p, hipStream_t s) {
    ZJAI_SPLIT(CK_1x1, 1, 1, 1, 1, 4, 4, 2, 1, 1, 2)
    ZJAI_SPLIT(CK_1x1, 1, 1, 1, 1, 4, 2, 2, 1, 1, 2)
    ZJAI_SPLIT(CK_1x1, 1, 1, 1, 1, 4, 1, 2, 1, 1, 2)
    ZJAI_SPLIT(CK_3x3, 3, 3, 1, 2, 2, 4, 4, 1, 2, 3)
    ZJAI_SPLIT(CK_3x3, 3, 3, 1, 1, 4, 4, 4, 1, 1, 3)
    ZJAI_SPLIT(CK_3x3, 3, 3, 1, 1, 4, 4, 2, 3, 1, 2)
    ZJAI_SPLIT(CK_3x3, 3, 3, 1, 1, 4, 2, 2, 3, 1, 2)
    ZJAI_SPLIT(CK_3x3, 3, 3, 1, 1, 4, 1, 2, 9, 1, 2)
    ZJAI_SPLIT(CK_3x3, 3, 3, 1, 1, 8, 1, 1, 9, 1, 2)
    ZJAI_SPLIT(CK_3x3_S2, 3, 3, 2, 2, 2, 4, 2, 1, 1, 3)
    ZJAI_SPLIT(CK_3x3_S2, 3, 3, 2, 1, 4, 4, 2, 1, 1, 2)
    ZJAI_SPLIT(CK_3x3_S2, 3, 3, 2, 1, 4, 4, 1, 3, 1, 2)
    ZJAI_SPLIT(CK_3x3_S2, 3, 3, 2, 1, 4, 2, 1, 3, 1, 2)
    ZJAI_SPLIT(CK_3x3_S2, 3, 3, 2, 1, 8, 1, 1, 3, 1, 2)
    ZJAI_SPLIT(CK_3x3_S2, 3, 3, 2, 1, 4, 1, 1, 9, 1, 2)
    ZJAI_SPLIT(CK_2x2, 2, 2, 1, 1, 4, 4, 2, 1, 1, 3)
    ZJAI_SPLIT(CK_2x2, 2, 2, 1, 1, 8, 2, 1, 4, 1, 2)
    ZJAI_SPLIT(CK_2x2, 2, 2, 1, 1, 4, 1, 2, 4, 1, 2)
    ZJAI_SPLIT(CK_2x2, 2, 2, 1, 1, 8, 1, 1, 4, 1, 2)
    ZJAI_SPLIT(CK_T3, 3, 3, 1, 1, 4, 4, 2, 4, 1, 2)
    ZJAI_SPLIT(CK_T3, 3, 3, 1, 1, 8, 2, 1, 4, 1, 2)
    ZJAI_SPLIT(CK_T3, 3, 3, 1, 1, 8, 1, 1, 4, 1, 2)
    return hipErrorInvalidValue;
}

bool conv1x1_ring_split_ok(const ConvParams& p) {
    auto al = [](const View& v) { return !(v.cs % 4) && !(v.c_off % 4) && !(v.row % 4) && !(v.bstride % 4); };
    return p.groups == 1 && p.N >= 1 && p.N <= MAXB && !p.relu6_in && p.H == p.OH && p.W == p.OW && p.pad_t == 0 &&
           p.pad_l == 0 && al(p.x) && (p.out_mode != OUT_NHWC || al(p.y)) && (!p.r1.p || al(p.r1)) && (!p.r2.p || al(p.r2));
}

hipError_t launch_conv1x1_ring_split(TileCfg c, const ConvParams& p, hipStream_t s) {
    if (!conv1x1_ring_split_ok(p)) return hipErrorInvalidValue;
#define ZJAI_1X1(A, B, C, D) \
    if (c.wc == A && c.wp == B && c.cf == C && c.pf == D) return go_1x1_split<A, B, C, D>(p, s);
    ZJAI_1X1(1, 4, 4, 2)
    ZJAI_1X1(1, 4, 4, 1)
    ZJAI_1X1(1, 4, 2, 1)
    ZJAI_1X1(1, 4, 1, 1)
#undef ZJAI_1X1
    return hipErrorInvalidValue;
}

bool conv_tr_merged_split_ok(const ConvParams& p) {
    // The 3x3 / padding-1 tap table (conv_tr_merged_split's constants, offsets from the input row).
    static const int n[4] = {1, 2, 2, 4};
    static const int dy[4][4] = {{1}, {1, 1}, {2, 1}, {2, 2, 1, 1}}, dx[4][4] = {{1}, {2, 1}, {1, 1}, {2, 1, 2, 1}};
    for (int ph = 0; ph < 4; ++ph) {
        if (p.ntaps[ph] != n[ph]) return false;
        for (int t = 0; t < n[ph]; ++t)
            if (p.tap_dy[ph][t] != dy[ph][t] || p.tap_dx[ph][t] != dx[ph][t]) return false;
    }
    return p.groups == 1 && p.nblk_g % TR_MERGED_NB == 0 && p.N >= 1 && p.N <= MAXB && p.out_mode == OUT_NHWC && p.ps == 1 &&
           !p.relu6_in && !p.w_bstride;
}

hipError_t launch_conv_tr_merged_split(const ConvParams& p0, hipStream_t s) {
    if (!conv_tr_merged_split_ok(p0)) return hipErrorInvalidValue;
    ConvParams p = p0;
    p.ntiles = p.nblk_g / TR_MERGED_NB;
    p.gx = ((p.OW + 1) / 2 + 15) / 16;
    p.gy = ((p.OH + 1) / 2 + 3) / 4;
    const long long total = (long long)p.gx * p.gy * p.N * p.ntiles;
    if (total <= 0 || total > (1ll << 30)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(conv_tr_merged_split, dim3((unsigned)total), dim3(256), 0, s, p);
    return hipGetLastError();
}

}  // namespace zjai
