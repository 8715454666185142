// Convolution forward and stride-1 data gradient on split bf16 operands, 32 channels a step (conv_split.h takes 16): the same tiles of
// flat pixels, staged runs and split filters, multiplied by v_mfma_f32_16x16x32_bf16.
//
// A loop of nothing but MFMAs on random operands is bound by what the matrix cores draw: it sustains 1.84 PFLOP/s in blocks of 32 x 32 x 16 and 2.10
// in blocks of 16 x 16 x 32, 2.46 either way on zeros. This kernel keeps the pipe busy 55 % of its CUs' time (64 -> 64 @56 batch 32: 798 tiles on 512 places
// leave a CU one workgroup in the second round); a wave stands 45 % of its life behind the other waves' instructions, 25 % at loads and barriers and 3 % at LDS, which is
// active 28 % of the time, eleven of these for bank conflicts. A wave owns 32 channels x 64 pixels as before, as 2 x 4 blocks, and its sums are rounded once per 32 channels instead of 16. The run has one place in LDS
// (two of 32 channels would leave a CU to one workgroup): the next chunk is requested ahead and split in the shadow of the last MFMAs, so that
// only its stores stand between two barriers, and the other workgroup of the CU multiplies meanwhile. Pixel fragments are read two blocks
// ahead, filters a tap ahead, which is 768 clocks of MFMAs.
//
// Against 32 x 32 x 16 (us, filters' launch and pass): 64 -> 64 @56 batch 32 55.6 -> 51.1, 128 -> 128 @28 50.2 -> 46.9, 32 -> 32 @48 20.0 -> 18.4, 28 -> 229
// @44x41 batch 17 36.0 -> 33.1; steps alone, two workgroups on every CU, 0.64 -> 0.59 a tap and 16 channels; distance from float64 the same. On a CU
// by itself a workgroup is bound by its chain of loads, barriers and MFMAs and no faster (conv_split_plan_for). Channels are padded to 32, so 48 or
// 80 of them stay on 16.
#pragma once
#include "conv_split.h"

namespace crb {

// WM x WN waves of 32 channels x 64 pixels each.
template <int WM_, int WN_, int MAXPX_>
struct ConvWideCfg {
    static constexpr int F = 3, FH = F, FW = F, S = 1, WM = WM_, WN = WN_, MAXPX = MAXPX_;
    static constexpr int NT = F * F, CI = 32, KG = 1, KO = CI / 8, NTH = 64 * WM * WN;
    static constexpr int OCT = 32 * WM, PXT = 64 * WN;
    static constexpr int PART = KO * MAXPX * 16, STAGE = kSplit * PART;  // bytes
    static constexpr int NP = KO * MAXPX / NTH;
    static_assert(KO * MAXPX % NTH == 0, "whole staging items per thread");
    static constexpr bool EARLY = NP <= 4;  // there are registers for the parts of a chunk before their place is free
    static constexpr u32 STEP = 2 * kSplit * 1024;  // bytes of a tap's fragments: 32 output channels x 32 channels
};

// Filters -> fragments: [output block of 32][chunk of 32][tap][half of the block][part] of 1 KB (lane l: output channel l % 16 of the half,
// channels 8 * (l / 16) + 0..7 of the chunk), zero beyond the channel counts.
template <bool DGRAD, bool SUM = false>
__global__ void __launch_bounds__(256) conv_wide_filters_kernel(const float *__restrict__ W, unsigned char *__restrict__ Wf, u32 C_IN, u32 C_OUT,
                                                                u32 NT, u32 chunks, u32 total, PendingSum sum) {
    if constexpr (SUM) {
        __shared__ __attribute__((aligned(16))) float red[kPendingSumFloats];
        if (blockIdx.x < sum.blocks) {
            pending_sum_block(sum, blockIdx.x, red);
            return;
        }
    }
    const u32 t = (blockIdx.x - (SUM ? sum.blocks : 0)) * 256 + threadIdx.x;
    if (t >= total) return;
    const u32 lane = t & 63, frag = t >> 6, half = frag & 1, step = frag >> 1;  // fragments in memory order
    const u32 tap = step % NT, rest = step / NT, ch = rest % chunks, ob = rest / chunks;
    const u32 oc = ob * 32 + half * 16 + (lane & 15), ic0 = ch * 32 + 8 * (lane >> 4);
    float w[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const u32 ic = ic0 + j;
        const bool ok = oc < C_OUT && ic < C_IN;
        // forward: W[oc][ic][tap]; data gradient: the filters are stored [C_IN (dY channels)][C_OUT][tap] and mirrored
        const float v = W[ok ? (DGRAD ? (size_t(ic) * C_OUT + oc) * NT + NT - 1 - tap : (size_t(oc) * C_IN + ic) * NT + tap) : 0];
        w[j] = ok ? v : 0.f;
    }
    u32x4 part[kSplit];
    split8(w, part);
    unsigned char *dst = Wf + size_t(frag) * (kSplit * 1024) + lane * 16;
#pragma unroll
    for (int p = 0; p < kSplit; ++p) *reinterpret_cast<u32x4 *>(dst + p * 1024) = part[p];
}

// PLAIN: for calls that no scratch can be had for (conv_split.h): every wave splits the filters as it reads them, slices are launched one
// after the other and add to Y. The same bits.
template <class C, bool PLAIN = false>
__global__ void __launch_bounds__(C::NTH, 2) conv_wide_kernel(ConvSplitArgs a) {
    constexpr int NT = C::NT, FW = C::FW, S = C::S, MAXPX = C::MAXPX;
    __shared__ __attribute__((aligned(16))) unsigned char smem[C::STAGE];
    // an XCD gets a contiguous run of tiles, the output-channel tiles of a pixel tile behind one another: they share X in its L2
    const u32 ntile = a.px_tiles * a.oc_tiles, q8 = ntile / kXcds, r8 = ntile % kXcds, xcd = blockIdx.x % kXcds, slice = blockIdx.z;
    const u32 tile = xcd * q8 + (xcd < r8 ? xcd : r8) + blockIdx.x / kXcds;
    const u32 pt = tile / a.oc_tiles, ot = tile % a.oc_tiles;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wave_m = wave / C::WN, wave_n = wave % C::WN, c16 = lane & 15, g4 = lane >> 4;

    // ---- the pixels and the staged run of padded rows --------------------------------------------------------------------
    const u32 p0 = pt * C::PXT, p1 = (p0 + C::PXT < a.npix ? p0 + C::PXT : a.npix) - 1;
    u32 n0, r0, y0, n1, r1, y1;
    a.ohw.divmod(p0, n0, r0);
    y0 = a.ow.div(r0);
    a.ohw.divmod(p1, n1, r1);
    y1 = a.ow.div(r1);
    const u32 R0 = n0 * a.prow + S * y0, wpx = (n1 * a.prow + S * y1 + C::FH - R0) * a.pitch;
    auto pixel = [&](int ni) {  // (past the last: the last one)
        const u32 p = p0 + wave_n * 64 + ni * 16 + c16;
        return p < a.npix ? p : a.npix - 1;
    };
    u32 b_lane[4];  // LDS byte of the pixel's first tap, this lane's channel octet
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) {
        u32 n, r, y, x;
        a.ohw.divmod(pixel(ni), n, r);
        a.ow.divmod(r, y, x);
        b_lane[ni] = ((n * a.prow + S * y - R0) * a.pitch + S * x) * 16 + g4 * (MAXPX * 16);
    }
    // staging: item i of a thread is the channel octet o of position s
    const u32 img0 = a.strip_d.div(n0);  // (n0, n: strips of all images, counted through)
    const BufferRange xrange = buffer_range(a.X + size_t(img0) * a.C_IN * a.HW, (size_t(a.images) - img0) * a.C_IN * a.HW);
    u32 off[C::NP];  // bytes from the chunk's first channel of image img0 (the host checks that they fit)
#pragma unroll
    for (int i = 0; i < C::NP; ++i) {
        const u32 u = threadIdx.x + i * C::NTH, o = u / MAXPX, s = u % MAXPX;
        u32 pr, pc, n, r;
        a.pitch_d.divmod(s, pr, pc);
        a.prow_d.divmod(R0 + pr, n, r);
        u32 img, strip;
        a.strip_d.divmod(n, img, strip);
        const int iy = int(r) - a.pad_y, ix = int(pc + S * strip * a.SW) - a.pad_x;
        const bool in = s < wpx && u32(iy) < a.H && u32(ix) < a.W;
        const u32 bytes = ((img - img0) * a.C_IN * a.HW + 8 * o * a.HW + u32(iy) * a.W + u32(ix)) * 4u;
        off[i] = in ? bytes : kOutside;
    }
    float reg[C::NP][8];
    u32x4 parts[C::EARLY ? C::NP : 1][kSplit];
    const bool ragged = a.C_IN % C::CI != 0;
    const u32 chunk0 = (slice + (PLAIN ? a.z0 : 0u)) * a.chunks_z, chunk1 = chunk0 + a.chunks_z < a.chunks ? chunk0 + a.chunks_z : a.chunks;
    auto fetch = [&](u32 chunk) {
        const u32 c0 = chunk * C::CI;
        if (ragged && chunk + 1 == a.chunks) {
#pragma unroll
            for (int i = 0; i < C::NP; ++i) {
                const u32 o = (threadIdx.x + i * C::NTH) / MAXPX;
#pragma unroll
                for (int j = 0; j < 8; ++j) {  // (channels past the last: kOutside, at an offset the range holds)
                    const u32 ch = c0 + j < a.C_IN ? c0 + j : a.C_IN - 1;
                    reg[i][j] = buffer_load(xrange, c0 + 8 * o + j < a.C_IN ? off[i] : kOutside, ch * a.HW * 4u);
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int i = 0; i < C::NP; ++i) reg[i][j] = buffer_load(xrange, off[i], (c0 + j) * a.HW * 4u);
        }
    };
    auto split_items = [&]() {
        if constexpr (C::EARLY)
#pragma unroll
            for (int i = 0; i < C::NP; ++i) split8(reg[i], parts[i]);
    };
    auto commit = [&]() {  // (positions behind the run are written too; nothing reads them)
#pragma unroll
        for (int i = 0; i < C::NP; ++i) {
            const u32 u = threadIdx.x + i * C::NTH, o = u / MAXPX, s = u % MAXPX;
            u32x4(&part)[kSplit] = parts[C::EARLY ? i : 0];
            if constexpr (!C::EARLY) split8(reg[i], part);
#pragma unroll
            for (int p = 0; p < kSplit; ++p) *reinterpret_cast<u32x4 *>(smem + p * C::PART + o * (MAXPX * 16) + s * 16) = part[p];
        }
    };

    // ---- filters: this wave's blocks, one tap after the other ---------------------------------------------------------------
    const unsigned char *wp = a.Wf + (size_t(ot * C::WM + wave_m) * a.chunks + chunk0) * NT * C::STEP;
    u32 plain_step = chunk0 * NT;
    bf16x8 fa[2][2][kSplit];
    auto load_filters = [&](int set, int mi) {  // half mi of the next step's fragments (behind the last step: padding at the buffer's end)
        if constexpr (PLAIN) {
            const u32 tap = plain_step % NT, ic0 = (plain_step / NT) * C::CI + 8 * g4, oc = ot * C::OCT + wave_m * 32 + mi * 16 + c16;
            float w[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const bool ok = oc < a.C_OUT && ic0 + j < a.C_IN;
                const float v = a.Wt[ok ? size_t(oc) * a.w_oc + size_t(ic0 + j) * a.w_ic + a.w_tap(tap, FW) : 0];
                w[j] = ok ? v : 0.f;
            }
            u32x4 part[kSplit];
            split8(w, part);
#pragma unroll
            for (int p = 0; p < kSplit; ++p) fa[set][mi][p] = __builtin_bit_cast(bf16x8, part[p]);
            plain_step += mi;
        } else {
#pragma unroll
            for (int p = 0; p < kSplit; ++p) fa[set][mi][p] = *reinterpret_cast<const bf16x8 *>(wp + (mi * kSplit + p) * 1024 + u32(lane) * 16u);
            wp += mi * C::STEP;
        }
    };

    v4f acc[2][4], small[2][4];  // sums of the leading part products and of the others (split_bf16.h)
#pragma unroll
    for (int mi = 0; mi < 2; ++mi)
#pragma unroll
        for (int ni = 0; ni < 4; ++ni)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[mi][ni][r] = small[mi][ni][r] = 0.0f;

    constexpr int NG = 4 * NT;  // groups of twelve MFMAs of a chunk: 16 pixels of a tap
    bf16x8 fb[3][kSplit];
    auto read_pixels = [&](int g) {
        const u32 at = b_lane[g % 4] + (g / 4 / FW * a.pitch + g / 4 % FW) * 16;
#pragma unroll
        for (int p = 0; p < kSplit; ++p) fb[g % 3][p] = *reinterpret_cast<const bf16x8 *>(smem + at + p * C::PART);
    };

    fetch(chunk0);
    load_filters(0, 0), load_filters(0, 1);
    split_items();
    commit();
    lds_barrier();
    for (u32 chunk = chunk0; chunk < chunk1; ++chunk) {
        if (chunk + 1 < chunk1) fetch(chunk + 1);
        read_pixels(0), read_pixels(1);
        // The scheduler is fenced group by group: left alone it sinks the requests made for later ones to where they are used.
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int tap = g / 4, ni = g % 4;
            __builtin_amdgcn_sched_barrier(0);
            if (ni < 2) load_filters((tap + 1) % 2, ni);
            if (g + 2 < NG) read_pixels(g + 2);
            if (g == NG - 3) split_items();  // (behind the last chunk: once more, for nobody)
#pragma unroll
            for (int t = 0; t < kTerms; ++t)
#pragma unroll
                for (int mi = 0; mi < 2; ++mi) {
                    v4f &sum = t + 1 < kTerms ? small[mi][ni] : acc[mi][ni];
                    sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[tap % 2][mi][kTermA[t]], fb[g % 3][kTermB[t]], sum, 0, 0, 0);
                }
#pragma unroll
            for (int i = 0; i < 2 * kTerms; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                if (C::EARLY && g >= NG - 3) __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // the next chunk's first tap is in the other set (F odd)
        static_assert(NT % 2 == 1, "taps of a square filter of odd size");
#pragma unroll
        for (int mi = 0; mi < 2; ++mi)
#pragma unroll
            for (int p = 0; p < kSplit; ++p) fa[0][mi][p] = fa[1][mi][p];
        lds_barrier();
        if (chunk + 1 < chunk1) commit();
        lds_barrier();
    }

    bool bad = false;
#pragma unroll
    for (int mi = 0; mi < 2; ++mi)
#pragma unroll
        for (int ni = 0; ni < 4; ++ni)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                acc[mi][ni][r] = (acc[mi][ni][r] + small[mi][ni][r]) * kSplitDown;
                bad |= !__builtin_isfinite(acc[mi][ni][r]);
            }
    // ---- sums that are not finite: this wave's blocks once more, on the fp32 MFMA from the fp32 operands (split_bf16.h) ------
    // Four channels of a tap per MFMA, 32 a step. Taps outside the image take no part (an infinite filter element would make NaN of the zero
    // read there): a lane's accumulators all belong to its pixel, so it keeps the old ones. Ends early where every sum is a NaN.
    if (__builtin_expect(__any(int(bad)), 0)) {
        struct Step {
            float w[8][2], x[8][4];
            bool in[4];
        };
        int py[4], px[4];
        u32 img_off[4];
#pragma unroll
        for (int ni = 0; ni < 4; ++ni) {
            u32 v, r, y, x, img, strip;
            a.ohw.divmod(pixel(ni), v, r);
            a.ow.divmod(r, y, x);
            a.strip_d.divmod(v, img, strip);
            py[ni] = int(S * y) - a.pad_y, px[ni] = int(S * (x + strip * a.SW)) - a.pad_x, img_off[ni] = (img - img0) * a.C_IN * a.HW;
        }
        const float *wrow[2];
#pragma unroll
        for (int mi = 0; mi < 2; ++mi) {
            const u32 oc = ot * C::OCT + wave_m * 32 + mi * 16 + c16;
            wrow[mi] = a.Wt + size_t(oc < a.C_OUT ? oc : a.C_OUT - 1) * a.w_oc;
        }
        auto fetch_step = [&](u32 s, Step &f) {
            const u32 tap = s % NT, c0 = (chunk0 + s / NT) * C::CI + g4;
#pragma unroll
            for (int ni = 0; ni < 4; ++ni) {
                const int iy = py[ni] + int(tap / FW), ix = px[ni] + int(tap % FW);
                f.in[ni] = u32(iy) < a.H && u32(ix) < a.W;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const u32 ic = c0 + 4 * j, bytes = (img_off[ni] + ic * a.HW + u32(iy) * a.W + u32(ix)) * 4u;
                    f.x[j][ni] = buffer_load(xrange, f.in[ni] && ic < a.C_IN ? bytes : kOutside, 0);
                }
            }
#pragma unroll
            for (int mi = 0; mi < 2; ++mi)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const u32 ic = c0 + 4 * j;
                    const float w = wrow[mi][ic < a.C_IN ? size_t(ic) * a.w_ic + a.w_tap(tap, FW) : 0];
                    f.w[j][mi] = ic < a.C_IN ? w : 0.f;
                }
        };
        const u32 count = (chunk1 - chunk0) * NT;
        Step next;
        fetch_step(0, next);
#pragma unroll
        for (int mi = 0; mi < 2; ++mi)
#pragma unroll
            for (int ni = 0; ni < 4; ++ni)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[mi][ni][r] = 0.0f;
#pragma unroll 1
        for (u32 s = 0; s < count; ++s) {
            const Step now = next;
            if (s + 1 < count) fetch_step(s + 1, next);
            u32 numbers = 0;
#pragma unroll
            for (int mi = 0; mi < 2; ++mi)
#pragma unroll
                for (int ni = 0; ni < 4; ++ni) {
                    v4f sum = acc[mi][ni];
#pragma unroll
                    for (int j = 0; j < 8; ++j) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(now.w[j][mi], now.x[j][ni], sum, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        acc[mi][ni][r] = now.in[ni] ? sum[r] : acc[mi][ni][r];
                        numbers |= __builtin_isnan(acc[mi][ni][r]) ? 0u : 1u;
                    }
                }
            if (!__any(int(numbers))) break;
        }
    }

    // ---- epilogue: 16 lanes store 16 consecutive pixels of a channel --------------------------------------------------------
    float bias[2][4];
#pragma unroll
    for (int mi = 0; mi < 2; ++mi)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const u32 oc = ot * C::OCT + wave_m * 32 + mi * 16 + 4 * g4 + r;
            bias[mi][r] = a.bias ? a.bias[oc < a.C_OUT ? oc : a.C_OUT - 1] : 0.f;
        }
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) {
        const u32 p = p0 + wave_n * 64 + ni * 16 + c16;
        u32 v, rem, img, strip, yy, xx;
        a.ohw.divmod(p, v, rem);
        a.ow.divmod(rem, yy, xx);
        a.strip_d.divmod(v, img, strip);
        xx += strip * a.SW;
        if (p >= a.npix || xx >= a.OW) continue;
        float *y = a.Y + slice * a.zstride + size_t(img) * a.C_OUT * a.OHW + yy * a.OW + xx;
#pragma unroll
        for (int mi = 0; mi < 2; ++mi)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const u32 oc = ot * C::OCT + wave_m * 32 + mi * 16 + 4 * g4 + r;
                float o = acc[mi][ni][r];
                if constexpr (PLAIN) {
                    if (a.add && oc < a.C_OUT) o = y[size_t(oc) * a.OHW] + o;
                }
                o += bias[mi][r];
                if (a.relu) o = o > 0.f ? o : 0.f;
                if (oc < a.C_OUT) y[size_t(oc) * a.OHW] = o;
            }
    }
}

template <class C>
inline size_t conv_wide_filter_bytes(u32 C_IN, u32 C_OUT) {  // (a tap more: filters are read one ahead)
    return (size_t(ceil_div(C_OUT, u32(C::OCT)) * C::WM) * ceil_div(C_IN, u32(C::CI)) * C::NT + 1) * C::STEP;
}

// As launch_conv_split.
template <class C, bool DGRAD>
inline int launch_conv_wide(const float *Wt, const float *X, float *Y, const float *bias, unsigned char *Wf, u32 N, u32 C_IN, u32 C_OUT, u32 H,
                            u32 W, u32 OH, u32 OW, u32 strips, u32 slices, float *part, int pad_y, int pad_x, u32 relu, hipStream_t s,
                            const char *what, const PendingSum *sum) {
    ConvSplitArgs a = conv_split_args<C>(Wt, X, Y, bias, Wf, N, C_IN, C_OUT, H, W, OH, OW, strips, slices, pad_y, pad_x);
    a.w_oc = DGRAD ? C::NT : C_IN * C::NT, a.w_ic = DGRAD ? C_OUT * C::NT : C::NT;
    a.tap0 = DGRAD ? C::NT - 1 : 0, a.tap_i = DGRAD ? -C::FW : C::FW, a.tap_j = DGRAD ? -1 : 1;
    a.relu = relu;
    if (slices > 1) a.Y = part, a.bias = nullptr, a.relu = 0;
    const u32 count = N * C_OUT * OH * OW;
    a.zstride = count;
    const uint64_t tiles = uint64_t(a.px_tiles) * a.oc_tiles;
    if (tiles > 0x7fffffffull) return fail(CRB_EINVAL_SHAPE, "%s: launch grid too large", what);
    if (!Wf) {
        a.Y = Y, a.zstride = 0;
        for (u32 z = 0; z < slices; ++z) {
            a.z0 = z, a.add = z > 0;
            if (z + 1 == slices) a.bias = bias, a.relu = relu;
            hipLaunchKernelGGL((conv_wide_kernel<C, true>), dim3(u32(tiles)), dim3(C::NTH), 0, s, a);
            if (int st = check_launch(what)) return st;
        }
        return CRB_OK;
    }
    const u32 total = a.oc_tiles * C::WM * a.chunks * C::NT * 128;
    if (DGRAD && sum)
        hipLaunchKernelGGL((conv_wide_filters_kernel<DGRAD, DGRAD>), dim3(sum->blocks + ceil_div(total, 256u)), dim3(256), 0, s, Wt, Wf, C_IN, C_OUT, u32(C::NT),
                           a.chunks, total, *sum);
    else
        hipLaunchKernelGGL(conv_wide_filters_kernel<DGRAD>, dim3(ceil_div(total, 256u)), dim3(256), 0, s, Wt, Wf, C_IN, C_OUT, u32(C::NT), a.chunks, total, PendingSum());
    if (int st = check_launch(what)) return st;
    hipLaunchKernelGGL((conv_wide_kernel<C>), dim3(u32(tiles), 1, slices), dim3(C::NTH), 0, s, a);
    int st = check_launch(what);
    if (st == CRB_OK && slices > 1) st = launch_ordered_reduce(part, Y, count, slices, ReduceEpi{bias, OH * OW, C_OUT, relu ? u32(EPI_RELU) : 0u}, s, what);
    return st;
}

}  // namespace crb
