// Convolution forward (stride S) and data gradient (stride 1; stride 2 by residue classes, below) on split bf16 operands (split_bf16.h), any image extent and any
// padding: Y[n][oc][y][x] = sum over (ic, fh, fw) of W[oc][ic][fh][fw] * X[n][ic][S*y + fh - pad][S*x + fw - pad]; the data
// gradient is the same with dY as X, the filters' channel roles swapped and their taps mirrored.
//
// Pixels are taken flat: images are cut into `strips` column strips of equal width (one where the image is narrow enough), and a
// workgroup owns PXT consecutive pixels of the (image, strip, row, column) sequence and OCT output channels, so hardly any image
// extent wastes a tile. What the taps of those pixels touch is a run of rows of the padded strips (S*(H-1)+F rows and
// S*(SW-1)+F columns each, halo included): CI = 16*KG channels of it at a time are staged in LDS as MFMA fragments, [part]
// [channel octet][position] units of 16 bytes, double-buffered. A tap is then a constant shift of a lane's position, whatever
// the width, and a B fragment (32 pixels, 16 channels) is one 16-byte read at lane base + shift.
// Filters are split by a kernel of their own into fragments in the order the waves consume them (conv_split_filters_kernel) and
// go from L2 straight into registers, two or four taps ahead: a filter element is used once per workgroup tile, so LDS would only add
// a copy, and without them a barrier stands only every F*F taps.
// KG wave groups take 16 channels each of every staged chunk and exchange their accumulators through LDS at the end.
//
// What bounds it: per tap a wave issues 6*TM*TN MFMAs (32 clocks each) against 3*TM KB of filters from L2 and 3*TN KB from LDS: with
// the 1 x 2 blocks of every configuration and eight waves on a CU 768 clocks of MFMAs on each SIMD against 384 of the vector
// memory path (64 bytes a clock) and 384 of LDS (128), so the MFMAs, between a first and a last phase that they do not fill.
#pragma once
#include "igemm_engine.h"
#include "split_bf16.h"

namespace crb {

template <int FH_, int FW_, int S_, int TM_, int TN_, int WM_, int WN_, int KG_, int MAXPX_, int AHEAD_ = 2, int BSET_ = 2, int NBUF_ = 2>
struct ConvSplitRect {
    static constexpr int FH = FH_, FW = FW_, S = S_, TM = TM_, TN = TN_, WM = WM_, WN = WN_, KG = KG_, MAXPX = MAXPX_;
    static constexpr int NT = FH * FW, CI = 16 * KG, KO = CI / 8, NTH = 64 * WM * WN * KG;
    static constexpr int OCT = 32 * TM * WM, PXT = 32 * TN * WN;
    static constexpr int PART = KO * MAXPX * 16, STAGE = kSplit * PART;  // bytes
    static constexpr int NP = KO * MAXPX / NTH;
    static_assert(KO * MAXPX % NTH == 0, "whole staging items per thread");
    static constexpr int AHEAD = AHEAD_;  // taps the filter fragments run ahead
    static constexpr int BSET = BSET_;    // 2: pixel fragments are read a tap ahead
    // 1: the run has one place in LDS and the next chunk takes it between two barriers. The run of a strided 5x5 tile is large, its
    // 25 taps per chunk many; two or three workgroups then share a CU, which two places would leave to one (96 KB).
    static constexpr int NBUF = NBUF_;
    // LDS of a chunk's filter fragments (16 bytes between two: the taps of a channel then start in different banks): residue classes, PLAIN
    static constexpr int FRAG = kSplit * 1024 + 16, FILTERS = NT * (OCT / 32) * FRAG;
};

template <int F_, int S_, int TM_, int TN_, int WM_, int WN_, int KG_, int MAXPX_, int AHEAD_ = 2, int BSET_ = 2, int NBUF_ = 2>
struct ConvSplitCfg : ConvSplitRect<F_, F_, S_, TM_, TN_, WM_, WN_, KG_, MAXPX_, AHEAD_, BSET_, NBUF_> {
    static constexpr int F = F_;
};

struct ConvSplitArgs {
    const float *X;
    const unsigned char *Wf;  // split filters
    const float *Wt;          // the filters: element (output channel, input channel, tap (i, j)) at oc * w_oc + ic * w_ic + tap0 + i * tap_i + j * tap_j
    u32 w_oc, w_ic;
    int tap0, tap_i, tap_j;
    float *Y;
    const float *bias;
    u32 C_IN, C_OUT, chunks;
    u32 images, H, W;  // of X
    u32 HW, OHW;     // pixels of an image of X, of Y
    u32 OW, SW, strips;  // width of Y, of a strip
    u32 npix;        // pixels of all strips (those past the image's last column are computed and dropped)
    u32 prow, pitch; // padded rows of a strip, positions of a padded row
    int pad_y, pad_x;
    u32 px_tiles, oc_tiles, relu;
    u32 chunks_z;    // chunks a slice (blockIdx.z) of the contraction takes; slices write partial results `zstride` floats apart
    size_t zstride;
    u32 z0, add;     // (PLAIN) the slice that blockIdx.z == 0 takes, and whether it adds to Y
    FastDiv ohw, ow, pitch_d, prow_d, strip_d;  // pixels of a strip, its width, ...
    u32 osy, osx, oy0, ox0, out_w;  // (SCATTER) pixel (y, x) of the grid is (osy*y + oy0, osx*x + ox0) of a result `out_w` wide, OHW its pixels
    __device__ __forceinline__ u32 w_tap(u32 tap, u32 fw) const { return u32(tap0 + int(tap / fw) * tap_i + int(tap % fw) * tap_j); }
};

// Filters -> fragments: [output block of 32][K group][chunk][tap][part] of 1 KB (lane l: output channel l % 32 of the block,
// channels 8 * (l / 32) + 0..7 of the group's 16), zero beyond the channel counts. A thread takes one channel octet of one
// output channel and tap: eight loads in flight, and enough threads to cover the chip (all taps per thread: 147 K filter
// elements took 14 us, a chain of 72 loads on 8 workgroups).
// SUM: the first workgroups sum a weight gradient's slices (of the call's other gradient): one launch for two that the chip is not filled by.
template <bool DGRAD, bool SUM = false>
__global__ void __launch_bounds__(256) conv_split_filters_kernel(const float *__restrict__ W, unsigned char *__restrict__ Wf, u32 C_IN, u32 C_OUT,
                                                                 u32 NT, u32 chunks, u32 KG, u32 total, PendingSum sum) {
    if constexpr (SUM) {
        __shared__ __attribute__((aligned(16))) float red[kPendingSumFloats];
        if (blockIdx.x < sum.blocks) {
            pending_sum_block(sum, blockIdx.x, red);
            return;
        }
    }
    const u32 t = (blockIdx.x - (SUM ? sum.blocks : 0)) * 256 + threadIdx.x;
    if (t >= total) return;
    const u32 lane = t & 63, frag = t >> 6;  // fragments in memory order
    const u32 tap = frag % NT, rest = frag / NT;
    const u32 ch = rest % chunks, g = (rest / chunks) % KG, ob = rest / (chunks * KG);
    const u32 oc = ob * 32 + (lane & 31), ic0 = (ch * KG + g) * 16 + 8 * (lane >> 5);
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

// PLAIN: for calls that no scratch can be had for. Slices of the contraction are launched one after the other, each adding to Y, and every
// workgroup splits the filters itself: the same bits, several times the time where each wave splits a tap's as it reads them, a lane's
// eight channels from eight places. The residue classes (SCATTER), behind which kernels stand that need no scratch, have a chunk's filters
// split by all threads, through LDS: lanes read the taps of a channel side by side, for the next chunk while one is multiplied. 699 random
// layers take 0.70 of the fp32 class kernels' time in the mean, 38 of them more than it, by 1.4 at the most (split as the waves read
// them: 0.93, 211 and 1.7; with scratch 0.57).
// The work of workgroup `bid` of `px_tiles * oc_tiles`, slice `slice` of the launch; `smem`: C::NBUF * C::STAGE bytes, PLAIN and SCATTER: and C::FILTERS.
template <class C, bool PLAIN, bool SCATTER>
__device__ __forceinline__ void conv_split_body(const ConvSplitArgs &a, const u32 bid, const u32 slice, unsigned char *smem) {
    constexpr int TM = C::TM, TN = C::TN, KG = C::KG, NT = C::NT, FH = C::FH, FW = C::FW, S = C::S, MAXPX = C::MAXPX, NSET = C::AHEAD + 1;
    // an XCD gets a contiguous run of tiles, the output-channel tiles of a pixel tile behind one another: they share X in its L2
    const u32 ntile = a.px_tiles * a.oc_tiles, q8 = ntile / kXcds, r8 = ntile % kXcds, xcd = bid % kXcds;
    const u32 tile = xcd * q8 + (xcd < r8 ? xcd : r8) + bid / kXcds;
    const u32 pt = tile / a.oc_tiles, ot = tile % a.oc_tiles;

    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wave = wv % (C::WM * C::WN), kgroup = wv / (C::WM * C::WN);
    const int wave_m = wave / C::WN, wave_n = wave % C::WN, i32 = lane & 31, h = lane >> 5;

    // ---- the pixels and the staged run of padded rows --------------------------------------------------------------------
    const u32 p0 = pt * C::PXT, p1 = (p0 + C::PXT < a.npix ? p0 + C::PXT : a.npix) - 1;
    u32 n0, r0, y0, n1, r1, y1;
    a.ohw.divmod(p0, n0, r0);
    y0 = a.ow.div(r0);
    a.ohw.divmod(p1, n1, r1);
    y1 = a.ow.div(r1);
    const u32 R0 = n0 * a.prow + S * y0, wpx = (n1 * a.prow + S * y1 + FH - R0) * a.pitch;
    u32 b_lane[TN];  // LDS byte of the pixel's first tap, this lane's channel half
#pragma unroll
    for (int ni = 0; ni < TN; ++ni) {
        u32 p = p0 + wave_n * (32 * TN) + ni * 32 + i32;
        p = p < a.npix ? p : a.npix - 1;
        u32 n, r, y, x;
        a.ohw.divmod(p, n, r);
        a.ow.divmod(r, y, x);
        b_lane[ni] = ((n * a.prow + S * y - R0) * a.pitch + S * x) * 16 + (2 * kgroup + h) * (MAXPX * 16);
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
    auto commit = [&](unsigned char *sm) {  // (positions behind the run are written too; nothing reads them)
#pragma unroll
        for (int i = 0; i < C::NP; ++i) {
            const u32 u = threadIdx.x + i * C::NTH, o = u / MAXPX, s = u % MAXPX;
            u32x4 part[kSplit];
            split8(reg[i], part);
#pragma unroll
            for (int p = 0; p < kSplit; ++p) *reinterpret_cast<u32x4 *>(sm + p * C::PART + o * (MAXPX * 16) + s * 16) = part[p];
        }
    };

    // ---- filters: this wave's blocks, one 3 KB step (tap) after the other ---------------------------------------------------
    const u32 steps = a.chunks * NT;
    const unsigned char *wp[TM];
#pragma unroll
    for (int mi = 0; mi < TM; ++mi)
        wp[mi] = a.Wf + ((size_t(ot * (TM * C::WM) + wave_m * TM + mi) * KG + kgroup) * steps + chunk0 * NT) * (kSplit * 1024);
    bf16x8 fa[NSET][kSplit][TM];
    // ---- a chunk's filter fragments in LDS -----------------------------------------------------------------------------------
    constexpr bool STAGED = PLAIN && SCATTER;
    static_assert(!STAGED || KG == 1, "filters of one K group");
    constexpr int FITEMS = NT * C::OCT * 2, FNP = STAGED ? (FITEMS + C::NTH - 1) / C::NTH : 1;  // channel octets of a chunk, of a thread
    unsigned char *fsm = smem + C::NBUF * C::STAGE;
    const BufferRange wrange = buffer_range(a.Wt, size_t(a.C_IN) * a.w_ic);  // (gradient: channels of dY outermost)
    float freg[FNP][8];
    u32 foff[FNP], fdst[FNP];  // of an item's first element, of its fragment in LDS
    if constexpr (STAGED) {
#pragma unroll
        for (int i = 0; i < FNP; ++i) {
            const u32 e = threadIdx.x + i * C::NTH, tap = e % NT, oc_l = e / NT % C::OCT, o = e / (NT * C::OCT), oc = ot * C::OCT + oc_l;
            foff[i] = e < FITEMS && oc < a.C_OUT ? (oc * a.w_oc + 8 * o * a.w_ic + a.w_tap(tap, FW)) * 4u : kOutside;
            fdst[i] = ((oc_l / 32) * NT + tap) * C::FRAG + (oc_l % 32 + 32 * o) * 16;
        }
    }
    auto fetch_filters = [&](u32 chunk) {
        const u32 c0 = chunk * C::CI;
#pragma unroll
        for (int i = 0; i < FNP; ++i) {
            const u32 o = (threadIdx.x + i * C::NTH) / (NT * C::OCT);
#pragma unroll
            for (int j = 0; j < 8; ++j) {  // (channels past the last: kOutside, at an offset the range holds)
                const u32 ch = c0 + j < a.C_IN ? c0 + j : a.C_IN - 1;
                freg[i][j] = buffer_load(wrange, !ragged || c0 + 8 * o + j < a.C_IN ? foff[i] : kOutside, ch * a.w_ic * 4u);
            }
        }
    };
    auto commit_filters = [&]() {
#pragma unroll
        for (int i = 0; i < FNP; ++i) {
            if (FITEMS % C::NTH != 0 && threadIdx.x + i * C::NTH >= FITEMS) continue;
            u32x4 part[kSplit];
            split8(freg[i], part);
#pragma unroll
            for (int p = 0; p < kSplit; ++p) *reinterpret_cast<u32x4 *>(fsm + fdst[i] + p * 1024) = part[p];
        }
    };
    u32 plain_step = chunk0 * NT;
    auto load_filters = [&](int set) {  // the next step's fragments; STAGED: those of tap `plain_step`
        if constexpr (STAGED) {
#pragma unroll
            for (int mi = 0; mi < TM; ++mi)
#pragma unroll
                for (int p = 0; p < kSplit; ++p)
                    fa[set][p][mi] = *reinterpret_cast<const bf16x8 *>(fsm + ((wave_m * TM + mi) * NT + plain_step) * C::FRAG + p * 1024 + lane * 16);
            return;
        }
        if constexpr (PLAIN) {
            const u32 tap = plain_step % NT, ic0 = (plain_step / NT) * C::CI + 16 * kgroup + 8 * h;
#pragma unroll
            for (int mi = 0; mi < TM; ++mi) {
                const u32 oc = ot * C::OCT + wave_m * (32 * TM) + mi * 32 + i32;
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
                for (int p = 0; p < kSplit; ++p) fa[set][p][mi] = __builtin_bit_cast(bf16x8, part[p]);
            }
            ++plain_step;
            return;
        }
#pragma unroll
        for (int mi = 0; mi < TM; ++mi) {
#pragma unroll
            for (int p = 0; p < kSplit; ++p) fa[set][p][mi] = *reinterpret_cast<const bf16x8 *>(wp[mi] + p * 1024 + u32(lane) * 16u);
            wp[mi] += kSplit * 1024;
        }
    };

    v16f acc[TM][TN], small[TM][TN];  // sums of the leading part products and of the others (split_bf16.h)
#pragma unroll
    for (int mi = 0; mi < TM; ++mi)
#pragma unroll
        for (int ni = 0; ni < TN; ++ni)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mi][ni][r] = small[mi][ni][r] = 0.0f;

    bf16x8 fb[C::BSET][kSplit][TN];
    auto read_pixels = [&](int set, u32 shift) {
#pragma unroll
        for (int p = 0; p < kSplit; ++p)
#pragma unroll
            for (int ni = 0; ni < TN; ++ni) fb[set][p][ni] = *reinterpret_cast<const bf16x8 *>(smem + b_lane[ni] + shift + p * C::PART);
    };

    fetch(chunk0);
    if constexpr (STAGED) {
        fetch_filters(chunk0);
    } else {
#pragma unroll
        for (int d = 0; d < C::AHEAD; ++d) load_filters(d);
    }
    commit(smem);
    lds_barrier();
    u32 buf = 0;
    for (u32 chunk = chunk0; chunk < chunk1; ++chunk, buf = (C::NBUF - 1) * C::STAGE - buf) {
        if (chunk + 1 < chunk1) fetch(chunk + 1);
        if (C::BSET == 2) read_pixels(0, buf);
        // The scheduler is fenced tap by tap: left alone it sinks the requests made for later taps to where they are used.
#pragma unroll
        for (int tap = 0; tap < NT; ++tap) {
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (STAGED) {
                if (tap == 0) {  // (the last readers of the chunk before are behind its barrier)
                    commit_filters();
                    lds_barrier();
                    if (chunk + 1 < chunk1) fetch_filters(chunk + 1);
                    plain_step = 0;
                    load_filters(0);
                }
                plain_step = tap + 1;
                if (tap + 1 < NT) load_filters((tap + 1) % NSET);
            } else {
                load_filters((tap + C::AHEAD) % NSET);  // (behind the last step: padding at the end of the filter buffer)
            }
            constexpr int BS = C::BSET;
            if (BS == 1) read_pixels(0, buf + (tap / FW * a.pitch + tap % FW) * 16);
            else if (tap + 1 < NT) read_pixels((tap + 1) % BS, buf + ((tap + 1) / FW * a.pitch + (tap + 1) % FW) * 16);
            // the next chunk: split and stored in the shadow of the last taps' MFMAs (once more behind the last chunk, for nobody)
            if (C::NBUF == 2 && tap == (NT > 1 ? NT - 2 : 0)) commit(smem + (C::STAGE - buf));
#pragma unroll
            for (int t = 0; t < kTerms; ++t)
#pragma unroll
                for (int mi = 0; mi < TM; ++mi)
#pragma unroll
                    for (int ni = 0; ni < TN; ++ni) {
                        v16f &sum = t + 1 < kTerms ? small[mi][ni] : acc[mi][ni];
                        sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[tap % NSET][kTermA[t]][mi], fb[tap % BS][kTermB[t]][ni], sum, 0, 0, 0);
                    }
#pragma unroll
            for (int i = 0; i < TM * TN * kTerms; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                if (C::NBUF == 2 && tap == (NT > 1 ? NT - 2 : 0)) {
                    __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
                    __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (NT % NSET != 0 && !STAGED) {  // the next chunk's first step is in set NT % NSET
            bf16x8 tmp[NSET][kSplit][TM];
#pragma unroll
            for (int s = 0; s < NSET; ++s)
#pragma unroll
                for (int p = 0; p < kSplit; ++p)
#pragma unroll
                    for (int mi = 0; mi < TM; ++mi) tmp[s][p][mi] = fa[(s + NT) % NSET][p][mi];
#pragma unroll
            for (int s = 0; s < NSET; ++s)
#pragma unroll
                for (int p = 0; p < kSplit; ++p)
#pragma unroll
                    for (int mi = 0; mi < TM; ++mi) fa[s][p][mi] = tmp[s][p][mi];
        }
        lds_barrier();
        if constexpr (C::NBUF == 1) {
            if (chunk + 1 < chunk1) commit(smem);
            lds_barrier();
        }
    }

    // ---- sums that are not finite: this wave's blocks once more, on the fp32 MFMA from the fp32 operands (split_bf16.h) ------
    // Two channels of a tap per MFMA, 16 a step, the next step's operands requested ahead. Taps outside the image take no part
    // (an infinite filter element would make NaN of the zero read there): a lane's accumulators all belong to its pixel, so
    // it keeps the old ones. Ends early where every sum is a NaN.
    add_small(acc, small);
    if (__builtin_expect(__any(int(scale_down(acc))), 0)) {
        struct Step {
            float w[8][TM], x[8][TN];
            bool in[TN];
        };
        int py[TN], px[TN];
        u32 img_off[TN];
        const float *wrow[TM];
#pragma unroll
        for (int ni = 0; ni < TN; ++ni) {
            u32 p = p0 + wave_n * (32 * TN) + ni * 32 + i32;
            p = p < a.npix ? p : a.npix - 1;
            u32 v, r, y, x, img, strip;
            a.ohw.divmod(p, v, r);
            a.ow.divmod(r, y, x);
            a.strip_d.divmod(v, img, strip);
            py[ni] = int(S * y) - a.pad_y, px[ni] = int(S * (x + strip * a.SW)) - a.pad_x, img_off[ni] = (img - img0) * a.C_IN * a.HW;
        }
#pragma unroll
        for (int mi = 0; mi < TM; ++mi) {
            const u32 oc = ot * C::OCT + wave_m * (32 * TM) + mi * 32 + i32;
            wrow[mi] = a.Wt + size_t(oc < a.C_OUT ? oc : a.C_OUT - 1) * a.w_oc;
        }
        auto fetch_step = [&](u32 s, Step &f) {
            const u32 tap = s % NT, c0 = (chunk0 + s / NT) * C::CI + 16 * kgroup;
#pragma unroll
            for (int ni = 0; ni < TN; ++ni) {
                const int iy = py[ni] + int(tap / FW), ix = px[ni] + int(tap % FW);
                f.in[ni] = u32(iy) < a.H && u32(ix) < a.W;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const u32 ic = c0 + 2 * j + h, bytes = (img_off[ni] + ic * a.HW + u32(iy) * a.W + u32(ix)) * 4u;
                    f.x[j][ni] = buffer_load(xrange, f.in[ni] && ic < a.C_IN ? bytes : kOutside, 0);
                }
            }
#pragma unroll
            for (int mi = 0; mi < TM; ++mi)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const u32 ic = c0 + 2 * j + h;
                    const float w = wrow[mi][ic < a.C_IN ? size_t(ic) * a.w_ic + a.w_tap(tap, FW) : 0];
                    f.w[j][mi] = ic < a.C_IN ? w : 0.f;
                }
        };
        const u32 count = (chunk1 - chunk0) * NT;
        Step next;
        fetch_step(0, next);
#pragma unroll
        for (int mi = 0; mi < TM; ++mi)
#pragma unroll
            for (int ni = 0; ni < TN; ++ni)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[mi][ni][r] = 0.0f;
#pragma unroll 1
        for (u32 s = 0; s < count; ++s) {
            const Step now = next;
            if (s + 1 < count) fetch_step(s + 1, next);
            u32 numbers = 0;
#pragma unroll
            for (int mi = 0; mi < TM; ++mi)
#pragma unroll
                for (int ni = 0; ni < TN; ++ni) {
                    v16f sum = acc[mi][ni];
#pragma unroll
                    for (int j = 0; j < 8; ++j) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(now.w[j][mi], now.x[j][ni], sum, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        acc[mi][ni][r] = now.in[ni] ? sum[r] : acc[mi][ni][r];
                        numbers |= __builtin_isnan(acc[mi][ni][r]) ? 0u : 1u;
                    }
                }
            if (!__any(int(numbers))) break;
        }
    }

    // ---- epilogue: 32 lanes store 32 consecutive pixels of a channel --------------------------------------------------------
    auto store_part = [&](int mi, int ni, int r0, auto nr_c, const float *res) {
        constexpr int NR = decltype(nr_c)::value;
        const u32 p = p0 + wave_n * (32 * TN) + ni * 32 + i32;
        const u32 oc0 = ot * C::OCT + wave_m * (32 * TM) + mi * 32 + 4 * h + 2 * r0;
        float b[NR];
#pragma unroll
        for (int r = 0; r < NR; ++r) b[r] = 0.f;
        if (a.bias) {
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const u32 oc = oc0 + 8 * (r / 4) + (r % 4);
                b[r] = a.bias[oc < a.C_OUT ? oc : a.C_OUT - 1];
            }
        }
        u32 v, rem, img, strip, yy, xx;
        a.ohw.divmod(p, v, rem);
        a.ow.divmod(rem, yy, xx);
        a.strip_d.divmod(v, img, strip);
        xx += strip * a.SW;
        if (p >= a.npix || xx >= a.OW) return;
        const u32 at = SCATTER ? (a.osy * yy + a.oy0) * a.out_w + a.osx * xx + a.ox0 : yy * a.OW + xx;
        float *y = a.Y + slice * a.zstride + size_t(img) * a.C_OUT * a.OHW + at;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const u32 oc = oc0 + 8 * (r / 4) + (r % 4);
            float o = res[r];
            if constexpr (PLAIN) {
                if (a.add && oc < a.C_OUT) o = y[size_t(oc) * a.OHW] + o;
            }
            o += b[r];
            if (a.relu) o = o > 0.f ? o : 0.f;
            if (oc < a.C_OUT) y[size_t(oc) * a.OHW] = o;
        }
    };
    if constexpr (KG == 1) {
#pragma unroll
        for (int mi = 0; mi < TM; ++mi)
#pragma unroll
            for (int ni = 0; ni < TN; ++ni) {
                float v[16];
#pragma unroll
                for (int r = 0; r < 16; ++r) v[r] = acc[mi][ni][r];
                store_part(mi, ni, 0, std::integral_constant<int, 16>(), v);
            }
    } else {
        // the K groups exchange their accumulators, BR blocks of every wave at a time; each sums (in group order) and stores a share
        constexpr int NB = TM * TN, BR = NB < KG ? NB : KG, NR = BR * 16 / KG;
        static_assert(NB % BR == 0 && NR % 4 == 0 && BR * 4096 * C::WM * C::WN * KG <= C::NBUF * C::STAGE, "exchange space");
        float *x = reinterpret_cast<float *>(smem);
#pragma unroll
        for (int q = 0; q < NB / BR; ++q) {
            if (q) lds_barrier();
            float *dst = x + (kgroup * C::WM * C::WN + wave) * BR * 1024 + lane;
#pragma unroll
            for (int f = 0; f < BR * 16; ++f) dst[f * 64] = acc[(q * BR + f / 16) / TN][(q * BR + f / 16) % TN][f % 16];
            lds_barrier();
            const int f0 = kgroup * NR;
            float v[NR];
            const float *src = x + wave * BR * 1024 + f0 * 64 + lane;
#pragma unroll
            for (int r = 0; r < NR; ++r) v[r] = src[r * 64];
#pragma unroll
            for (int g = 1; g < KG; ++g)
#pragma unroll
                for (int r = 0; r < NR; ++r) v[r] += src[g * C::WM * C::WN * BR * 1024 + r * 64];
            const int b = q * BR + f0 / 16;
            store_part(b / TN, b % TN, f0 % 16, std::integral_constant<int, NR>(), v);
        }
    }
}

template <class C, bool PLAIN = false>
__global__ void __launch_bounds__(C::NTH, 2) conv_split_kernel(ConvSplitArgs a) {
    __shared__ __attribute__((aligned(16))) unsigned char smem[C::NBUF * C::STAGE];
    conv_split_body<C, PLAIN, false>(a, blockIdx.x, blockIdx.z, smem);
}

// Positions of the longest run of padded rows that a tile of PXT consecutive pixels touches. Tiles start at multiples of PXT, so
// their places inside an image repeat; where that takes long, the bound for any start.
inline u32 conv_split_window(u32 pxt, u32 OH, u32 OW, u32 F, u32 FW, u32 S) {  // F: rows of the filter
    const u32 ohw = OH * OW, prow = S * (OH - 1) + F, pitch = S * (OW - 1) + FW;
    u32 g = pxt, r = ohw;
    while (r) {
        const u32 t = g % r;
        g = r, r = t;
    }
    const u32 period = ohw / g;
    if (period > 64) {
        const u32 rows = (pxt - 2) / OW + 2, crossings = (pxt - 2) / ohw + 1;
        const int gap = int(prow) - int(S * OH);  // padded rows that an image boundary adds
        return (S * (rows - 1) + F + (gap > 0 ? u32(gap) * crossings : 0u)) * pitch;
    }
    u32 most = 0;
    for (u32 k = 0; k < period; ++k) {
        const u32 b = k * pxt % ohw, e = b + pxt - 1;  // first and last pixel, counted from the first one's image
        const u32 rows = e / ohw * prow + S * (e % ohw / OW) + F - S * (b / OW);
        most = rows > most ? rows : most;
    }
    return most * pitch;
}

// Column strips of an output of extent OH x OW for a configuration: the fewest whose run fits its LDS; 0: none does.
template <class C>
inline u32 conv_split_strips(u32 OH, u32 OW) {
    for (u32 ns = ceil_div(OW, 64u); ns <= OW && ns <= 16; ++ns)
        if (conv_split_window(C::PXT, OH, ceil_div(OW, ns), C::FH, C::FW, C::S) <= u32(C::MAXPX)) return ns;
    return 0;
}

template <class C>
inline size_t conv_split_filter_bytes(u32 C_IN, u32 C_OUT) {
    const size_t chunks = ceil_div(C_IN, u32(C::CI)), blocks = ceil_div(C_OUT, u32(C::OCT)) * (C::OCT / 32);
    return (blocks * C::KG * chunks * C::NT + C::AHEAD) * kSplit * 1024;
}

// What does not depend on where the filters and the result lie. (OH, OW): pixel grid, (H, W): extent of X.
template <class C>
inline ConvSplitArgs conv_split_args(const float *Wt, const float *X, float *Y, const float *bias, unsigned char *Wf, u32 N, u32 C_IN, u32 C_OUT, u32 H,
                                     u32 W, u32 OH, u32 OW, u32 strips, u32 slices, int pad_y, int pad_x) {
    ConvSplitArgs a = {};
    a.Wt = Wt, a.X = X, a.Wf = Wf, a.Y = Y, a.bias = bias;
    a.C_IN = C_IN, a.C_OUT = C_OUT, a.chunks = ceil_div(C_IN, u32(C::CI));
    a.strips = strips, a.SW = ceil_div(OW, strips);
    a.images = N, a.H = H, a.W = W, a.HW = H * W, a.OHW = OH * OW, a.OW = OW, a.npix = N * strips * OH * a.SW;
    a.prow = C::S * (OH - 1) + C::FH, a.pitch = C::S * (a.SW - 1) + C::FW;
    a.pad_y = pad_y, a.pad_x = pad_x;
    a.px_tiles = ceil_div(a.npix, u32(C::PXT)), a.oc_tiles = ceil_div(C_OUT, u32(C::OCT));
    a.chunks_z = ceil_div(a.chunks, slices);
    a.ohw.init(OH * a.SW), a.ow.init(a.SW), a.pitch_d.init(a.pitch), a.prow_d.init(a.prow), a.strip_d.init(strips);
    return a;
}

// Wf: conv_split_filter_bytes of scratch, or null (PLAIN). (OH, OW): extent of the result, (H, W): of X; window origin (-pad_y, -pad_x); strips:
// conv_split_strips. slices > 1: the contraction is cut; partial results go to `part` (slices x the result) and are summed in
// fixed order by one more launch, which applies bias and ReLU.
template <class C, bool DGRAD>
inline int launch_conv_split(const float *Wt, const float *X, float *Y, const float *bias, unsigned char *Wf, u32 N, u32 C_IN, u32 C_OUT, u32 H,
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
    const u32 total = a.oc_tiles * (C::OCT / 32) * C::KG * a.chunks * C::NT * 64;
    if (!Wf) {
        a.Y = Y, a.zstride = 0;
        for (u32 z = 0; z < slices; ++z) {
            a.z0 = z, a.add = z > 0;
            if (z + 1 == slices) a.bias = bias, a.relu = relu;
            hipLaunchKernelGGL((conv_split_kernel<C, true>), dim3(u32(tiles)), dim3(C::NTH), 0, s, a);
            if (int st = check_launch(what)) return st;
        }
        return CRB_OK;
    }
    if (DGRAD && sum)
        hipLaunchKernelGGL((conv_split_filters_kernel<DGRAD, DGRAD>), dim3(sum->blocks + ceil_div(total, 256u)), dim3(256), 0, s, Wt, Wf, C_IN, C_OUT, u32(C::NT),
                           a.chunks, u32(C::KG), total, *sum);
    else
        hipLaunchKernelGGL(conv_split_filters_kernel<DGRAD>, dim3(ceil_div(total, 256u)), dim3(256), 0, s, Wt, Wf, C_IN, C_OUT, u32(C::NT), a.chunks,
                           u32(C::KG), total, PendingSum());
    if (int st = check_launch(what)) return st;
    hipLaunchKernelGGL((conv_split_kernel<C>), dim3(u32(tiles), 1, slices), dim3(C::NTH), 0, s, a);
    int st = check_launch(what);
    if (st == CRB_OK && slices > 1) st = launch_ordered_reduce(part, Y, count, slices, ReduceEpi{bias, OH * OW, C_OUT, relu ? u32(EPI_RELU) : 0u}, s, what);
    return st;
}

// ---- data gradient at stride 2: the four residue classes of input pixels -----------------------------------------------------------
// dX(2y + py, 2x + px) only receives the taps fh = (py + pad) mod 2, + 2, ...: each class is a correlation of dY at stride 1 with 1 to 3 x 1
// to 3 taps. One launch runs all four, the larger tap grids first; a workgroup belongs to one. R: taps of the largest grid on a side.
template <int R_, int WM, int WN, int MAXPX>
struct ConvSplitClassCfg {
    static constexpr int R = R_;
    typedef ConvSplitRect<R, R, 1, 1, 2, WM, WN, 1, MAXPX, 2, 2> C0;
    typedef ConvSplitRect<R, R - 1, 1, 1, 2, WM, WN, 1, MAXPX, 2, 2> C1;
    typedef ConvSplitRect<R - 1, R, 1, 1, 2, WM, WN, 1, MAXPX, 2, 2> C2;
    typedef ConvSplitRect<R - 1, R - 1, 1, 1, 2, WM, WN, 1, MAXPX, 2, 2> C3;
};
struct ConvSplitClassArgs {
    ConvSplitArgs c[4];
    u32 first[4];  // workgroups of a class begin here
};
template <class Set, bool PLAIN>
__global__ void __launch_bounds__(Set::C0::NTH, PLAIN && Set::R == 3 ? 1 : 2) conv_split_class_kernel(ConvSplitClassArgs a) {
    __shared__ __attribute__((aligned(16))) unsigned char smem[2 * Set::C0::STAGE + (PLAIN ? Set::C0::FILTERS : 0)];
    const u32 b = blockIdx.x;
    if (b < a.first[1]) conv_split_body<typename Set::C0, PLAIN, true>(a.c[0], b, 0, smem);
    else if (b < a.first[2]) conv_split_body<typename Set::C1, PLAIN, true>(a.c[1], b - a.first[1], 0, smem);
    else if (b < a.first[3]) conv_split_body<typename Set::C2, PLAIN, true>(a.c[2], b - a.first[2], 0, smem);
    else conv_split_body<typename Set::C3, PLAIN, true>(a.c[3], b - a.first[3], 0, smem);
}
// Fragments of the four classes' filters behind one another, each as conv_split_filters_kernel lays them. (C_IN: channels of dY)
struct ConvSplitClassFilters {
    u32 first[4], nt[4], fw[4];  // first 1 KB step of a class, its taps, taps in a row
    int tap0[4], tap_i, tap_j;
    u32 c_in, c_out, nt_all, chunks, total;
};
template <bool SUM>
static __global__ void __launch_bounds__(256) conv_split_class_filters_kernel(const float *__restrict__ W, unsigned char *__restrict__ Wf,
                                                                              ConvSplitClassFilters a, PendingSum sum) {
    if constexpr (SUM) {
        __shared__ __attribute__((aligned(16))) float red[kPendingSumFloats];
        if (blockIdx.x < sum.blocks) {
            pending_sum_block(sum, blockIdx.x, red);
            return;
        }
    }
    const u32 t = (blockIdx.x - (SUM ? sum.blocks : 0)) * 256 + threadIdx.x;
    if (t >= a.total) return;
    const u32 lane = t & 63, frag = t >> 6, k = frag < a.first[1] ? 0 : (frag < a.first[2] ? 1 : (frag < a.first[3] ? 2 : 3));
    const u32 f = frag - a.first[k], tap = f % a.nt[k], rest = f / a.nt[k], ch = rest % a.chunks, ob = rest / a.chunks;
    const u32 oc = ob * 32 + (lane & 31), ic0 = ch * 16 + 8 * (lane >> 5);
    const u32 w_tap = u32(a.tap0[k] + int(tap / a.fw[k]) * a.tap_i + int(tap % a.fw[k]) * a.tap_j);
    float w[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const bool ok = oc < a.c_out && ic0 + j < a.c_in;
        const float v = W[ok ? (size_t(ic0 + j) * a.c_out + oc) * a.nt_all + w_tap : 0];
        w[j] = ok ? v : 0.f;
    }
    u32x4 part[kSplit];
    split8(w, part);
    unsigned char *dst = Wf + size_t(frag) * (kSplit * 1024) + lane * 16;
#pragma unroll
    for (int p = 0; p < kSplit; ++p) *reinterpret_cast<u32x4 *>(dst + p * 1024) = part[p];
}

// Class k: its taps begin at (fh0, fw0) and are nfh x nfw, its pixels at (py, px) and CH x CW.
struct ConvSplitClass {
    u32 nfh, nfw, fh0, fw0, py, px, CH, CW;
};
inline ConvSplitClass conv_split_class(u32 k, u32 R, u32 IH, u32 IW, u32 pH, u32 pW) {
    ConvSplitClass c;
    c.nfh = R - k / 2, c.nfw = R - k % 2, c.fh0 = k / 2, c.fw0 = k % 2;  // (of an odd filter's taps, one more begin at 0)
    c.py = (c.fh0 + pH) & 1, c.px = (c.fw0 + pW) & 1;
    c.CH = IH > c.py ? ceil_div(IH - c.py, 2u) : 0, c.CW = IW > c.px ? ceil_div(IW - c.px, 2u) : 0;
    return c;
}
// Column strips of the four classes; false: a class does not fit the LDS.
template <class Set>
inline bool conv_split_class_strips(u32 IH, u32 IW, u32 pH, u32 pW, u32 (&strips)[4]) {
    for (u32 k = 0; k < 4; ++k) {
        const ConvSplitClass c = conv_split_class(k, Set::R, IH, IW, pH, pW);
        strips[k] = 1;
        if (!c.CH || !c.CW) continue;
        strips[k] = k == 0   ? conv_split_strips<typename Set::C0>(c.CH, c.CW)
                    : k == 1 ? conv_split_strips<typename Set::C1>(c.CH, c.CW)
                    : k == 2 ? conv_split_strips<typename Set::C2>(c.CH, c.CW)
                             : conv_split_strips<typename Set::C3>(c.CH, c.CW);
        if (!strips[k]) return false;
    }
    return true;
}
template <class Set>
inline size_t conv_split_class_filter_bytes(u32 C_IN, u32 C_OUT) {
    typedef typename Set::C0 C;
    const size_t blocks = ceil_div(C_OUT, u32(C::OCT)) * (C::OCT / 32), chunks = ceil_div(C_IN, 16u), taps = (2 * Set::R - 1) * (2 * Set::R - 1);
    return (blocks * chunks * taps + C::AHEAD) * kSplit * 1024;
}
// F = 2R - 1. Wf: conv_split_class_filter_bytes of scratch, or null (PLAIN).
template <class Set>
inline int launch_conv_split_classes(const float *Wt, const float *dY, float *dX, unsigned char *Wf, u32 N, u32 IC, u32 OC, u32 IH, u32 IW, u32 OH, u32 OW,
                                     const u32 (&strips)[4], u32 pH, u32 pW, hipStream_t s, const char *what, const PendingSum *sum) {
    typedef typename Set::C0 C;
    constexpr u32 F = 2 * Set::R - 1;
    ConvSplitClassArgs a = {};
    ConvSplitClassFilters f = {};
    f.c_in = OC, f.c_out = IC, f.nt_all = F * F, f.chunks = ceil_div(OC, 16u), f.tap_i = -2 * int(F), f.tap_j = -2;
    const u32 blocks = ceil_div(IC, u32(C::OCT)) * (C::OCT / 32);
    u32 steps = 0;
    uint64_t tiles = 0;
    for (u32 k = 0; k < 4; ++k) {
        const ConvSplitClass g = conv_split_class(k, Set::R, IH, IW, pH, pW);
        a.first[k] = u32(tiles);
        f.first[k] = steps, f.nt[k] = g.nfh * g.nfw, f.fw[k] = g.nfw;
        f.tap0[k] = int((g.fh0 + 2 * (g.nfh - 1)) * F + g.fw0 + 2 * (g.nfw - 1));  // (the last tap meets the window's first row and column)
        const u32 first = steps;
        steps += blocks * f.chunks * f.nt[k];
        if (!g.CH || !g.CW) continue;
        // tap i of pixel y reads row y + (py + pH) / 2 - i of dY
        const int pad_y = int(g.nfh) - 1 - int((g.py + pH) / 2), pad_x = int(g.nfw) - 1 - int((g.px + pW) / 2);
        auto fill = [&](auto cfg) {
            ConvSplitArgs &c = a.c[k];
            c = conv_split_args<decltype(cfg)>(Wt, dY, dX, nullptr, Wf ? Wf + size_t(first) * (kSplit * 1024) : nullptr, N, OC, IC, OH, OW, g.CH, g.CW,
                                               strips[k], 1, pad_y, pad_x);
            c.w_oc = F * F, c.w_ic = IC * F * F, c.tap0 = f.tap0[k], c.tap_i = f.tap_i, c.tap_j = f.tap_j;
            c.OHW = IH * IW, c.out_w = IW, c.osy = c.osx = 2, c.oy0 = g.py, c.ox0 = g.px;
            tiles += uint64_t(c.px_tiles) * c.oc_tiles;
        };
        if (k == 0) fill(typename Set::C0());
        if (k == 1) fill(typename Set::C1());
        if (k == 2) fill(typename Set::C2());
        if (k == 3) fill(typename Set::C3());
    }
    if (tiles > 0x7fffffffull) return fail(CRB_EINVAL_SHAPE, "%s: launch grid too large", what);
    if (!Wf) {
        hipLaunchKernelGGL((conv_split_class_kernel<Set, true>), dim3(u32(tiles)), dim3(C::NTH), 0, s, a);
        return check_launch(what);
    }
    f.total = steps * 64;
    if (sum)
        hipLaunchKernelGGL(conv_split_class_filters_kernel<true>, dim3(sum->blocks + ceil_div(f.total, 256u)), dim3(256), 0, s, Wt, Wf, f, *sum);
    else
        hipLaunchKernelGGL(conv_split_class_filters_kernel<false>, dim3(ceil_div(f.total, 256u)), dim3(256), 0, s, Wt, Wf, f, PendingSum());
    if (int st = check_launch(what)) return st;
    hipLaunchKernelGGL((conv_split_class_kernel<Set, false>), dim3(u32(tiles)), dim3(C::NTH), 0, s, a);
    return check_launch(what);
}

}  // namespace crb
