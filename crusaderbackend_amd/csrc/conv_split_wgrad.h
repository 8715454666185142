// Convolution weight gradient on split bf16 operands (split_bf16.h), stride S, any image extent and any padding:
//   dW[oc][ic][fh][fw] += sum over pixels (n, y, x) of dY[n][oc][y][x] * X[n][ic][S*y + fh - pad][S*x + fw - pad].
//
// For every tap a product (oc x ic) whose contraction index is the pixel. Pixels are taken flat over column strips of the images,
// as in conv_split.h: a tile is PXT consecutive pixels, of which each K group of the workgroup's waves takes sixteen -
// one MFMA step for each of its taps. Both operands are staged channel-fastest, [part][channel octet][position] units of 16 bytes (the
// split happens on the way), X with the halo its taps need; the fragments, which want eight consecutive pixels of one channel, are
// read with the transposing LDS read (ds_read_b64_tr_b16: sixteen lanes name four positions x sixteen channels and receive four
// positions of one channel each). A tap is then a constant shift of a lane's position and nothing is staged twice.
// A wave owns 32 output x 32 input channels and NTW taps (16*NTW accumulators); a workgroup WM x WN such blocks and a slice of
// the tiles. The K groups are summed through LDS in group order, the slices by the split reduction: bit-reproducible.
//
// What bounds it: a tile costs a wave 6*NTW MFMAs (32 clocks each) against 6*(NTW + 1) LDS reads of 512 bytes; the split of the
// staged elements is a fifth of the MFMAs' time and runs beside the other wave's. Every workgroup writes a slice of its block,
// 18 MB for the 256 of a launch, which the reduction reads back: 64 x 32 channels per workgroup keep that under the staging that
// smaller blocks would repeat.
#pragma once
#include "igemm_engine.h"
#include "split_bf16.h"

#include <type_traits>

namespace crb {

template <int F_, int S_, int WM_, int WN_, int KG_, int MAXPX_>
struct SplitWgradCfg {
    static constexpr int F = F_, S = S_, WM = WM_, WN = WN_, KG = KG_, MAXPX = MAXPX_;
    // filter rows, taps of a workgroup. 5x5: one row, blockIdx.y; of X it then stages only the rows that its filter row meets, one for
    // each row of dY (against the rows of all five: 1650 random layers at stride 1 take 0.85 of the time in the mean, one in a hundred more, by 1.24 at the most)
    static constexpr int ROWS = F <= 3 ? F : 1, NTW = ROWS * F;
    static constexpr int NTH = 64 * WM * WN * KG, PXT = 16 * KG, OCT = 32 * WM, ICT = 32 * WN;
    static constexpr int XO = ICT / 8, DO = OCT / 8;             // channel octets
    // 64 bytes behind each octet: the four octets a transposing read touches then start 64 bytes apart in a 256-byte bank row
    static constexpr int XOCT = MAXPX * 16 + 64, DOCT = PXT * 16 + 64, XPART = XO * XOCT, DPART = DO * DOCT;
    static constexpr int STAGE = kSplit * (XPART + DPART);
    static constexpr int XNP = XO * MAXPX / NTH, DNP = DO * PXT / NTH;
    static_assert(XO * MAXPX % NTH == 0 && DO * PXT % NTH == 0, "whole staging items per thread");
    static constexpr int RT = 8 * WM * WN * KG <= 64 && NTW % 3 == 0 ? 3 : 1;  // taps exchanged at a time
    static constexpr int LDS = 2 * STAGE;
    static_assert(WM * WN * KG * RT * 4096 <= LDS && OCT * ICT * NTW * 4 <= LDS && LDS <= 160 * 1024, "LDS");
};

struct SplitWgradArgs {
    const float *dY, *X;
    float *out;      // slices (splits > 1), or dW (accumulated)
    u32 images, IC, OC, H, W, HW, OHW, OW, SW, strips, npix, prow, pitch;
    int pad_y, pad_x;
    u32 ic_tiles, splits, tiles, tiles_z;  // tiles_z: tiles of a slice
    u32 OH;
    FastDiv ohw, ow, pitch_d, strip_d;
    u32 m_ow, m_oh, m_prow, m_strip;  // SmallDiv multipliers of SW, OH, prow, strips
};

// floor(n / d) for n * d < 2^20 and n / d < 4095 (the product stays under 2^32) as one full-rate 24-bit multiplication and a shift,
// m = ceil(2^20 / d): decoding the positions of every tile with 32-bit high multiplications (a quarter of the rate) cost as much as
// a third of a tile's MFMAs.
__device__ __forceinline__ u32 small_div(u32 n, u32 m) { return __umul24(n, m) >> 20; }

__device__ __forceinline__ bf16x8 read_transposed(const unsigned char *lds0, const unsigned char *lds1) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4 *lp;
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)(lds0)), b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)(lds1));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Sums that are not finite are formed again on the fp32 MFMA from the fp32 operands (split_bf16.h). x: the block in dW's order.
// The waves take the 32 x 32 channels of one tap in turn, over all pixels of the slice: two per MFMA, eight a step, the next
// step's operands requested ahead. Where the tap of a pixel lies outside the image both operands are zero (an infinite
// gradient would make NaN of the zero read there). Ends early where every sum is a NaN.
// p0, p1: the slice's pixels, as pixel_of counts them: whether tap (fh, fw) of one lies inside the image, and if so which image, and where in a
// plane of dY and of X.
template <class C, class PixelOf>
__device__ __forceinline__ void split_wgrad_again(float *x, const float *dY, const float *X, u32 IC, u32 OC, u32 HW, u32 OHW, u32 oc0, u32 ic0, int fh0, u32 p0,
                                                  u32 p1, PixelOf pixel_of) {
    constexpr int F = C::F, KG = C::KG, NTW = C::NTW, NW = C::WM * C::WN;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int unit = wv; unit < NW * NTW; unit += NW * KG) {
        const int tap = unit % NTW, um = unit / NTW / C::WN, un = unit / NTW % C::WN, i32 = lane & 31, h = lane >> 5;
        float *const res = x + ((um * 32 + 4 * h) * C::ICT + un * 32 + i32) * NTW + tap;  // register r: row 8 * (r / 4) + r % 4
        bool again = false;
#pragma unroll
        for (int r = 0; r < 16; ++r) again |= !__builtin_isfinite(res[(8 * (r / 4) + r % 4) * C::ICT * NTW]);
        if (!__any(int(again))) continue;
        struct Step {
            float d[4], x[4];
        };
        const u32 oc = oc0 + um * 32 + i32, ic = ic0 + un * 32 + i32;
        const float *drow = dY + size_t(oc < OC ? oc : OC - 1) * OHW, *xrow = X + size_t(ic < IC ? ic : IC - 1) * HW;
        auto fetch_step = [&](u32 start, Step &f) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const u32 p = start + 2 * q + h;
                u32 img, dpix, xpix;  // image, place in a plane of dY and of X
                const bool in = pixel_of(p, fh0 + tap / F, tap % F, img, dpix, xpix);
                const float d = drow[in ? size_t(img) * OC * OHW + dpix : 0];
                const float e = xrow[in ? size_t(img) * IC * HW + xpix : 0];
                f.d[q] = in && oc < OC ? d : 0.f, f.x[q] = in && ic < IC ? e : 0.f;
            }
        };
        v16f sum;
#pragma unroll
        for (int r = 0; r < 16; ++r) sum[r] = 0.0f;
        Step next;
        fetch_step(p0, next);
#pragma unroll 1
        for (u32 p = p0; p < p1; p += 8) {
            const Step now = next;
            fetch_step(p + 8, next);  // (behind the slice's last pixel: for nobody)
            u32 numbers = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(now.d[q], now.x[q], sum, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 16; ++r) numbers |= __builtin_isnan(sum[r]) ? 0u : 1u;
            if (!__any(int(numbers))) break;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) res[(8 * (r / 4) + r % 4) * C::ICT * NTW] = sum[r];
    }
    lds_barrier();
}

// The end of a workgroup: sums over its K groups and out with the block.
template <class C, class PixelOf>
__device__ __forceinline__ void split_wgrad_finish(v16f (&acc)[C::NTW], unsigned char *smem, const float *dY, const float *X, float *dst0, u32 splits, u32 IC,
                                                   u32 OC, u32 HW, u32 OHW, u32 z, u32 oc0, u32 ic0, int fh0, u32 p0, u32 p1, PixelOf pixel_of) {
    constexpr int F = C::F, KG = C::KG, NTW = C::NTW;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wave = wv % (C::WM * C::WN), kgroup = wv / (C::WM * C::WN);
    const int wm = wave / C::WN, wn = wave % C::WN;
    // ---- sum the K groups (each its share of the registers), bring the block into dW's order, store whole rows of it ---------
    constexpr int NW = C::WM * C::WN, NR = 16 / KG;
    float own[NTW][NR];
    float *x = reinterpret_cast<float *>(smem);
#pragma unroll
    for (int q = 0; q < NTW / C::RT; ++q) {
        if (q) lds_barrier();
#pragma unroll
        for (int t = 0; t < C::RT; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) x[((kgroup * NW + wave) * C::RT + t) * 1024 + r * 64 + lane] = acc[q * C::RT + t][r];
        lds_barrier();
#pragma unroll
        for (int t = 0; t < C::RT; ++t)
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                float v = x[(wave * C::RT + t) * 1024 + (kgroup * NR + i) * 64 + lane];
#pragma unroll
                for (int g = 1; g < KG; ++g) v += x[((g * NW + wave) * C::RT + t) * 1024 + (kgroup * NR + i) * 64 + lane];
                own[q * C::RT + t][i] = v * kSplitDown;
            }
    }
    lds_barrier();
#pragma unroll
    for (int i = 0; i < NR; ++i) {
        const int r = kgroup * NR + i, row = wm * 32 + 8 * (r / 4) + 4 * (lane >> 5) + r % 4;
#pragma unroll
        for (int t = 0; t < NTW; ++t) x[(row * C::ICT + wn * 32 + (lane & 31)) * NTW + t] = own[t][i];
    }
    bool bad = false;
#pragma unroll
    for (int t = 0; t < NTW; ++t)
#pragma unroll
        for (int i = 0; i < NR; ++i) bad |= !__builtin_isfinite(own[t][i]);
    if (__builtin_expect(__syncthreads_or(bad), 0)) split_wgrad_again<C>(x, dY, X, IC, OC, HW, OHW, oc0, ic0, fh0, p0, p1, pixel_of);
    constexpr u32 ROW = C::ICT * NTW;
    const u32 nic = IC - ic0 < u32(C::ICT) ? IC - ic0 : u32(C::ICT);
    float *out = dst0 + (splits > 1 ? size_t(z) * OC * IC * (F * F) : 0);
    for (u32 e = threadIdx.x; e < u32(C::OCT) * ROW; e += C::NTH) {
        const u32 oc = e / ROW, rest = e % ROW, ic = rest / NTW, t = rest % NTW;
        if (oc0 + oc < OC && ic < nic) {
            float *dst = out + ((size_t(oc0 + oc) * IC + ic0 + ic) * (F * F) + fh0 * F + t);
            if (splits > 1) *dst = x[e]; else *dst += x[e];
        }
    }
}

template <class C>
__global__ void __launch_bounds__(C::NTH, 2) split_wgrad_kernel(SplitWgradArgs a) {
    constexpr int F = C::F, S = C::S, NTW = C::NTW, MAXPX = C::MAXPX, PXT = C::PXT;
    __shared__ __attribute__((aligned(256))) unsigned char smem[C::LDS];
    // slice z of all channel blocks has ids equal mod `splits`: with a multiple of 8 of them they share an XCD's L2
    const u32 z = blockIdx.x % a.splits, pair = blockIdx.x / a.splits, ot = pair / a.ic_tiles, it = pair % a.ic_tiles;
    const u32 oc0 = ot * C::OCT, ic0 = it * C::ICT;
    const int fh0 = C::ROWS == F ? 0 : int(blockIdx.y);
    const u32 t0 = z * a.tiles_z, t1 = t0 + a.tiles_z < a.tiles ? t0 + a.tiles_z : a.tiles;

    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wave = wv % (C::WM * C::WN), kgroup = wv / (C::WM * C::WN);
    const int wm = wave / C::WN, wn = wave % C::WN;
    // transposing read: this lane names channels 4*(lane%4).. of the block's half (lane/16)%2, position (lane%16)/4 (+ 8 in the upper half-wave)
    const u32 ch = ((lane >> 4) & 1) * 16 + (lane & 3) * 4, ch_off = (ch / 8), ch_byte = (ch % 8) * 2;
    const u32 kpos = 16 * kgroup + 8 * (lane >> 5) + ((lane & 15) >> 2);
    const u32 d_lane = (wm * 4 + ch_off) * C::DOCT + kpos * 16 + ch_byte, x_lane = (wn * 4 + ch_off) * C::XOCT + ch_byte;

    float xreg[C::XNP][8], dreg[C::DNP][8];
    // padded row and column of this thread's position of X inside a tile's run (its items are octets of one position)
    static_assert(C::NTH % MAXPX == 0 && C::NTH % PXT == 0, "a thread's items share their position");
    u32 xpr, xpc;
    a.pitch_d.divmod(threadIdx.x % MAXPX, xpr, xpc);
    // first pixel of a tile: image, strip, row, column; tiles are walked in order, so the next one's is a few scalar steps away
    struct First {
        u32 p, img, strip, y, x;
    };
    auto first_pixel = [&](u32 p0) {
        First f;
        u32 v, r;
        f.p = p0;
        a.ohw.divmod(p0, v, r);
        a.ow.divmod(r, f.y, f.x);
        a.strip_d.divmod(v, f.img, f.strip);
        return f;
    };
    // pixel k of a tile: strips behind the first one, row, column
    auto pixel = [&](const First &f, u32 k, u32 &dv, u32 &y, u32 &x) {
        const u32 xx = f.x + k, q = small_div(xx, a.m_ow), yy = f.y + q;
        x = xx - q * a.SW;
        dv = small_div(yy, a.m_oh);
        y = yy - dv * a.OH;
    };
    auto image = [&](const First &f, u32 dv, u32 &dimg, u32 &strip) {
        const u32 sv = f.strip + dv;
        dimg = small_div(sv, a.m_strip);
        strip = sv - dimg * a.strips;
    };
    auto following = [&](const First &f) {
        First n;
        u32 dv, dimg;
        n.p = f.p + PXT;
        pixel(f, PXT, dv, n.y, n.x);
        image(f, dv, dimg, n.strip);
        n.img = f.img + dimg;
        return n;
    };
    auto fetch = [&](const First &f, auto ragged_c) {
        constexpr bool RAG = decltype(ragged_c)::value;
        const size_t left = a.images - f.img;
        const BufferRange xr = buffer_range(a.X + (size_t(f.img) * a.IC + ic0) * a.HW, (left * a.IC - ic0) * a.HW);
        const BufferRange dr = buffer_range(a.dY + (size_t(f.img) * a.OC + oc0) * a.OHW, (left * a.OC - oc0) * a.OHW);
        const u32 ox = threadIdx.x / MAXPX, od = threadIdx.x / PXT, k = threadIdx.x % PXT;  // first items' octets
        u32 dv, y, x, dimg, strip;
        const u32 rr = (C::ROWS == 1 ? 1 : S) * f.y + xpr;
        dv = small_div(rr, a.m_prow);
        image(f, dv, dimg, strip);
        const int iy = (C::ROWS == 1 ? S * int(rr - dv * a.prow) + fh0 : int(rr - dv * a.prow)) - a.pad_y, ix = int(xpc + S * strip * a.SW) - a.pad_x;
        // (positions behind the run are read too where they exist; no pixel names them)
        const bool xin = dimg < u32(left) && u32(iy) < a.H && u32(ix) < a.W;
        const u32 xbytes = ((dimg * a.IC + 8 * ox) * a.HW + u32(iy) * a.W + u32(ix)) * 4u, xoff = xin ? xbytes : kOutside;
        pixel(f, k, dv, y, x);
        image(f, dv, dimg, strip);
        x += strip * a.SW;
        const bool din = f.p + k < a.npix && x < a.OW;
        const u32 dbytes = ((dimg * a.OC + 8 * od) * a.OHW + y * a.OW + x) * 4u, doff = din ? dbytes : kOutside;
        constexpr u32 XSTEP = C::NTH / MAXPX, DSTEP = C::NTH / PXT;  // octets between a thread's items
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            // (channels past the last: kOutside, at an offset the range holds)
#pragma unroll
            for (int i = 0; i < C::XNP; ++i) {
                const u32 c = 8 * XSTEP * i + j, ch = !RAG || ic0 + c < a.IC ? c : a.IC - ic0 - 1;
                xreg[i][j] = buffer_load(xr, !RAG || ic0 + 8 * ox + c < a.IC ? xoff : kOutside, ch * a.HW * 4u);
            }
#pragma unroll
            for (int i = 0; i < C::DNP; ++i) {
                const u32 c = 8 * DSTEP * i + j, ch = !RAG || oc0 + c < a.OC ? c : a.OC - oc0 - 1;
                dreg[i][j] = buffer_load(dr, !RAG || oc0 + 8 * od + c < a.OC ? doff : kOutside, ch * a.OHW * 4u);
            }
        }
    };
    auto store_unit = [](unsigned char *dst, int part_stride, const float (&r)[8]) {
        u32x4 part[kSplit];
        split8(r, part);
#pragma unroll
        for (int p = 0; p < kSplit; ++p) *reinterpret_cast<u32x4 *>(dst + p * part_stride) = part[p];
    };
    constexpr int ITEMS = C::XNP + C::DNP;
    auto commit_item = [&](unsigned char *sm, int i) {
        if (i < C::XNP) {
            const u32 u = threadIdx.x + i * C::NTH;
            store_unit(sm + (u / MAXPX) * C::XOCT + (u % MAXPX) * 16, C::XPART, xreg[i < C::XNP ? i : 0]);
        } else {
            const int d = i - C::XNP;
            const u32 u = threadIdx.x + d * C::NTH;
            store_unit(sm + kSplit * C::XPART + (u / PXT) * C::DOCT + (u % PXT) * 16, C::DPART, dreg[d >= 0 ? d : 0]);
        }
    };

    v16f acc[NTW];
#pragma unroll
    for (int t = 0; t < NTW; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] = 0.0f;

    // LDS positions of this lane's two pixels (the second four positions on)
    u32 xs[2];
    auto positions = [&](const First &f) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            u32 k = kpos + 4 * i, dv, y, x;
            k = f.p + k < a.npix ? k : 0;  // (dY is zero there)
            pixel(f, k, dv, y, x);
            xs[i] = ((dv * a.prow + (C::ROWS == 1 ? 1 : S) * (y - f.y)) * a.pitch + S * x) * 16 + x_lane;
        }
    };
    auto main_loop = [&](auto ragged_c) {
        First cur = first_pixel((t0 < t1 ? t0 : 0u) * PXT);
        if (t0 < t1) {
            fetch(cur, ragged_c);
            positions(cur);
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) commit_item(smem, i);
        }
        lds_barrier();
        u32 buf = 0;
        for (u32 tile = t0; tile < t1; ++tile, buf = C::STAGE - buf) {
            if (tile + 1 < t1) cur = following(cur);  // (behind the last tile: that tile once more, for nobody)
            bf16x8 fa[kSplit], fb[2][kSplit];
            auto read_x = [&](int set, int tap) {
                const u32 shift = ((tap / F) * a.pitch + tap % F) * 16 + buf;
#pragma unroll
                for (int p = 0; p < kSplit; ++p) fb[set][p] = read_transposed(smem + xs[0] + shift + p * C::XPART, smem + xs[1] + shift + p * C::XPART);
            };
            const unsigned char *dsm = smem + buf + kSplit * C::XPART + d_lane;
            v16f small;
            const v16f zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
            for (int p = 0; p < kSplit; ++p) fa[p] = read_transposed(dsm + p * C::DPART, dsm + p * C::DPART + 64);
            // A block of six MFMAs per tap; X's fragments are read a block ahead. The next tile is requested beside the first blocks,
            // split and stored beside the last ones, one item each; the positions of its pixels follow. Each of these regions is
            // fenced, and inside it the other work is spread between the MFMAs.
            constexpr int HEAD = NTW >= 9 ? 3 : 1;
            read_x(0, 0);
#pragma unroll
            for (int m = 0; m < NTW; ++m) {
                const int item = m - (NTW - ITEMS);
                if (m == 0) __builtin_amdgcn_sched_barrier(0);
                else if (m >= HEAD) __builtin_amdgcn_sched_barrier(0x2);  // (the last block's additions may stand beside this one's MFMAs)
                if (m == 0) fetch(cur, ragged_c);
                if (m + 1 < NTW) read_x((m + 1) & 1, m + 1);
                if (item >= 0) commit_item(smem + (C::STAGE - buf), item);
                // The five small part products are summed by themselves and then added (a second set of accumulators does not fit): two
                // roundings of the sum instead of six, 64 -> 64 @56 batch 32 behind a ReLU 3.43e-7 -> 1.45e-7 from float64 (fp32 2.71e-7),
                // for 16 additions a block: 65.5 -> 75.4 us, 256 -> 256 @14 55.5 -> 64.4.
                acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[kTermA[kTerms - 1]], fb[m & 1][kTermB[kTerms - 1]], acc[m], 0, 0, 0);
#pragma unroll
                for (int t = 0; t + 1 < kTerms; ++t) small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[kTermA[t]], fb[m & 1][kTermB[t]], t ? small : zero, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[m][r] += small[r];
                if (m == NTW - 1) positions(cur);
#pragma unroll
                for (int t = 0; t < kTerms; ++t) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 9, 0);
                    if (m < HEAD) __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
                    if (item >= 0) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            lds_barrier();
        }
    };
    if (a.IC - ic0 < u32(C::ICT) || a.OC - oc0 < u32(C::OCT)) main_loop(std::true_type()); else main_loop(std::false_type());

    split_wgrad_finish<C>(acc, smem, a.dY, a.X, a.out, a.splits, a.IC, a.OC, a.HW, a.OHW, z, oc0, ic0, fh0, t0 * PXT, t1 * PXT,
                          [&](u32 p, int fh, int fw, u32 &img, u32 &dpix, u32 &xpix) {
                              u32 v, rem, py, px, strip;
                              a.ohw.divmod(p < a.npix ? p : a.npix - 1, v, rem);
                              a.ow.divmod(rem, py, px);
                              a.strip_d.divmod(v, img, strip);
                              px += strip * a.SW;
                              const int iy = int(S * py) + fh - a.pad_y, ix = int(S * px) + fw - a.pad_x;
                              dpix = py * a.OW + px, xpix = u32(iy) * a.W + u32(ix);
                              return p < a.npix && px < a.OW && u32(iy) < a.H && u32(ix) < a.W;
                          });
}

struct SplitWgradPlan {
    u32 strips = 0, pairs = 0, splits = 0, tiles = 0, tiles_z = 0;
    size_t workspace_bytes = 0;
};
// Padded rows of an image, positions of the longest run a tile touches.
template <class C>
inline u32 split_wgrad_prow(u32 OH) { return C::ROWS == 1 ? OH : C::S * (OH - 1) + C::F; }
template <class C>
inline u32 split_wgrad_window(u32 OH, u32 SW) {
    const u32 pitch = C::S * (SW - 1) + C::F;
    return C::ROWS == 1 ? conv_split_window(C::PXT, OH, SW, 1, 1, 1) / SW * pitch : conv_split_window(C::PXT, OH, SW, C::F, C::F, C::S);
}
// most: bytes the slices may take
template <class C>
inline SplitWgradPlan split_wgrad_plan(u32 N, u32 IC, u32 OC, u32 H, u32 W, u32 OH, u32 OW, size_t most) {
    SplitWgradPlan p;
    for (u32 ns = ceil_div(OW, 64u); ns <= OW && ns <= 16; ++ns)
        if (split_wgrad_window<C>(OH, ceil_div(OW, ns)) <= u32(C::MAXPX)) {
            p.strips = ns;
            break;
        }
    // small_div's range (quotients are rows, images or strips of one tile, so at most its pixels or run and the 16 strips), and the
    // images a tile touches within 2 GiB (buffer loads)
    static_assert(C::PXT + 16 < 4095 && C::MAXPX + 16 < 4095, "quotients of small_div");
    const uint64_t sw = p.strips ? ceil_div(OW, p.strips) : 0, prow = split_wgrad_prow<C>(OH), run = C::MAXPX;
    const bool small = (C::PXT + sw) * sw < (1u << 20) && (OH + C::PXT) * uint64_t(OH) < (1u << 20) && (prow + run) * prow < (1u << 20);
    const uint64_t images = p.strips ? uint64_t(C::PXT) / (uint64_t(OH) * ceil_div(OW, p.strips)) + 3 : 0;
    if (!p.strips || !small || images * IC * H * W * 4 > 0x7fffffffull || images * OC * OH * OW * 4 > 0x7fffffffull) {
        p.strips = 0;
        return p;
    }
    p.tiles = ceil_div(N * p.strips * OH * ceil_div(OW, p.strips), u32(C::PXT));
    p.pairs = ceil_div(OC, u32(C::OCT)) * ceil_div(IC, u32(C::ICT));
    const u32 rows = C::F / C::ROWS;
    u32 splits = p.pairs * rows >= 256 ? 1 : 256 / (p.pairs * rows);  // one workgroup per CU
    if (splits > ceil_div(p.tiles, 4u)) splits = ceil_div(p.tiles, 4u);
    const size_t slice = size_t(OC) * IC * C::F * C::F * sizeof(float);
    if (splits > 1 && splits > most / slice) splits = most / slice > 1 ? u32(most / slice) : 1;
    p.tiles_z = ceil_div(p.tiles, splits);
    p.splits = ceil_div(p.tiles, p.tiles_z);
    p.workspace_bytes = p.splits > 1 ? p.splits * slice : 0;
    return p;
}

// later: null, or where the slices' sum is left for another launch.
template <class C>
inline int launch_split_wgrad(const SplitWgradPlan &p, const float *dY, const float *X, float *dW, float *ws, u32 N, u32 IC, u32 OC, u32 H, u32 W,
                              u32 OH, u32 OW, int pad_y, int pad_x, hipStream_t s, const char *what, PendingSum *later) {
    SplitWgradArgs a;
    a.dY = dY, a.X = X, a.out = p.splits > 1 ? ws : dW;
    a.images = N, a.IC = IC, a.OC = OC, a.H = H, a.W = W, a.HW = H * W, a.OHW = OH * OW, a.OW = OW;
    a.strips = p.strips, a.SW = ceil_div(OW, p.strips), a.npix = N * p.strips * OH * a.SW;
    a.prow = split_wgrad_prow<C>(OH), a.pitch = C::S * (a.SW - 1) + C::F;
    a.pad_y = pad_y, a.pad_x = pad_x;
    a.ic_tiles = ceil_div(IC, u32(C::ICT)), a.splits = p.splits, a.tiles = p.tiles, a.tiles_z = p.tiles_z;
    a.ohw.init(OH * a.SW), a.ow.init(a.SW), a.pitch_d.init(a.pitch), a.strip_d.init(p.strips);
    auto mul = [](u32 d) { return ((1u << 20) + d - 1) / d; };
    a.OH = OH, a.m_ow = mul(a.SW), a.m_oh = mul(OH), a.m_prow = mul(a.prow), a.m_strip = mul(p.strips);
    if (uint64_t(p.pairs) * p.splits > 0x7fffffffull) return fail(CRB_EINVAL_SHAPE, "%s: launch grid too large", what);
    hipLaunchKernelGGL((split_wgrad_kernel<C>), dim3(p.pairs * p.splits, C::F / C::ROWS), dim3(C::NTH), 0, s, a);
    if (int st = check_launch(what)) return st;
    if (p.splits > 1 && later) return *later = pending_sum(ws, dW, OC * IC * C::F * C::F, p.splits), CRB_OK;
    if (p.splits > 1) return launch_splitk_reduce(ws, dW, OC * IC * C::F * C::F, p.splits, ReduceEpi{nullptr, 1, 1, EPI_ACCUM}, s, what);
    return CRB_OK;
}

}  // namespace crb
