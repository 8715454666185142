// Weight gradient of 3x3 layers at stride 1, pad 1, on split bf16 operands, pixels in the order they lie in memory.
//   dW[oc][ic][fh][fw] += sum over q of dY[q - (fw - 1)] * X[q + (fh - 1) * P], q over rows of P positions.
//
// The contraction index is the pixel, and in NCHW eight consecutive pixels of a channel lie side by side: an MFMA fragment (eight k of a
// channel a lane) is then one 16-byte LDS read from [part][channel][position], where conv_split_wgrad.h, whose LDS holds channels fastest,
// needs two transposing reads of 8 bytes for every tap. Images are laid out as rows of P = 8 * ceil((W + 1) / 8) positions with one row of
// zeros between two images, so that column and row borders are zeros of their own and a tap is a shift of the flat position. The
// rows of a filter shift X by whole octets, in its address. Its columns shift dY by one position, in registers: three fragments of dY
// are formed from one read and the words on either side of it, twelve instructions, and serve all three filter rows. A wave reads 9 KB of X
// and 4.5 KB of dY for its 54 MFMAs, against 30 KB.
// LDS holds a ring of octets for either operand, X's with the two rows that the taps reach over: nothing is staged twice. A tile is sixteen
// octets, each of the eight waves of a workgroup taking two, one MFMA step of each tap; a thread stages one octet of X and one of dY of a
// channel for the next tile.
// The price is the padding: (W + 1 -> P) * (H + 1), 16 % of the MFMAs at 56 x 56, 22 % at 14 x 14.
#pragma once
#include "conv_split_wgrad.h"

namespace crb {

struct RowsWgradCfg {
    static constexpr int F = 3, WM = 1, WN = 1, KG = 8, NTW = 9, NTH = 512, OCT = 32, ICT = 32;  // (KG: waves, as split_wgrad_again counts them)
    static constexpr u32 ND = 34;        // ring of dY, octets: a tile, one octet on either side, the next tile
    static constexpr u32 MAXP8 = 16;     // octets of a row, at most
    static constexpr u32 MAXNX = 32 + 2 * MAXP8;
    static constexpr u32 OCTET = 32 * 16;  // bytes of an octet: 32 channels
    static constexpr u32 DPART = ND * OCTET, LDS = kSplit * (MAXNX * OCTET + DPART);
    static constexpr u32 TS = 1032;      // floats from tap to tap where the waves' sums meet: consecutive elements of dW in different banks
    static_assert(LDS <= 160 * 1024 && 4 * NTW * TS * 4 <= LDS, "LDS");
};

struct RowsWgradArgs {
    const float *dY, *X;
    float *out;          // slices (splits > 1), or dW (accumulated)
    u32 images, IC, OC, H, W, HW;
    u32 P8, RI, NX;      // octets of a row, rows of an image (H + 1), octets of X's ring
    u32 ic_tiles, splits, tiles, tiles_z;
    FastDiv p8, ri;
};

typedef float f32x4 __attribute__((ext_vector_type(4)));
// Eight floats in VEC-wide loads, of which vector j lies `off` + 4 * VEC * j bytes in and exists where j * VEC < count.
template <int VEC>
__device__ __forceinline__ void load_octet(BufferRange r, u32 off, int count, float (&v)[8]) {
#pragma unroll
    for (int j = 0; j < 8 / VEC; ++j) {
        const int at = int(j * VEC < count ? off + 4 * VEC * j : kOutside);
        if constexpr (VEC == 4) {
            const f32x4 q = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0));
#pragma unroll
            for (int i = 0; i < 4; ++i) v[4 * j + i] = q[i];
        } else if constexpr (VEC == 2) {
            const f32x2 q = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(r, at, 0, 0));
#pragma unroll
            for (int i = 0; i < 2; ++i) v[2 * j + i] = q[i];
        } else {
            v[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, at, 0, 0));
        }
    }
}

// VEC: floats of a load; rows are whole vectors (W % VEC == 0) at addresses of whole vectors.
template <int VEC>
__global__ void __launch_bounds__(RowsWgradCfg::NTH, 2) rows_wgrad_kernel(RowsWgradArgs a) {
    typedef RowsWgradCfg C;
    __shared__ __attribute__((aligned(256))) unsigned char smem[C::LDS];
    // slice z of all channel blocks has ids equal mod `splits`: with a multiple of 8 of them they share an XCD's L2
    const u32 z = blockIdx.x % a.splits, pair = blockIdx.x / a.splits, ot = pair / a.ic_tiles, it = pair % a.ic_tiles;
    const u32 oc0 = ot * C::OCT, ic0 = it * C::ICT;
    const u32 t0 = z * a.tiles_z, tiles = t0 + a.tiles_z < a.tiles ? a.tiles_z : a.tiles - t0, d0 = 16 * t0;
    const u32 xpart = a.NX * C::OCTET;
    unsigned char *const xsm = smem + kSplit * C::DPART;

    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // staging: octet of a tile, channel (a wave: sixteen runs of 128 bytes in memory, all banks twice in LDS)
    const u32 i16 = (lane & 3) + 4 * (wv & 3), ch = (lane & 12) + (lane >> 4) + 16 * (wv >> 2);
    const bool xch = ic0 + ch < a.IC, dch = oc0 + ch < a.OC;
    const BufferRange xr = buffer_range(a.X, size_t(a.images) * a.IC * a.HW), dr = buffer_range(a.dY, size_t(a.images) * a.OC * a.HW);
    const u32 w4 = a.W * 4;
    // A thread's octet of an operand: the image's first byte (of this block's channel), row of the image's rows, column octet.
    struct Place {
        u32 img, y, c;
    };
    auto place = [&](u32 octet, u32 image_bytes, u32 channel_bytes) {
        Place f;
        u32 row, img;
        a.p8.divmod(octet, row, f.c);
        a.ri.divmod(row, img, f.y);
        f.img = img * image_bytes + channel_bytes;
        return f;
    };
    const u32 dr16 = 16 / a.P8, dc16 = 16 % a.P8;
    auto step = [&](Place &f, u32 image_bytes) {  // sixteen octets on: at most one image (rows_wgrad_plan)
        const u32 c = f.c + dc16;
        const bool carry = c >= a.P8;
        f.c = carry ? c - a.P8 : c;
        const u32 y = f.y + dr16 + carry;
        const bool over = y >= a.RI;
        f.y = over ? y - a.RI : y;
        f.img += over ? image_bytes : 0u;
    };
    const u32 ximg = a.IC * a.HW * 4, dimg = a.OC * a.HW * 4, xch_off = (ic0 + ch) * a.HW * 4 - w4, dch_off = (oc0 + ch) * a.HW * 4;
    // (behind the last image the range check reads zeros)
    auto fetch_x = [&](const Place &f, float (&reg)[8]) {  // row y of an image's rows is row y - 1 of X; row 0 lies between two images
        load_octet<VEC>(xr, f.img + __umul24(f.y, w4) + 32 * f.c, xch && f.y > 0 ? int(a.W - 8 * f.c) : 0, reg);
    };
    auto fetch_d = [&](const Place &f, float (&reg)[8]) {
        load_octet<VEC>(dr, f.img + __umul24(f.y, w4) + 32 * f.c, dch && f.y < a.H ? int(a.W - 8 * f.c) : 0, reg);
    };
    auto commit = [](unsigned char *dst, u32 part_stride, const float (&r)[8]) {
        u32x4 part[kSplit];
        split8(r, part);
#pragma unroll
        for (int p = 0; p < kSplit; ++p) *reinterpret_cast<u32x4 *>(dst + p * part_stride) = part[p];
    };
    auto wrap = [](u32 s, u32 n) { return s >= n ? s - n : s; };

    // Octet `slot` of a ring, channel c. The two low bits of the slot are in the channel's place, so that neither the stores of four octets of a
    // channel nor the reads of sixteen channels meet in a bank.
    auto unit = [](u32 slot, u32 c) { return slot * C::OCTET + (c ^ (slot & 3)) * 16; };

    // ---- the first tile: octet d0 - 1 + s of dY in place s of its ring, octet d0 + s of X in place s --------------------------
    // (a place is written before it is read: every commit covers the sixteen octets behind the ones before it)
    float xreg[8], dreg[8];
    u32 sx = 2 * a.P8 + i16, sd = 2 + i16;  // this thread's next places
    Place xnext = place(d0 + 2 * a.P8 + i16, ximg, xch_off), dnext = place(d0 + 1 + i16, dimg, dch_off);
    {
        float first[8], before[8];
        for (u32 e = 16; e < 2 * a.P8; e += 16) {  // (what runs over into the first tile's octets is what that stores there)
            fetch_x(place(d0 + e + i16, ximg, xch_off), first);
            commit(xsm + unit(e + i16, ch), xpart, first);
        }
        fetch_x(place(d0 + i16, ximg, xch_off), first);
        fetch_d(place(d0 + i16 ? d0 + i16 - 1 : 0, dimg, dch_off), before);
        fetch_x(xnext, xreg);
        fetch_d(dnext, dreg);
        if (d0 == 0 && i16 == 0) {  // (nothing before the first image)
#pragma unroll
            for (int j = 0; j < 8; ++j) before[j] = 0.f;
        }
        commit(xsm + unit(i16, ch), xpart, first);
        if (i16 < 2) commit(smem + unit(i16, ch), C::DPART, before);
        commit(xsm + unit(sx, ch), xpart, xreg);
        commit(smem + unit(sd, ch), C::DPART, dreg);
    }
    step(xnext, ximg), step(dnext, dimg);
    fetch_x(xnext, xreg), fetch_d(dnext, dreg);
    lds_barrier();

    // ---- Waves w and w + 4 take the same four octets of a tile, 32 k, and sixteen output channels each. Lane: channel l % 16 of a block, octet l / 16,
    // in place kd of dY's ring and kx (+ P8 for every filter row) of X's.
    const u32 c16 = lane & 15, dc = 16 * (wv >> 2) + c16;
    u32 kx = 4 * (wv & 3) + (lane >> 4), kd = 1 + kx;
    v4f acc[9][2], small[9][2];
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[t][b][r] = small[t][b][r] = 0.0f;
    for (u32 tile = 0; tile < tiles; ++tile) {
        sx = wrap(sx + 16, a.NX), sd = wrap(sd + 16, C::ND);
        const u32 up = wrap(kd + 1, C::ND), down = wrap(kd + C::ND - 1, C::ND);
        bf16x8 f[3][kSplit], x[2][kSplit];
        auto read_x = [&](int g) {
            const unsigned char *src = xsm + unit(wrap(kx + g / 2 * a.P8, a.NX), c16 + 16 * (g % 2));
#pragma unroll
            for (int p = 0; p < kSplit; ++p) x[g % 2][p] = *reinterpret_cast<const bf16x8 *>(src + p * xpart);
        };
        read_x(0);
#pragma unroll
        for (int p = 0; p < kSplit; ++p) {
            const u32x4 w = *reinterpret_cast<const u32x4 *>(smem + unit(kd, dc) + p * C::DPART);
            const u32 before = *reinterpret_cast<const u32 *>(smem + unit(down, dc) + p * C::DPART + 12), behind = *reinterpret_cast<const u32 *>(smem + unit(up, dc) + p * C::DPART);
            const u32x4 to_next = {__builtin_amdgcn_alignbit(w[1], w[0], 16), __builtin_amdgcn_alignbit(w[2], w[1], 16), __builtin_amdgcn_alignbit(w[3], w[2], 16),
                                   __builtin_amdgcn_alignbit(behind, w[3], 16)};
            const u32x4 to_last = {__builtin_amdgcn_alignbit(w[0], before, 16), __builtin_amdgcn_alignbit(w[1], w[0], 16), __builtin_amdgcn_alignbit(w[2], w[1], 16),
                                   __builtin_amdgcn_alignbit(w[3], w[2], 16)};
            f[0][p] = __builtin_bit_cast(bf16x8, to_next), f[1][p] = __builtin_bit_cast(bf16x8, w), f[2][p] = __builtin_bit_cast(bf16x8, to_last);
        }
        // Six groups of eighteen MFMAs, a filter row and sixteen input channels each. The next tile goes into LDS beside the fourth and the fifth; the one behind
        // it is requested beside the last (behind the last tile: what follows it, for nobody).
#pragma unroll
        for (int g = 0; g < 6; ++g) {
            __builtin_amdgcn_sched_barrier(0);
            if (g < 5) read_x(g + 1);
            if (g == 3) commit(xsm + unit(sx, ch), xpart, xreg);
            if (g == 4) commit(smem + unit(sd, ch), C::DPART, dreg);
            if (g == 5) {
                step(xnext, ximg), step(dnext, dimg);
                fetch_x(xnext, xreg), fetch_d(dnext, dreg);
            }
#pragma unroll
            for (int t = 0; t < kTerms; ++t)
#pragma unroll
                for (int fw = 0; fw < 3; ++fw) {
                    v4f &sum = t + 1 < kTerms ? small[g / 2 * 3 + fw][g % 2] : acc[g / 2 * 3 + fw][g % 2];
                    sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[fw][kTermA[t]], x[g % 2][kTermB[t]], sum, 0, 0, 0);
                }
        }
        __builtin_amdgcn_sched_barrier(0);
        lds_barrier();
        kx = wrap(kx + 16, a.NX), kd = wrap(kd + 16, C::ND);
    }

    // ---- the four waves of a tap meet in LDS; a thread sums eighteen elements of the block, in dW's order ----------------------
    float *const x = reinterpret_cast<float *>(smem);
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) x[((wv & 3) * C::NTW + t) * C::TS + (8 * (wv >> 2) + 4 * b + r) * 64 + lane] = acc[t][b][r] + small[t][b][r];
    lds_barrier();
    constexpr int NE = C::OCT * C::ICT * C::NTW / C::NTH;
    static_assert(NE * C::NTH == C::OCT * C::ICT * C::NTW, "whole elements per thread");
    float own[NE];
    bool bad = false;
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        const u32 e = threadIdx.x + i * C::NTH, tap = e % 9, ic = e / 9 % 32, oc = e / 288;
        const float *src = x + tap * C::TS + (8 * (oc / 16) + 4 * (ic / 16) + oc % 4) * 64 + 16 * (oc / 4 % 4) + ic % 16;
        float v = src[0];
#pragma unroll
        for (int g = 1; g < 4; ++g) v += src[g * C::NTW * C::TS];
        own[i] = v * kSplitDown;
        bad |= !__builtin_isfinite(own[i]);
    }
    if (__builtin_expect(__syncthreads_or(bad), 0)) {
#pragma unroll
        for (int i = 0; i < NE; ++i) x[threadIdx.x + i * C::NTH] = own[i];
        lds_barrier();
        split_wgrad_again<C>(x, a.dY, a.X, a.IC, a.OC, a.HW, a.HW, oc0, ic0, 0, 8 * d0, 8 * (d0 + 16 * tiles),
                             [&](u32 q, int fh, int fw, u32 &img, u32 &dpix, u32 &xpix) {
                                 u32 row, c8, y;
                                 a.p8.divmod(q / 8, row, c8);
                                 a.ri.divmod(row, img, y);
                                 const int x = int(8 * c8 + q % 8), dx = x - fw + 1, iy = int(y) + fh - 1;
                                 dpix = y * a.W + u32(dx), xpix = u32(iy) * a.W + u32(x);
                                 return img < a.images && y < a.H && u32(iy) < a.H && u32(x) < a.W && u32(dx) < a.W;
                             });
#pragma unroll
        for (int i = 0; i < NE; ++i) own[i] = x[threadIdx.x + i * C::NTH];
    }
    // (channels past the last are dropped by the range check)
    const BufferRange out = buffer_range(a.out + (a.splits > 1 ? size_t(z) * a.OC * a.IC * 9 : 0), size_t(a.OC) * a.IC * 9);
    u32 at[NE];
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        const u32 e = threadIdx.x + i * C::NTH, ic = ic0 + e / 9 % 32, oc = oc0 + e / 288;
        at[i] = oc < a.OC && ic < a.IC ? ((oc * a.IC + ic) * 9 + e % 9) * 4 : kOutside;
    }
    if (a.splits == 1) {
        float old[NE];
#pragma unroll
        for (int i = 0; i < NE; ++i) old[i] = buffer_load(out, at[i], 0);
#pragma unroll
        for (int i = 0; i < NE; ++i) own[i] += old[i];
    }
#pragma unroll
    for (int i = 0; i < NE; ++i) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(u32, own[i]), out, int(at[i]), 0, 0);
}

// most: bytes the slices may take. (strips == 0: not for this kernel)
inline SplitWgradPlan rows_wgrad_plan(u32 N, u32 IC, u32 OC, u32 H, u32 W, size_t most) {
    typedef RowsWgradCfg C;
    SplitWgradPlan p;
    const u32 P8 = W / 8 + 1, RI = H + 1;
    if (P8 > C::MAXP8 || W % 2) return p;  // (odd rows are read a word at a time: 70 -> 50 @20x37 batch 16 28.9 -> 31.4 us)
    const uint64_t octets = uint64_t(N) * RI * P8;
    // a tile goes on into the next image, not beyond it; operands and gradient within 2 GiB (buffer loads), offsets behind the last image within
    // 4 GiB, rows within 24-bit multiplication
    const uint64_t image = uint64_t(IC > OC ? IC : OC) * H * W * 4;
    if (RI < 16 / P8 + 1 || octets > 0x0fffffffull || N * image > 0x7fffffffull || image > 0x1fffffffull || RI >= (1u << 24) ||
        uint64_t(OC) * IC * 36 > 0x7fffffffull)
        return p;
    p.strips = 1;
    p.tiles = ceil_div(u32(octets), 16u);
    p.pairs = ceil_div(OC, u32(C::OCT)) * ceil_div(IC, u32(C::ICT));
    u32 splits = p.pairs >= 256 ? 1 : 256 / p.pairs;  // one workgroup per CU
    if (splits > ceil_div(p.tiles, 4u)) splits = ceil_div(p.tiles, 4u);
    const size_t slice = size_t(OC) * IC * 9 * sizeof(float);
    if (splits > 1 && splits > most / slice) splits = most / slice > 1 ? u32(most / slice) : 1;
    p.tiles_z = ceil_div(p.tiles, splits);
    p.splits = ceil_div(p.tiles, p.tiles_z);
    p.workspace_bytes = p.splits > 1 ? p.splits * slice : 0;
    return p;
}

inline int launch_rows_wgrad(const SplitWgradPlan &p, const float *dY, const float *X, float *dW, float *ws, u32 N, u32 IC, u32 OC, u32 H, u32 W, hipStream_t s,
                             const char *what, PendingSum *later) {
    RowsWgradArgs a;
    a.dY = dY, a.X = X, a.out = p.splits > 1 ? ws : dW;
    a.images = N, a.IC = IC, a.OC = OC, a.H = H, a.W = W, a.HW = H * W;
    a.P8 = W / 8 + 1, a.RI = H + 1, a.NX = 32 + 2 * a.P8;
    a.ic_tiles = ceil_div(IC, u32(RowsWgradCfg::ICT)), a.splits = p.splits, a.tiles = p.tiles, a.tiles_z = p.tiles_z;
    a.p8.init(a.P8), a.ri.init(a.RI);
    if (uint64_t(p.pairs) * p.splits > 0x7fffffffull) return fail(CRB_EINVAL_SHAPE, "%s: launch grid too large", what);
    const dim3 grid(p.pairs * p.splits), block(RowsWgradCfg::NTH);
    const uintptr_t at = reinterpret_cast<uintptr_t>(dY) | reinterpret_cast<uintptr_t>(X) | (uintptr_t(W) * 4);
    if (at % 16 == 0) hipLaunchKernelGGL((rows_wgrad_kernel<4>), grid, block, 0, s, a);
    else if (at % 8 == 0) hipLaunchKernelGGL((rows_wgrad_kernel<2>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((rows_wgrad_kernel<1>), grid, block, 0, s, a);
    if (int st = check_launch(what)) return st;
    if (p.splits > 1 && later) return *later = pending_sum(ws, dW, OC * IC * 9, p.splits), CRB_OK;
    if (p.splits > 1) return launch_splitk_reduce(ws, dW, OC * IC * 9, p.splits, ReduceEpi{nullptr, 1, 1, EPI_ACCUM}, s, what);
    return CRB_OK;
}

}  // namespace crb
