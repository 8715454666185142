// Forward pass of 3x3 / pad 1 / stride 1 layers on few pixels (inference on a handful of images), fp32 MFMA.
//
// Such a layer is its filters read once (512 -> 512 on one 4 x 4 image: 9.4 MB against 64 KB of images) and 75 MFLOP, half a
// microsecond of the matrix pipe if every CU had a share. So tiles are as small as the MFMA allows, 16 output channels x 16
// pixels, the eight waves of a workgroup share a tile's contraction instead of its results (wave w takes two times four channels
// of every 64, nine MFMAs each, one per tap), and where there are fewer tiles than CUs the contraction is cut into slices. Chunks of 64
// channels are staged: the filters' rows lie in memory as [channel][tap], so sixteen of them are read 16 bytes a lane, side by
// side (read as operands, with the lanes of a load on sixteen rows, they came at a quarter of that rate), and a lane's operand of
// a tap is one LDS read (rows 578 floats apart: sixteen rows start in the even banks, the second channel's in the odd ones); of
// the images the window of the tile's pixels with its halo. The next chunk is on its way while one is multiplied. Chains of
// twelve terms are summed by themselves, and the waves' sums in order at the end: bit-reproducible.
//
// What bounds it: 3.5 us of launch, first loads and last sum, 1.3 us a chunk (0.55 of it MFMAs, the rest LDS, loads and barriers of
// a workgroup that is alone on its CU), 2.6 us for summing slices. Against split operands, whose filters take a launch of their
// own and are written and read back (one / four images, us; behind: relative distance from float64, one image):
// 64 -> 64 @32 16.9 -> 5.6 / 17.4 -> 13.1 (8.1e-8 -> 7.2e-8), 128 -> 128 @16 17.9 -> 7.0 / 19.2 -> 11.0 (6.8 -> 6.7), 256 -> 256 @8 20.8 -> 8.1 /
// 22.8 -> 11.4 (7.7 -> 7.2), 512 -> 512 @4 24.6 -> 9.2 / 25.6 -> 13.8 (6.8 -> 6.9), and on 2 x 2 images against the fp32 engine 11.7 -> 7.9 /
// 12.2 -> 8.6 (8.9 -> 6.3).
#pragma once
#include "igemm_engine.h"
#include "split_bf16.h"

namespace crb {

struct ConvFewArgs {
    const float *W, *X, *bias;
    float *Y;
    u32 N, IC, OC, IH, IW;
    u32 tc, tr, imgs;       // a tile: tr rows of tc pixels in each of imgs images, 16 pixels
    u32 tiles_x, tiles_y;   // tiles of an image (imgs == 1)
    u32 px_tiles, oc_tiles, relu;
    u32 ch_z;        // channels of a slice of the contraction (blockIdx.z), whose partial results lie `zstride` floats apart
    u32 z0, add;     // the slice that blockIdx.z == 0 takes, and whether it is added to Y
    size_t zstride;
};

constexpr int kFewCh = 64;         // channels of a chunk
constexpr int kFewWs = 9 * kFewCh + 2, kFewXs = 80;  // floats between two filter rows, two channels' windows

static __global__ void __launch_bounds__(512, 4) conv_few_kernel(ConvFewArgs a) {
    __shared__ __attribute__((aligned(16))) float ws[16 * kFewWs];
    __shared__ __attribute__((aligned(16))) float xs[kFewCh * kFewXs];
    __shared__ __attribute__((aligned(16))) float red[8 * 256];
    // an XCD gets a contiguous run of tiles, the pixel tiles of 16 output channels behind one another: they share filters in its L2
    const u32 ntile = a.px_tiles * a.oc_tiles, q8 = ntile / kXcds, r8 = ntile % kXcds, xcd = blockIdx.x % kXcds;
    const u32 tile = xcd * q8 + (xcd < r8 ? xcd : r8) + blockIdx.x / kXcds;
    const u32 ot = tile / a.px_tiles, pt = tile % a.px_tiles;
    const u32 tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), i16 = lane & 15, q = lane >> 4;
    const u32 HW = a.IH * a.IW, oc0 = ot * 16;
    const u32 z = blockIdx.z + a.z0, cbeg = z * a.ch_z, cend = cbeg + a.ch_z < a.IC ? cbeg + a.ch_z : a.IC;

    // ---- the tile's place, and what this thread stages and reads of it ------------------------------------------------------
    const u32 per_img = a.tiles_x * a.tiles_y, n0 = a.imgs > 1 ? pt * a.imgs : pt / per_img, in_img = a.imgs > 1 ? 0u : pt % per_img;
    const u32 y0 = in_img / a.tiles_x * a.tr, x0 = in_img % a.tiles_x * a.tc;
    const u32 pc = a.tc + 2, win = (a.tr + 2) * pc;  // a window row, an image's window
    const BufferRange xr = buffer_range(a.X, size_t(a.N) * a.IC * HW);
    u32 xoff;  // position `lane` of the window of channel 0
    {
        const u32 m = lane / win, r = lane % win, iy = y0 + r / pc - 1, ix = x0 + r % pc - 1;
        xoff = m < a.imgs && n0 + m < a.N && iy < a.IH && ix < a.IW ? ((n0 + m) * a.IC * HW + iy * a.IW + ix) * 4u : kOutside;
    }
    const u32 pm = i16 / (a.tc * a.tr), pr = i16 / a.tc % a.tr, px = i16 % a.tc;  // this lane's pixel of the tile
    u32 b_at[9];
    u32 inside = 0;  // taps inside the image
#pragma unroll
    for (int t = 0; t < 9; ++t) {
        b_at[t] = q * kFewXs + pm * win + (pr + t / 3) * pc + px + t % 3;
        const u32 iy = y0 + pr + t / 3 - 1, ix = x0 + px + t % 3 - 1;
        if (iy < a.IH && ix < a.IW) inside |= 1u << t;
    }
    const u32 a_at = i16 * kFewWs + q * 9;
    // 16-byte pieces of the filter rows: 144 a row and chunk, the last of a thread's five for half of the threads
    constexpr u32 kQuads = 9 * kFewCh / 4;
    u32 wp[5], quad[5], wl[5];  // (filters: under 2^31 elements)
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        const u32 e = (tid + 512 * i) % (16 * kQuads), row = e / kQuads;
        quad[i] = e % kQuads;
        const u32 oc = oc0 + row < a.OC ? oc0 + row : a.OC - 1;
        wp[i] = oc * a.IC * 9 + (4 * quad[i] < 9 * a.IC ? 4 * quad[i] : 0);
        wl[i] = row * kFewWs + 4 * quad[i];
    }
    const u32 e_oc = oc0 + (tid >> 4), e_i = tid & 15;  // the element this thread finishes (the first 256)
    const bool e_ok = tid < 256 && e_oc < a.OC;
    const float e_bias = a.bias && e_ok ? a.bias[e_oc] : 0.f;

    typedef float v4fu __attribute__((ext_vector_type(4), aligned(4)));
    v4f fw[5];
    float fx[8];
    // (channels past the last read as zero, their filters count as zero)
    auto fetch = [&](u32 c0) {
#pragma unroll
        for (int i = 0; i < 5; ++i) fw[i] = *reinterpret_cast<const v4fu *>(a.W + (wp[i] + (4 * quad[i] < 9 * (a.IC - c0) ? 9 * c0 : 0)));
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const u32 c = c0 + wave + 8 * i;
            fx[i] = buffer_load(xr, c < a.IC ? xoff : kOutside, (c < a.IC ? c : 0u) * HW * 4u);
        }
    };
    auto commit = [&]() {
#pragma unroll
        for (int i = 0; i < 5; ++i)
            if (i < 4 || tid < 256) {
                *reinterpret_cast<v2f *>(ws + wl[i]) = v2f{fw[i].x, fw[i].y};
                *reinterpret_cast<v2f *>(ws + wl[i] + 2) = v2f{fw[i].z, fw[i].w};
            }
#pragma unroll
        for (int i = 0; i < 8; ++i) xs[(wave + 8 * i) * kFewXs + lane] = fx[i];
    };
    // careful: taps outside the image take no part (an infinite filter element makes NaN of the zero read there)
    auto contract = [&](auto careful_c) {
        v4f acc = {0.f, 0.f, 0.f, 0.f};
        // a wave's eight channels of the chunk in six chains of twelve terms, so that a product is rounded into small sums
        auto multiply = [&](u32 c0) {
            float av[2][9], bv[2][9];
            v4f part[2][3];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const u32 unit = wave + 8 * k;  // four channels
#pragma unroll
                for (int c = 0; c < 3; ++c) part[k][c] = v4f{0.f, 0.f, 0.f, 0.f};
                const bool live = c0 + 4 * unit < a.IC;
#pragma unroll
                for (int t = 0; t < 9; ++t) {
                    const float w = ws[a_at + unit * 36 + t];
                    av[k][t] = live ? w : 0.f, bv[k][t] = xs[b_at[t] + unit * (4 * kFewXs)];
                }
            }
#pragma unroll
            for (int j = 0; j < 3; ++j)
#pragma unroll
                for (int c = 0; c < 6; ++c) {
                    const int k = c / 3, t = c % 3 * 3 + j;
                    v4f &p = part[k][c % 3];
                    const v4f sum = __builtin_amdgcn_mfma_f32_16x16x4f32(av[k][t], bv[k][t], p, 0, 0, 0);
                    if constexpr (decltype(careful_c)::value)
#pragma unroll
                        for (int r = 0; r < 4; ++r) p[r] = inside >> t & 1 ? sum[r] : p[r];
                    else
                        p = sum;
                }
            acc += ((part[0][0] + part[0][1]) + part[0][2]) + ((part[1][0] + part[1][1]) + part[1][2]);
        };
        fetch(cbeg);
        for (u32 c0 = cbeg; c0 < cend; c0 += kFewCh) {
            commit();
            lds_barrier();
            if (c0 + kFewCh < cend) fetch(c0 + kFewCh);
            multiply(c0);
            lds_barrier();
        }
        *reinterpret_cast<v4f *>(red + wave * 256 + lane * 4) = acc;
        __syncthreads();
        // element (channel tid / 16, pixel tid % 16): register channel % 4 of lane (channel / 4) * 16 + pixel
        const u32 e = ((tid >> 6 & 3) * 16 + e_i) * 4 + (tid >> 4 & 3);
        float v = red[e];
#pragma unroll
        for (int w = 1; w < 8; ++w) v += red[w * 256 + e];
        return v;
    };
    float v = contract(std::false_type());
    if (__syncthreads_or(tid < 256 && !__builtin_isfinite(v))) v = contract(std::true_type());
    const u32 em = e_i / (a.tc * a.tr), y = y0 + e_i / a.tc % a.tr, x = x0 + e_i % a.tc;
    if (!e_ok || n0 + em >= a.N) return;
    float *yp = a.Y + blockIdx.z * a.zstride + ((n0 + em) * a.OC + e_oc) * HW + y * a.IW + x;
    if (a.add) v = *yp + v;
    v += e_bias;
    if (a.relu) v = v > 0.f ? v : 0.f;
    *yp = v;
}

// Images whose width and height a tile of 16 pixels divides, 2 x 2 images four to a tile.
inline bool conv_few_shape(u32 N, u32 IC, u32 IH, u32 IW) {
    const bool tiles = IW % 16 == 0 || (IW == 8 && IH % 2 == 0) || (IW == 4 && IH % 4 == 0) || (IW == 2 && IH == 2);
    return tiles && IC % 16 == 0 && uint64_t(N) * IC * IH * IW * 4 <= 0x7fffffffull;
}

struct ConvFewPlan {
    u32 px_tiles = 0, oc_tiles, slices, ch_z;  // px_tiles == 0: not taken
};
// Tiles and slices. A chunk takes a workgroup 1.3 us beside 3.5 for the launch, two share a CU (2.3 us for both), and summing
// slices is a launch of 2.6 us.
inline ConvFewPlan conv_few_plan(u32 N, u32 IC, u32 OC, u32 IH, u32 IW) {
    ConvFewPlan p;
    p.px_tiles = IW == 2 ? ceil_div(N, 4u) : N * (IH * IW / 16), p.oc_tiles = ceil_div(OC, 16u);
    const u32 tiles = p.px_tiles * p.oc_tiles, chunks = ceil_div(IC, u32(kFewCh));
    float best = 3e38f;
    for (u32 z = 1; z <= chunks && z <= 16; ++z) {
        const u32 cz = ceil_div(chunks, z);
        if (ceil_div(chunks, cz) != z || (z > 1 && tiles * z > 512)) continue;
        const float us = 1.3f * cz * (tiles * z <= 256 ? 1.f : float(tiles * z) * (2.3f / 1.3f / 256.f)) + (z > 1 ? 2.6f : 0.f);
        if (us < best) best = us, p.slices = z, p.ch_z = cz * kFewCh;
    }
    return p;
}

// part: the slices' partial results, or null (each slice a launch of its own, added to Y: the same bits)
inline int launch_conv_few(const ConvFewPlan &p, const float *W, const float *X, float *Y, const float *bias, float *part, u32 N, u32 IC, u32 OC,
                           u32 IH, u32 IW, u32 relu, hipStream_t s, const char *what) {
    ConvFewArgs a{W, X, bias, Y, N, IC, OC, IH, IW, 0, 0, 1, 0, 0, p.px_tiles, p.oc_tiles, relu, p.ch_z, 0, 0, 0};
    a.tc = IW < 16 ? IW : 16, a.tr = IW == 2 ? 2 : 16 / a.tc, a.imgs = IW == 2 ? 4 : 1;
    a.tiles_x = IW / a.tc, a.tiles_y = IH / a.tr;
    const uint64_t tiles = uint64_t(p.px_tiles) * p.oc_tiles;
    if (tiles > 0x7fffffffull) return fail(CRB_EINVAL_SHAPE, "%s: launch grid too large", what);
    if (p.slices > 1) a.bias = nullptr, a.relu = 0;
    if (p.slices > 1 && part) {
        const u32 count = N * OC * IH * IW;
        a.Y = part, a.zstride = count;
        hipLaunchKernelGGL(conv_few_kernel, dim3(u32(tiles), 1, p.slices), dim3(512), 0, s, a);
        if (int st = check_launch(what)) return st;
        return launch_ordered_reduce(part, Y, count, p.slices, ReduceEpi{bias, IH * IW, OC, relu ? u32(EPI_RELU) : 0u}, s, what);
    }
    for (; a.z0 < p.slices; ++a.z0, a.add = 1) {
        if (a.z0 + 1 == p.slices) a.bias = bias, a.relu = relu;
        hipLaunchKernelGGL(conv_few_kernel, dim3(u32(tiles)), dim3(512), 0, s, a);
        if (int st = check_launch(what)) return st;
    }
    return CRB_OK;
}

}  // namespace crb
