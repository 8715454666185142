// Small dense products in ONE launch: C (M x N) = A * B with a result of at most a few hundred thousand elements and a
// contraction too short to be worth a split over workgroups plus a second reduction launch (the dense layers of the CIFAR
// networks: 128 x 512 x 512, 128 x 10 x 512 and their gradients). A workgroup owns one 16 x 16 block of C; its four (long contractions:
// eight, sixteen) waves each take their share of the contraction, fed straight from global memory (the operands are L2-resident at these sizes,
// so there is no LDS staging), and their accumulators are summed through LDS in wave order: bit-reproducible.
//
// v_mfma_f32_16x16x4_f32 (wave64, lane l): A value = A[i = l%16][k = l/16], B value = B[k = l/16][j = l%16], accumulator
// register r = C[4*(l/16) + r][l%16]. When both operands are contiguous along k, a lane loads 16 bytes — the k values
// 16 s + 4 (l/16) + t, t = 0..3 — and feeds them to four MFMAs in turn (A and B agree on the order, which is all the
// contraction needs). That load asks for no more than the element's alignment: rows of any length at any address take it, and
// up to three k past the last quad are one MFMA more. Element by element a lane's 64 loads of a row share a line with three
// other lanes only, sixteen lines an instruction (NT, K no multiple of 4, us: 255 x 257 x 2047 38.1 -> 16.4, 63 x 1025 x 2047
// 37.9 -> 17.2, 30 x 510 x 4090 44.2 -> 16.1, 126 x 510 x 1022 12.9 -> 5.9, 62 x 1022 x 1022 12.9 -> 6.1).
#pragma once
#include "igemm_engine.h"

#include <type_traits>

namespace crb {

struct TinyGemmArgs {
    const float *A, *B;
    float *C;
    const float *col_bias;  // per column, or nullptr
    const float *row_bias;  // per row, or nullptr
    u32 M, N, K;
    u32 a_rs, a_ks;  // element (i, k) of A at A[i * a_rs + k * a_ks]
    u32 b_ks, b_cs;  // element (k, j) of B at B[k * b_ks + j * b_cs]
    u32 ldc, flags;  // EPI_ACCUM | EPI_RELU
    u32 k_per_wave;  // multiple of 16
    u32 tiles_n;
    // K-concatenated batch (the accumulate-NT form): contraction index kk = nd * kb_len + k addresses A + nd * a_bs, B + nd * b_bs;
    // K is then batch * kb_len. Without a batch kb_len = K.
    u32 a_bs, b_bs;
    FastDiv kb_len;
    // optional second result: a_rowsum[i] += sum over k of A(i, k), formed by the workgroups of the first block column
    // (lanes, then waves, in fixed order: bit-reproducible)
    float *a_rowsum = nullptr;
};

// Register t of lane group g (of four) <-> register g of lane group t.
__device__ __forceinline__ v4f exchange_groups(v4f v) {
    typedef u32 u32x4 __attribute__((ext_vector_type(4)));
    u32x4 r = __builtin_bit_cast(u32x4, v);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const auto p = __builtin_amdgcn_permlane32_swap(r[t], r[t + 2], false, false);
        r[t] = p[0], r[t + 2] = p[1];
    }
#pragma unroll
    for (int t = 0; t < 4; t += 2) {
        const auto p = __builtin_amdgcn_permlane16_swap(r[t], r[t + 1], false, false);
        r[t] = p[0], r[t + 1] = p[1];
    }
    return __builtin_bit_cast(v4f, r);
}

// A lane's place in a K-concatenated batch: offsets of its element of A and of B, which go on by addition (behind the batch's end they are not used).
struct BatchWalk {
    u32 kr, oa, ob;
    __device__ __forceinline__ BatchWalk(const TinyGemmArgs &a, const float *pa, const float *pb, u32 kk) {
        u32 nd;
        a.kb_len.divmod(kk, nd, kr);
        oa = u32(pa - a.A) + nd * a.a_bs + kr * a.a_ks, ob = u32(pb - a.B) + nd * a.b_bs + kr * a.b_ks;
    }
    __device__ __forceinline__ void step(const TinyGemmArgs &a, u32 n) {
        const u32 len = a.kb_len.d;
        kr += n, oa += n * a.a_ks, ob += n * a.b_ks;
        if (len >= n) {  // at most one entry on
            const bool over = kr >= len;
            kr -= over ? len : 0u, oa += over ? a.a_bs - len * a.a_ks : 0u, ob += over ? a.b_bs - len * a.b_ks : 0u;
        } else {
            u32 nd;
            a.kb_len.divmod(kr, nd, kr);
            oa += nd * (a.a_bs - len * a.a_ks), ob += nd * (a.b_bs - len * a.b_ks);
        }
    }
};

// BATCH: a K-concatenated batch of more than one entry. Without one, whole groups of sixteen k are loaded from addresses that are a lane's
// constant offset behind a uniform one and need no vector arithmetic (a division by the entry's length, a 64-bit product and the tests of
// row, column and k for every load were most of the kernel's instructions). Us, before / after: NN 128 x 512 x 512 6.6 / 4.0, 256 x 256 x 1024 11.2 /
// 5.8, TN 128 x 512 x 512 5.4 / 3.3, 128 x 128 x 2048 15.1 / 7.1, NT 128 x 512 x 512 4.5 / 4.0, 256 x 256 x 1024 6.7 / 5.7; up to 640 terms the same bits (beyond
// them the contraction is cut over more waves: tiny_gemm_waves). What bounds it now is a launch (3 us of these) and the reading of every block's rows from L2.
template <bool KVEC, bool BATCH, int WAVES>
__global__ void __launch_bounds__(64 * WAVES) tiny_gemm_kernel(TinyGemmArgs a) {
    __shared__ __attribute__((aligned(16))) float red[WAVES * 256];
    __shared__ float rsum[WAVES * 64];
    const u32 t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const u32 li = lane & 15, g = lane >> 4;
    const u32 row0 = (blockIdx.x / a.tiles_n) * 16, col0 = (blockIdx.x % a.tiles_n) * 16;
    const u32 kb = wave * a.k_per_wave;
    const u32 ke = kb + a.k_per_wave < a.K ? kb + a.k_per_wave : a.K;
    // What the epilogue adds to the element this thread finishes (row t / 16, column t % 16) is requested now: loaded at
    // the end, bias and previous value would each cost a memory round trip of their own.
    const u32 er = t >> 4 & 15, ec = t & 15;
    const u32 erow = row0 + er, ecol = col0 + ec;
    const bool e_ok = t < 256 && erow < a.M && ecol < a.N;
    float *ep = a.C + size_t(e_ok ? erow : 0) * a.ldc + (e_ok ? ecol : 0);
    const float e_cb = (a.col_bias && e_ok) ? a.col_bias[ecol] : 0.f;
    const float e_rb = (a.row_bias && e_ok) ? a.row_bias[erow] : 0.f;
    const float e_old = ((a.flags & EPI_ACCUM) && e_ok) ? *ep : 0.f;
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    float asum = 0.f;  // this lane's share of row li's sum of A
    // (rows and columns past the last are read from the last one: nothing is stored of them)
    const float *pa = a.A + size_t(row0 + li < a.M ? row0 + li : a.M - 1) * a.a_rs;
    const float *pb = a.B + size_t(col0 + li < a.N ? col0 + li : a.N - 1) * a.b_cs;
    u32 k = kb;
    // `whole(n)`: the next n groups of sixteen k, all inside; requested together
    auto groups = [&](auto whole) {
        for (; k + 64 <= ke; k += 64) whole(std::integral_constant<int, 4>());
        const u32 left = k < ke ? (ke - k) / 16 : 0;
        if (left == 3) whole(std::integral_constant<int, 3>());
        else if (left == 2) whole(std::integral_constant<int, 2>());
        else if (left == 1) whole(std::integral_constant<int, 1>());
        k += 16 * left;
    };
    typedef float v4fu __attribute__((ext_vector_type(4), aligned(4)));
    if constexpr (KVEC) {
        // both operands contiguous along k; a batch entry's contraction a multiple of 4
        const u32 kq = ke & ~3u;
        auto add = [&](const v4f &va, const v4f &vb) {
            asum += (va.x + va.y) + (va.z + va.w);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(va.x, vb.x, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(va.y, vb.y, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(va.z, vb.z, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(va.w, vb.w, acc, 0, 0, 0);
        };
        if constexpr (!BATCH) {
            const float *qa = pa + 4 * g, *qb = pb + 4 * g;
            groups([&](auto n_c) {
                constexpr int n = decltype(n_c)::value;
                v4f va[n], vb[n];
#pragma unroll
                for (int u = 0; u < n; ++u) va[u] = *reinterpret_cast<const v4fu *>(qa + k + 16 * u), vb[u] = *reinterpret_cast<const v4fu *>(qb + k + 16 * u);
#pragma unroll
                for (int u = 0; u < n; ++u) add(va[u], vb[u]);
            });
        }
        constexpr int U = BATCH ? 4 : 1;  // 16-k groups requested together (without a batch: what is left of the last one)
        BatchWalk at(a, pa, pb, k + 4 * g);
        for (; k < kq; k += 16 * U) {
            v4f va[U], vb[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const u32 kk = k + 16 * u + 4 * g;
                const bool in = kk < kq;  // kq, kk and a batch entry's length are multiples of 4: a quad is inside or outside as a whole
                if constexpr (BATCH) {
                    va[u] = *reinterpret_cast<const v4fu *>(a.A + (in ? at.oa : 0)), vb[u] = *reinterpret_cast<const v4fu *>(a.B + (in ? at.ob : 0));
                    at.step(a, 16);
                } else {
                    va[u] = *reinterpret_cast<const v4fu *>(pa + (in ? kk : 0)), vb[u] = *reinterpret_cast<const v4fu *>(pb + (in ? kk : 0));
                }
                if (!in) va[u] = vb[u] = v4f{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int u = 0; u < U; ++u) add(va[u], vb[u]);
        }
        if (kq < ke && kb <= kq) {  // K % 4 more (no batch then), in the wave that holds them
            const bool in = kq + g < ke;
            const float va = in ? pa[kq + g] : 0.f, vb = in ? pb[kq + g] : 0.f;
            asum += va;
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(va, vb, acc, 0, 0, 0);
        }
    } else {
        auto add = [&](float va, float vb) {
            asum += va;
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(va, vb, acc, 0, 0, 0);
        };
        if constexpr (!BATCH) {
            const u32 la = u32(pa - a.A) + g * a.a_ks, lb = u32(pb - a.B) + g * a.b_ks;
            const float *qa = pa + 4 * g;
            auto fetch_b = [&](auto n_c, float *vb) {
#pragma unroll
                for (int u = 0; u < 4 * decltype(n_c)::value; ++u) vb[u] = (a.B + size_t(k + 4 * u) * a.b_ks)[lb];
            };
            if (a.a_ks == 1) {
                // A contiguous along k: a lane loads four k and the lane groups exchange them (register t of group g, k = 4 g + t, becomes register
                // g of group t), so that the sum's order is the same
                groups([&](auto n_c) {
                    constexpr int n = decltype(n_c)::value;
                    v4f va[n];
                    float vb[4 * n];
#pragma unroll
                    for (int u = 0; u < n; ++u) va[u] = *reinterpret_cast<const v4fu *>(qa + k + 16 * u);
                    fetch_b(n_c, vb);
#pragma unroll
                    for (int u = 0; u < n; ++u) {
                        const v4f q = exchange_groups(va[u]);
#pragma unroll
                        for (int i = 0; i < 4; ++i) add(q[i], vb[4 * u + i]);
                    }
                });
            } else {
                groups([&](auto n_c) {
                    constexpr int n = decltype(n_c)::value;
                    float va[4 * n], vb[4 * n];
#pragma unroll
                    for (int u = 0; u < 4 * n; ++u) va[u] = (a.A + size_t(k + 4 * u) * a.a_ks)[la];
                    fetch_b(n_c, vb);
#pragma unroll
                    for (int u = 0; u < 4 * n; ++u) add(va[u], vb[u]);
                });
            }
        }
        constexpr int U = BATCH ? 16 : 4;  // MFMA steps requested together (without a batch: what is left of the last group)
        BatchWalk at(a, pa, pb, k + g);
        for (; k < ke; k += 4 * U) {
            float va[U], vb[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const u32 kk = k + 4 * u + g;
                const bool in = kk < ke;
                if constexpr (BATCH) {
                    va[u] = a.A[in ? at.oa : 0], vb[u] = a.B[in ? at.ob : 0];
                    at.step(a, 4);
                } else {
                    va[u] = pa[size_t(in ? kk : 0) * a.a_ks], vb[u] = pb[size_t(in ? kk : 0) * a.b_ks];
                }
                if (!in) va[u] = vb[u] = 0.f;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) add(va[u], vb[u]);
        }
    }
    *reinterpret_cast<v4f *>(red + wave * 256 + lane * 4) = acc;
    const bool do_rowsum = a.a_rowsum && col0 == 0;
    if (do_rowsum) rsum[t] = asum;
    __syncthreads();
    if (do_rowsum && t < 16 && row0 + t < a.M) {
        float v = 0.f;
#pragma unroll
        for (int q = 0; q < 4 * WAVES; ++q) v += rsum[q * 16 + t];  // wave q / 4, k lane group q % 4
        a.a_rowsum[row0 + t] += v;
    }
    // thread t finishes element (row t / 16, column t % 16): register row % 4 of lane (row / 4) * 16 + column
    if (!e_ok) return;
    const u32 e = ((er >> 2) * 16 + ec) * 4 + (er & 3);
    float v = red[e];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) v += red[w * 256 + e];
    if (a.col_bias) v += e_cb;
    if (a.row_bias) v += e_rb;
    if (a.flags & EPI_ACCUM) v += e_old;
    if (a.flags & EPI_RELU) v = v > 0.f ? v : 0.f;
    *ep = v;
}

// Whether the one-launch form takes a product ahead of all others: a small result, a contraction short enough that a quarter of it per wave is
// a few dozen MFMA steps, and enough 16 x 16 blocks (or little enough work) that the chip is not left idle for long.
// K: the whole contraction (batch * K for the K-concatenated accumulate-NT form); batch: independent products (must be 1).
// kfast: both operands are contiguous along k (the NT forms: 16-byte loads). Every block re-reads its operand rows from L2,
// so beyond 2^27 multiply-adds (2^26 with scalar loads) the staged engine wins again (measured, batch 128: 1024 x 1024 one
// launch 9.6 us against 12.9, 1024 x 4096 32.4 against 22.6; data-gradient form 1024 x 512 9.6 against 11.4, 1024 x 1024
// 17.7 against 12.8).
inline bool tiny_gemm_fits(u32 M, u32 N, u32 K, u32 batch, bool kfast = false) {
    if (batch != 1 || uint64_t(M) * N > 512u * 512u || K > 4096u) return false;
    if (uint64_t(M) * N * K > (uint64_t(1) << (kfast ? 27 : 26))) return false;
    const u32 blocks = ceil_div(M, 16u) * ceil_div(N, 16u);
    return blocks >= 64u || uint64_t(M) * N * K <= (1u << 22);
}

// Products that would go to the fp32 engine: where that has too few tiles for the chip or cuts the contraction, a workgroup for every 16 x 16 block is
// ahead as long as the chip takes the blocks in two rounds of eight on a CU and they re-read no more than `blocks_k` k of their operands (us, engine / here:
// 128 x 96 x 352 11.3 / 3.7, 41 x 315 x 818 12.0 / 4.2, 2304 x 144 x 224 11.0 / 5.9, 1088 x 256 x 64 4.7 / 3.4, 60 x 3268 x 526 12.5 / 11.7; beyond,
// 1958 x 802 x 18, 6273 blocks, 6.5 / 9.9).
// `blocks_k` goes by the form: 2^20 for NN, which the engine is slowest at (368 x 784 x 896 19.2 / 13.8, 3136 x 80 x 608 17.2 / 10.0), 5 * 2^17 for NT (117 x 951 x
// 1284 15.6 / 9.0; beyond 64 x 3584 x 896 14.0 / 15.1), 27 * 2^14 for TN (beyond 1984 x 64 x 960 10.8 / 11.1, 1064 x 124 x 1640 16.2 / 20.1).
// Blocks go to the XCDs in turn, so each of these reads all rows of A that its columns meet and, unless a row of blocks is a multiple of eight, all columns
// of B: a number of floats from beyond the L2s that is held to `far`. Sixteen waves (more than 1024 terms) hide less of it, two workgroups on a CU instead of eight, and
// are held to `far_long`. Beyond, 103 x 3732 x 640 16.5 / 24.5, 64 x 2240 x 1536 14.9 / 22.2, NT 1104 x 64 x 2016 11.4 / 17.2, TN 1536 x 64 x 1152 10.9 / 13.2. NT rows that
// are no whole quads, which the engine loads a float at a time, gain in all cases. Of 24000 random products of up to 2048 blocks and terms, 2^14 to 2^20 block rows (0.63 / 0.69 / 0.83
// of the engine's time in the mean, NN / TN / NT), 22 are slower by more than a twentieth, by 1.23 at most; of 9000 of all sizes none.
struct TinyLines {
    u32 blocks_k, far, far_long;
};
constexpr TinyLines kTinyNN{1u << 20, 10000000, 8000000}, kTinyTN{27u << 14, 10000000, 6000000}, kTinyNT{5u << 17, ~0u, 8000000}, kTinyNTRagged{5u << 17, ~0u, ~0u};
inline bool tiny_gemm_beats_engine(u32 M, u32 N, u32 K, u32 batch, const TinyLines &most) {
    const uint64_t tm = ceil_div(M, 16u), tn = ceil_div(N, 16u), blocks = tm * tn;
    if (batch != 1 || K > 2048u || blocks > 2048u || blocks * K > most.blocks_k) return false;
    const uint64_t far = K * (M * (tn < kXcds ? tn : kXcds) + N * (tn % kXcds == 0 ? 1 : tm < kXcds ? tm : kXcds));
    return far <= (K > 1024u ? most.far_long : most.far);
}

// Waves of a workgroup, which share its contraction. More of them keep the chains of a long one short, in time (us, 4 / 8 / 16 waves: NT 11 x 2012 x
// 3053 15.1 / 10.5 / 10.8, 13 x 107 x 2127 7.5 / 6.8 / 7.0) and in roundings (TN 112 x 112 x 1200 3.2 / 2.3 / 1.8e-7 from float64, the engine, which
// cuts it, 2.2e-7; 502 x 15 x 614 2.3e-7 on either). Up to 640 terms four stay: these products were here before there were others, the bits of a VGG-16 head among
// them, and eight from 257 on would bring little: 6000 random products 0.99 of the time in the mean, 110 slower by more than a twentieth, by 1.23 at most, nearly all of
// these under 480 terms (480 to 640: 0.98).
// A batch stays on four, whose loads are more arithmetic than a chain (NTA 82 x 14 x 10 * 225 on sixteen: a 1x1 layer's three passes 35.6 -> 41.4).
inline u32 tiny_gemm_waves(u32 K, bool batch) { return batch || K <= 640u ? 4u : (K <= 1024u ? 8u : 16u); }

// kb_len: length of one batch entry's contraction (a.K for a plain product); a.K = the whole contraction.
inline int launch_tiny_gemm(TinyGemmArgs a, u32 kb_len, u32 a_bs, u32 b_bs, hipStream_t s, const char *what) {
    a.kb_len = FastDiv(kb_len), a.a_bs = a_bs, a.b_bs = b_bs;
    a.tiles_n = ceil_div(a.N, 16u);
    const u32 blocks = ceil_div(a.M, 16u) * a.tiles_n, waves = tiny_gemm_waves(a.K, kb_len != a.K);
    a.k_per_wave = ceil_div(ceil_div(a.K, waves), 16u) * 16u;
    const bool kvec = a.a_ks == 1 && a.b_ks == 1 && (kb_len == a.K || (kb_len % 4 == 0 && a_bs % 4 == 0 && b_bs % 4 == 0));
    auto launch = [&](auto w_c) {
        constexpr int W = decltype(w_c)::value;
        if (kvec) hipLaunchKernelGGL((tiny_gemm_kernel<true, false, W>), dim3(blocks), dim3(64 * W), 0, s, a);
        else hipLaunchKernelGGL((tiny_gemm_kernel<false, false, W>), dim3(blocks), dim3(64 * W), 0, s, a);
    };
    if (kb_len != a.K) {
        if (kvec) hipLaunchKernelGGL((tiny_gemm_kernel<true, true, 4>), dim3(blocks), dim3(256), 0, s, a);
        else hipLaunchKernelGGL((tiny_gemm_kernel<false, true, 4>), dim3(blocks), dim3(256), 0, s, a);
    } else if (waves == 4) launch(std::integral_constant<int, 4>());
    else if (waves == 8) launch(std::integral_constant<int, 8>());
    else launch(std::integral_constant<int, 16>());
    return check_launch(what);
}

}  // namespace crb
