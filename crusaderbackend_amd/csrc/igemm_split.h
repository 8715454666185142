// Contraction engine on split bf16 operands (split_bf16.h):  D(M x N) = sum_k A(m,k) * B(k,n), fp32 in and out.
//
// A workgroup of WM x WN waves owns a BM x BN macro-tile; a wave owns TM x TN blocks of 32 x 32. Operand panels travel
// global -> registers (fp32) -> three bf16 parts -> LDS, one K slab ahead of the MFMAs, double-buffered, one barrier per slab.
// Whatever the operand's orientation in memory, LDS holds MFMA fragments: [part][k / 8][row] units of 16 bytes (eight k of one
// row), so a fragment read is one 16-byte read, 32 lanes on consecutive units. The orientation only decides which elements a
// thread loads: its eight k of a row are consecutive floats (k-contiguous), or it loads RV neighbouring rows of eight
// consecutive k (row-contiguous) and the transposition happens in the packing of its registers, for nothing.
//
// What bounds it: per K step of 16 a wave issues 6 * TM * TN MFMAs (192 clocks per block) against 3 * (TM + TN) fragment reads
// of 1 KB and its share of the split (6.5 VALU operations per staged element), so the ratio of all three goes with the tile
// edge; 2 x 2 blocks per wave keep LDS under the MFMA time, smaller tiles do not.
//
// MFMA 32x32x16 bf16 operand mapping (wave64, lane l): A = A[i = l%32][k = 8*(l/32) + 0..7], B = B[k = 8*(l/32) + 0..7][j = l%32],
// accumulator register r = D[8*(r/4) + 4*(l/32) + r%4][l%32].
#pragma once
#include "igemm_engine.h"
#include "split_bf16.h"

#include <type_traits>

namespace crb {

typedef float v4fu __attribute__((ext_vector_type(4), aligned(4)));  // global loads need no more than the element's alignment
typedef float v2fu __attribute__((ext_vector_type(2), aligned(4)));

// How an operand of the split engine is read.
enum SplitLoad {
    LOAD_K8,   // k-contiguous: a cursor's fetch gives eight k of one row
    LOAD_ROWS  // row-contiguous: eight k of RV neighbouring rows
};

// ---- plain matrices, any size and alignment ----------------------------------------------------------------------------
// A cursor is what a thread keeps of an item: eight consecutive k of RV neighbouring rows. Rows past the matrix are read from
// its last row (their results are never stored); only the last slab of a contraction that BK does not divide is tested (TAIL).

// element(row, k) = base[row*ld + k]; with cat_k a K-concatenated batch (cat_k a multiple of 8): k = nd*cat_k + kk lives at
// base + nd*cat_stride + row*ld + kk
template <bool CAT = false>
struct SMatK {
    static constexpr SplitLoad kLoad = LOAD_K8;
    const float *base;
    u32 rows, ld, zstride;
    u32 cat_stride = 0;
    FastDiv cat_k = FastDiv();
    struct Cursor {
        const float *p;
        u32 k;  // offset of the item's octet inside a slab
    };
    __device__ __forceinline__ void bind(u32 z) { base += size_t(z) * zstride; }
    __device__ __forceinline__ Cursor cursor(u32 row, u32 k) const { return {base + size_t(row < rows ? row : rows - 1) * ld, k}; }
    template <bool TAIL>
    __device__ __forceinline__ void fetch(const Cursor &c, u32 k0, u32 klimit, float (&out)[8]) const {
        const u32 k = k0 + c.k;
        const float *p = c.p;
        if constexpr (CAT) {
            u32 nd, kk;
            cat_k.divmod(TAIL && k >= klimit ? klimit - 8 : k, nd, kk);
            p += size_t(nd) * cat_stride + kk;
        } else {
            p += k;
        }
        if constexpr (!TAIL) {
            const v4fu a = *reinterpret_cast<const v4fu *>(p), b = *reinterpret_cast<const v4fu *>(p + 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) out[i] = a[i], out[4 + i] = b[i];
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                // (past the end: element 0 of the row, which exists, and its value is dropped)
                const float v = *(k + i < klimit ? p + i : c.p);
                out[i] = k + i < klimit ? v : 0.f;
            }
        }
    }
};

// element(row, k) = base[k*ld + row]
struct SMatR {
    static constexpr SplitLoad kLoad = LOAD_ROWS;
    const float *base;
    u32 rows, ld, zstride;
    struct Cursor {
        const float *p;
        u32 k, left;  // rows from the item's first to the matrix' end (0: none, the item repeats the last row)
    };
    __device__ __forceinline__ void bind(u32 z) { base += size_t(z) * zstride; }
    __device__ __forceinline__ Cursor cursor(u32 row, u32 k) const {
        return {base + (row < rows ? row : rows - 1), k, row < rows ? rows - row : 0u};
    }
    // whether some item of the panel at row0 is cut by the matrix' edge and needs element-wise loads
    template <int RV>
    __device__ __forceinline__ bool ragged(u32 row0, u32 panel) const { return RV > 1 && row0 + panel > rows; }
    template <int RV, bool TAIL, bool RAGGED>
    __device__ __forceinline__ void fetch(const Cursor &c, u32 k0, u32 klimit, float (&out)[RV][8]) const {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const u32 k = k0 + c.k + j;
            const bool ok = !TAIL || k < klimit;
            const float *p = c.p + size_t(ok ? k : 0u) * ld;
            float v[RV];
            if constexpr (RAGGED || RV == 1) {
#pragma unroll
                for (int r = 0; r < RV; ++r) v[r] = p[u32(r) < c.left ? r : 0];
            } else if constexpr (RV == 4) {
                const v4fu t = *reinterpret_cast<const v4fu *>(p);
                v[0] = t[0], v[1] = t[1], v[2] = t[2], v[3] = t[3];
            } else {
                const v2fu t = *reinterpret_cast<const v2fu *>(p);
                v[0] = t[0], v[1] = t[1];
            }
#pragma unroll
            for (int r = 0; r < RV; ++r) out[r][j] = ok ? v[r] : 0.f;
        }
    }
};

// KG: wave groups along K (a wave multiplies every KG-th step of a slab; the groups' accumulators are summed through LDS in
// group order at the end), for tiles whose waves would otherwise hold a single block each.
template <int BM_, int BN_, int BK_, int WM_, int WN_, int KG_, int OCC_, bool AHEAD_ = false>
struct SplitCfg {
    static constexpr int BM = BM_, BN = BN_, BK = BK_, WM = WM_, WN = WN_, KG = KG_, OCC = OCC_;
    static constexpr bool AHEAD = AHEAD_;
    static constexpr int NTH = 64 * WM * WN * KG;
    static constexpr int WTM = BM / WM, WTN = BN / WN, TM = WTM / 32, TN = WTN / 32;
    static_assert(TM * 32 * WM == BM && TN * 32 * WN == BN && BK % (16 * KG) == 0, "tile shape");
    static_assert(!AHEAD || BK == 16 * KG, "fragments of the next slab are read ahead one step per wave and slab");
};

// global -> registers -> LDS staging of one ROWS x BK panel
template <class Op, int ROWS, int BK, int NTH>
struct SplitPanel {
    static constexpr int KO = BK / 8;  // octets of a row
    // unit (part p, octet o, row r) at bytes p*PART + o*OCT + 16*r; the pad behind each octet spreads the stores of the
    // k-contiguous loaders (neighbouring lanes on neighbouring octets of one row) over the banks
    static constexpr int OCT = ROWS * 16 + (KO >= 8 ? 16 : (KO >= 4 ? 32 : 64)), PART = KO * OCT, BYTES = kSplit * PART;
    static constexpr int UNITS = ROWS * KO;
    static constexpr SplitLoad L = Op::kLoad;
    static constexpr int RV = L == LOAD_ROWS ? (UNITS / 4 >= NTH ? 4 : (UNITS / 2 >= NTH ? 2 : 1)) : 1;
    static constexpr int ITEMS = UNITS / RV, NP = (ITEMS + NTH - 1) / NTH;
    static_assert(ITEMS % NTH == 0 || ITEMS < NTH, "panel must split evenly over the workgroup");
    float reg[NP][RV][8];
    typename Op::Cursor cur[NP];

    static __device__ __forceinline__ bool active() { return ITEMS >= NTH || threadIdx.x < ITEMS; }
    // Row r of an octet sits in slot r ^ ((r / 8) % 4): eight neighbouring lanes then store to eight different 16-byte slots of a
    // 128-byte bank row whether they hold neighbouring rows or every second or fourth one, and eight neighbouring rows are
    // still read from eight different ones.
    static __device__ __forceinline__ u32 slot(u32 row) { return (row ^ ((row >> 3) & 3)) * 16; }
    // item -> (row, octet): k-contiguous operands put neighbouring lanes on neighbouring octets, the others on neighbouring rows
    static __device__ __forceinline__ void place(int i, u32 &row, u32 &oct) {
        const u32 it = threadIdx.x + i * NTH;
        if constexpr (L == LOAD_K8)
            row = it / KO, oct = it % KO;
        else
            row = (it % (ROWS / RV)) * RV, oct = it / (ROWS / RV);
    }
    __device__ __forceinline__ void init(const Op &op, u32 row0) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            u32 row, oct;
            place(i, row, oct);
            cur[i] = op.cursor(row0 + row, 8 * oct);
        }
    }
    static __device__ __forceinline__ bool ragged(const Op &op, u32 row0) {
        if constexpr (L == LOAD_ROWS) return op.template ragged<RV>(row0, ROWS); else return false;
    }
    // the slab at k0; its K extent is whole unless TAIL, its row groups are whole unless RAGGED
    template <bool TAIL, bool RAGGED>
    __device__ __forceinline__ void fetch(const Op &op, u32 k0, u32 klimit) {
        if (!active()) return;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            if constexpr (L == LOAD_K8)
                op.template fetch<TAIL>(cur[i], k0, klimit, reg[i][0]);
            else
                op.template fetch<RV, TAIL, RAGGED>(cur[i], k0, klimit, reg[i]);
        }
    }
    // sum: null, or the running sums of the rows this thread stages
    __device__ __forceinline__ void commit(unsigned char *lds, float (*sum)[RV] = nullptr) const {
        if (!active()) return;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            u32 row, oct;
            place(i, row, oct);
#pragma unroll
            for (int r = 0; r < RV; ++r) {
                if (sum) {
                    const float *x = reg[i][r];
                    sum[i][r] += ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
                }
                u32x4 part[kSplit];
                split8(reg[i][r], part);
#pragma unroll
                for (int p = 0; p < kSplit; ++p) *reinterpret_cast<u32x4 *>(lds + p * PART + oct * OCT + slot(row + r)) = part[p];
            }
        }
    }
};

template <class Cfg, class AOp, class BOp, class Epi>
__global__ void __launch_bounds__(Cfg::NTH, Cfg::OCC) igemm_split_kernel(AOp a, BOp b, Epi epi, IgemmDims d) {
    constexpr int BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK, TM = Cfg::TM, TN = Cfg::TN, KG = Cfg::KG;
    using PA = SplitPanel<AOp, BM, BK, Cfg::NTH>;
    using PB = SplitPanel<BOp, BN, BK, Cfg::NTH>;
    constexpr int STAGE = PA::BYTES + PB::BYTES;
    __shared__ __attribute__((aligned(16))) unsigned char smem[2 * STAGE];

    u32 tm, tn;
    swizzled_tile(blockIdx.x, d.tiles_m, d.tiles_n, tm, tn);
    const u32 z = blockIdx.z + d.z0;
    u32 kbeg = 0, kend = d.K;
    if (d.split_k) {
        kbeg = z * d.k_per_z;
        kend = kbeg + d.k_per_z < d.K ? kbeg + d.k_per_z : d.K;
        a.bind(0), b.bind(0);
    } else {
        a.bind(z), b.bind(z);
    }
    epi.bind(blockIdx.z);

    const int lane = threadIdx.x & 63, wave = (threadIdx.x >> 6) % (Cfg::WM * Cfg::WN), kgroup = (threadIdx.x >> 6) / (Cfg::WM * Cfg::WN);
    const int wave_m = wave / Cfg::WN, wave_n = wave % Cfg::WN;
    const int i32 = lane & 31, h = lane >> 5;
    const u32 row0 = tm * BM, col0 = tn * BN;

    // epilogues that carry `a_rowsum`: a_rowsum[m] += sum over k of A(m, k), from the registers the panel is staged through, by the
    // workgroups of the first tile column (every workgroup sums, so that no branch stands between the MFMAs)
    constexpr bool kRowSum = Epi::kRowSum && AOp::kLoad == LOAD_ROWS;
    float rsum[PA::NP][PA::RV];
    if constexpr (kRowSum) {
#pragma unroll
        for (int i = 0; i < PA::NP; ++i)
#pragma unroll
            for (int r = 0; r < PA::RV; ++r) rsum[i][r] = 0.f;
    }
    float(*const sum_a)[PA::RV] = kRowSum ? rsum : nullptr;

    PA pa;
    PB pb;
    pa.init(a, row0);
    pb.init(b, col0);
    // the five small part products have accumulators of their own on the 64 x 64 tiles (split_bf16.h)
    constexpr bool kSmall = TM * TN <= 2;
    constexpr int SM = kSmall ? TM : 1, SN = kSmall ? TN : 1;
    v16f acc[TM][TN], small[SM][SN];
#pragma unroll
    for (int mi = 0; mi < TM; ++mi)
#pragma unroll
        for (int ni = 0; ni < TN; ++ni)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mi][ni][r] = 0.0f;
#pragma unroll
    for (int mi = 0; mi < SM; ++mi)
#pragma unroll
        for (int ni = 0; ni < SN; ++ni)
#pragma unroll
            for (int r = 0; r < 16; ++r) small[mi][ni][r] = 0.0f;

    const u32 a_lane = (2 * kgroup + h) * PA::OCT + PA::slot(wave_m * Cfg::WTM + i32);
    const u32 b_lane = (2 * kgroup + h) * PB::OCT + PB::slot(wave_n * Cfg::WTN + i32) + PA::BYTES;
    struct Frags {
        bf16x8 a[kSplit][TM], b[kSplit][TN];
    };
    auto read_frags = [&](Frags &f, const unsigned char *sm, int st) {
#pragma unroll
        for (int i = 0; i < kSplit; ++i) {
            const int p = kPartOrderA[i], q = kPartOrderB[i];
#pragma unroll
            for (int mi = 0; mi < TM; ++mi) f.a[p][mi] = *reinterpret_cast<const bf16x8 *>(sm + a_lane + p * PA::PART + 2 * st * KG * PA::OCT + mi * 512);
#pragma unroll
            for (int ni = 0; ni < TN; ++ni) f.b[q][ni] = *reinterpret_cast<const bf16x8 *>(sm + b_lane + q * PB::PART + 2 * st * KG * PB::OCT + ni * 512);
        }
    };
    auto mfmas = [&](const Frags &f) {
#pragma unroll
        for (int t = 0; t < kTerms; ++t)
#pragma unroll
            for (int mi = 0; mi < TM; ++mi)
#pragma unroll
                for (int ni = 0; ni < TN; ++ni) {
                    v16f &sum = kSmall && t + 1 < kTerms ? small[kSmall ? mi : 0][kSmall ? ni : 0] : acc[mi][ni];
                    sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[kTermA[t]][mi], f.b[kTermB[t]][ni], sum, 0, 0, 0);
                }
    };
    auto multiply = [&](const unsigned char *sm) {
#pragma unroll
        for (int st = 0; st < BK / 16 / KG; ++st) {
            Frags f;
            read_frags(f, sm, st);
            mfmas(f);
        }
    };

    // Two register sets: while slab s is multiplied out of LDS, slab s + 1 (requested one slab ago) is split and stored, and
    // slab s + 2 is requested into the set slab s came in. The split and the LDS traffic are spread between the MFMAs, so that
    // they run in the matrix pipe's shadow even with one wave on a SIMD.
    PA pa2 = pa;
    PB pb2 = pb;
    const u32 nslab = kbeg < kend ? (kend - kbeg + BK - 1) / BK : 0, nwhole = kbeg < kend ? (kend - kbeg) / BK : 0;
    auto main_loop = [&](auto ragged_c) {
        constexpr bool RG = decltype(ragged_c)::value;
        auto fetch = [&](u32 sl, PA &qa, PB &qb) {
            if (sl < nwhole) {
                qa.template fetch<false, RG>(a, kbeg + sl * BK, kend);
                qb.template fetch<false, RG>(b, kbeg + sl * BK, kend);
            } else if (sl < nslab) {
                qa.template fetch<true, true>(a, kbeg + sl * BK, kend);
                qb.template fetch<true, true>(b, kbeg + sl * BK, kend);
            }
        };
        constexpr int NM = TM * TN * kTerms * (BK / 16 / KG);
        constexpr int VPM = ((PA::NP * PA::RV + PB::NP * PB::RV) * 56 + NM - 1) / NM;
        // between two MFMAs: one fragment read, a share of the split's arithmetic, one store to LDS
        auto interleave = [&]() {
#pragma unroll
            for (int i = 0; i < NM; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, VPM, 0);
                __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
            }
        };
        u32 sl = 0;
        if constexpr (Cfg::AHEAD) {
            // Fragments one slab ahead as well: slab s is multiplied out of registers while slab s + 1's fragments are read,
            // slab s + 2 is split and stored over slab s (whose fragments everyone has read), and slab s + 3 is requested. No
            // MFMA waits behind the barrier for a fragment.
            Frags f0, f1;
            if (nslab) {
                fetch(0, pa, pb);
                fetch(1, pa2, pb2);
                pa.commit(smem, sum_a);
                pb.commit(smem + PA::BYTES);
                fetch(2, pa, pb);
                if (1 < nslab) {
                    pa2.commit(smem + STAGE, sum_a);
                    pb2.commit(smem + STAGE + PA::BYTES);
                }
            }
            lds_barrier();
            if (nslab) read_frags(f0, smem, 0);
            lds_barrier();
            // buf: where slab sl lies (and slab sl + 2 will)
            auto step = [&](u32 buf, PA &far_a, PB &far_b, PA &next_a, PB &next_b, const Frags &now, Frags &then) {
                far_a.template fetch<false, RG>(a, kbeg + (sl + 3) * BK, kend);
                far_b.template fetch<false, RG>(b, kbeg + (sl + 3) * BK, kend);
                read_frags(then, smem + (STAGE - buf), 0);
                next_a.commit(smem + buf, sum_a);
                next_b.commit(smem + buf + PA::BYTES);
                mfmas(now);
                interleave();
                lds_barrier();
                ++sl;
            };
            while (sl + 4 < nwhole) {
                step(0, pa2, pb2, pa, pb, f0, f1);
                step(STAGE, pa, pb, pa2, pb2, f1, f0);
            }
            auto last = [&](u32 buf, PA &far_a, PB &far_b, PA &next_a, PB &next_b, const Frags &now, Frags &then) {
                fetch(sl + 3, far_a, far_b);
                if (sl + 1 < nslab) read_frags(then, smem + (STAGE - buf), 0);
                if (sl + 2 < nslab) {
                    next_a.commit(smem + buf, sum_a);
                    next_b.commit(smem + buf + PA::BYTES);
                }
                mfmas(now);
                lds_barrier();
                ++sl;
            };
            while (sl < nslab) {
                last(0, pa2, pb2, pa, pb, f0, f1);
                if (sl < nslab) last(STAGE, pa, pb, pa2, pb2, f1, f0);
            }
        } else {
            if (nslab) {
                fetch(0, pa, pb);
                fetch(1, pa2, pb2);
                pa.commit(smem, sum_a);
                pb.commit(smem + PA::BYTES);
            }
            lds_barrier();
            auto step = [&](u32 buf, PA &free_a, PB &free_b, PA &next_a, PB &next_b) {  // slabs sl + 1, sl + 2 exist and are whole
                free_a.template fetch<false, RG>(a, kbeg + (sl + 2) * BK, kend);
                free_b.template fetch<false, RG>(b, kbeg + (sl + 2) * BK, kend);
                next_a.commit(smem + (STAGE - buf), sum_a);
                next_b.commit(smem + (STAGE - buf) + PA::BYTES);
                multiply(smem + buf);
                __builtin_amdgcn_sched_group_barrier(0x100, TM + TN, 0);
                interleave();
                lds_barrier();
                ++sl;
            };
            while (sl + 3 < nwhole) {
                step(0, pa, pb, pa2, pb2);
                step(STAGE, pa2, pb2, pa, pb);
            }
            auto last = [&](u32 buf, PA &free_a, PB &free_b, PA &next_a, PB &next_b) {
                fetch(sl + 2, free_a, free_b);
                if (sl + 1 < nslab) {
                    next_a.commit(smem + (STAGE - buf), sum_a);
                    next_b.commit(smem + (STAGE - buf) + PA::BYTES);
                }
                multiply(smem + buf);
                lds_barrier();
                ++sl;
            };
            while (sl < nslab) {
                last(0, pa, pb, pa2, pb2);
                if (sl < nslab) last(STAGE, pa2, pb2, pa, pb);
            }
        }
    };
    if (PA::ragged(a, row0) || PB::ragged(b, col0)) main_loop(std::true_type()); else main_loop(std::false_type());

    if constexpr (kRowSum) {
        if (tn == 0 && d.split_k == 0 && epi.a_rowsum) {
            // octets of a row in ascending order (bit-reproducible)
            float *red = reinterpret_cast<float *>(smem);
            if (PA::active()) {
#pragma unroll
                for (int i = 0; i < PA::NP; ++i) {
                    u32 row, oct;
                    PA::place(i, row, oct);
#pragma unroll
                    for (int r = 0; r < PA::RV; ++r) red[oct * BM + row + r] = rsum[i][r];
                }
            }
            __syncthreads();
            for (u32 r = threadIdx.x; r < u32(BM) && row0 + r < d.M; r += Cfg::NTH) {
                float v = red[r];
#pragma unroll
                for (int o = 1; o < PA::KO; ++o) v += red[o * BM + r];
                epi.a_rowsum[row0 + r] += v;
            }
            __syncthreads();
        }
    }
    // ---- sums that are not finite: the block (mi, ni) once more, on the fp32 MFMA from the fp32 operands (split_bf16.h) ------
    // A lane's eight k of a row per step, as the panels are read; two k per MFMA. Ends early where every sum is a NaN.
    auto fp32_block = [&](int mi, int ni) {
        const typename AOp::Cursor ca = a.cursor(row0 + wave_m * Cfg::WTM + mi * 32 + i32, 8 * h);
        const typename BOp::Cursor cb = b.cursor(col0 + wave_n * Cfg::WTN + ni * 32 + i32, 8 * h);
        auto octet = [&](const auto &op, const auto &cur, u32 k0, float (&out)[1][8]) {
            if constexpr (std::decay_t<decltype(op)>::kLoad == LOAD_K8)
                op.template fetch<true>(cur, k0, kend, out[0]);
            else
                op.template fetch<1, true, false>(cur, k0, kend, out);
        };
        v16f sum;
#pragma unroll
        for (int r = 0; r < 16; ++r) sum[r] = 0.0f;
#pragma unroll 1
        for (u32 k0 = kbeg; k0 < kend; k0 += 16) {
            float av[1][8], bv[1][8];
            octet(a, ca, k0, av);
            octet(b, cb, k0, bv);
#pragma unroll
            for (int j = 0; j < 8; ++j) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(av[0][j], bv[0][j], sum, 0, 0, 0);
            u32 numbers = 0;
#pragma unroll
            for (int r = 0; r < 16; ++r) numbers |= __builtin_isnan(sum[r]) ? 0u : 1u;
            if (!__any(int(numbers))) break;
        }
        return sum;
    };

    // ---- epilogue: 32 lanes store 32 consecutive columns of a row ---------------------------------------------------------
    const bool whole = row0 + BM <= d.M && col0 + BN <= d.N;
    const bool accumulates = epi.accumulates(), row_biased = epi.has_row_bias();
    // NR accumulators of block (mi, ni), from register r0 on. Row biases and (accumulating forms, whole tiles) previous values are
    // requested together, ahead of the stores.
    auto store_part = [&](int mi, int ni, int r0, auto nr_c, const float *v) {
        constexpr int NR = decltype(nr_c)::value;
        const u32 col = col0 + wave_n * Cfg::WTN + ni * 32 + i32;
        const typename Epi::ColS cs = epi.prep_col(col, d.N);
        const u32 rbase = row0 + wave_m * Cfg::WTM + mi * 32 + 4 * h + 2 * r0;  // r0 a multiple of 4: register r is row 8 * (r / 4) + r % 4
        float rowb[NR], oldv[NR];
#pragma unroll
        for (int r = 0; r < NR; ++r) rowb[r] = 0.f, oldv[r] = 0.f;
        if (row_biased) {
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const u32 row = rbase + 8 * (r / 4) + (r % 4);
                rowb[r] = epi.row_bias_at(row < d.M ? row : d.M - 1);
            }
        }
        // (nothing is on its way past this point on either path to it: without the wait here the compiler puts one for every
        // load that may have been made, on whichever path, in front of each store: 1003 x 1505 x 777 28.0 -> 29.3 us)
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
        if (whole) {
            if (accumulates) {
#pragma unroll
                for (int r = 0; r < NR; ++r) oldv[r] = *epi.at(rbase + 8 * (r / 4) + (r % 4), col);
            }
#pragma unroll
            for (int r = 0; r < NR; ++r) epi.put(rbase + 8 * (r / 4) + (r % 4), cs, v[r], rowb[r], oldv[r]);
        } else {
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const u32 row = rbase + 8 * (r / 4) + (r % 4);
                if (row < d.M) epi.store(row, cs, v[r], rowb[r]);
            }
        }
    };
    if constexpr (kSmall) add_small(acc, small);
    auto not_finite = [](const float *v, int n) {
        bool bad = false;
        for (int r = 0; r < n; ++r) bad |= !__builtin_isfinite(v[r]);
        return __builtin_expect(__any(int(bad)), 0);
    };
    if constexpr (KG == 1) {
        // (blocks that are not finite wait until the accumulators of the others have been stored: both do not fit the registers)
        u32 again = 0;
#pragma unroll
        for (int ni = 0; ni < TN; ++ni)
#pragma unroll
            for (int mi = 0; mi < TM; ++mi) {
                float v[16];
#pragma unroll
                for (int r = 0; r < 16; ++r) v[r] = acc[mi][ni][r] * kSplitDown;
                if (not_finite(v, 16)) again |= 1u << (mi * TN + ni);
                else store_part(mi, ni, 0, std::integral_constant<int, 16>(), v);
            }
#pragma unroll 1
        for (; again; again &= again - 1) {
            const int blk = __builtin_ctz(again);
            const v16f sum = fp32_block(blk / TN, blk % TN);
            float v[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) v[r] = sum[r];
            store_part(blk / TN, blk % TN, 0, std::integral_constant<int, 16>(), v);
        }
    } else {
        // The groups exchange their accumulators through the staging space (idle: the last slab's barrier has passed), BR blocks
        // of every wave at a time, and each group sums (in group order) and stores its share of them: all waves store.
        constexpr int NB = TM * TN, BR = NB < KG ? NB : KG, NR = BR * 16 / KG;
        static_assert(BR >= 1 && NB % BR == 0 && NR % 4 == 0 && NR <= 16 && BR * 4096 * Cfg::WM * Cfg::WN * KG <= 2 * STAGE, "exchange space");
        float *x = reinterpret_cast<float *>(smem);
        const int f0 = kgroup * NR;  // this group's share of BR blocks' registers
#pragma unroll
        for (int q = 0; q < NB / BR; ++q) {
            if (q) lds_barrier();
            float *dst = x + (kgroup * Cfg::WM * Cfg::WN + wave) * BR * 1024 + lane;
#pragma unroll
            for (int f = 0; f < BR * 16; ++f) dst[f * 64] = acc[(q * BR + f / 16) / TN][(q * BR + f / 16) % TN][f % 16];
            lds_barrier();
            float v[NR];
            const float *src = x + wave * BR * 1024 + f0 * 64 + lane;
#pragma unroll
            for (int r = 0; r < NR; ++r) v[r] = src[r * 64];
#pragma unroll
            for (int g = 1; g < KG; ++g)
#pragma unroll
                for (int r = 0; r < NR; ++r) v[r] += src[g * Cfg::WM * Cfg::WN * BR * 1024 + r * 64];
#pragma unroll
            for (int r = 0; r < NR; ++r) v[r] *= kSplitDown;
            const int blk = q * BR + f0 / 16;
            if (not_finite(v, NR)) {
                const v16f sum = fp32_block(blk / TN, blk % TN);
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    v[r] = sum[r];
#pragma unroll
                    for (int at = NR; at < 16; at += NR) v[r] = f0 % 16 == at ? sum[at + r] : v[r];
                }
            }
            store_part(blk / TN, blk % TN, f0 % 16, std::integral_constant<int, NR>(), v);
        }
    }
}

template <class Cfg, class AOp, class BOp, class Epi>
inline int launch_split(const AOp &a, const BOp &b, const Epi &epi, u32 M, u32 N, u32 K, u32 zdim, u32 k_per_z, hipStream_t stream,
                        const char *what, u32 z0 = 0) {
    IgemmDims d;
    d.M = M, d.N = N, d.K = K;
    d.tiles_m = ceil_div(M, u32(Cfg::BM)), d.tiles_n = ceil_div(N, u32(Cfg::BN));
    d.split_k = k_per_z != 0, d.k_per_z = k_per_z, d.z0 = z0;
    const uint64_t tiles = uint64_t(d.tiles_m) * d.tiles_n;
    if (tiles > 0x7fffffffull || zdim > 65535u) return fail(CRB_EINVAL_SHAPE, "%s: launch grid too large", what);
    hipLaunchKernelGGL((igemm_split_kernel<Cfg, AOp, BOp, Epi>), dim3(u32(tiles), 1, zdim), dim3(Cfg::NTH), 0, stream, a, b, epi, d);
    return check_launch(what);
}

}  // namespace crb
