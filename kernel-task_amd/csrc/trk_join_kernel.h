#pragma once
// The joined-core family of the fused tensor-ring kernel (ring3_join), for token counts that
// amortise forming weight tiles: G2 and G3 are joined over their shared ring link, the joined
// slice meets G1, and x meets the result last.
//
//   H[(j,k)][(a,b)]   = sum_c G2[b,q,j,c] G3[c,r,k,a]               for one output pair (q,r)
//   Wt[(j,k)][p]      = sum_{a,b} H[(j,k)][(a,b)] G1[a,p,i,b]       for one input digit i
//   Y[t][p]          += sum_{(j,k)} x[t,i,(j,k)] Wt[(j,k)][p]
//
// The chains of trk_mfma_kernel.h take x through one core after another, which costs
// R^3 per (stage-2 input, output) pair and token; here a token costs its share of the
// in x out products plus R^2 / TT of them for the tile's formation, TT tokens sharing one.
// No weight is ever stored: a wave forms 32 x 16 values at a time, in the registers that its
// next MFMAs read, and drops them.
//
// Everything between the core loads and y is held in registers. (Two kinds of kernels spill some:
// 1920 -> 2880 R16 fp16 with 256 tokens a workgroup, 19 VGPRs, and most fused pairs, which keep the
// gate's results through the second pass, up to 189; their times chose them all the same.) In a
// 16x16 MFMA a lane holds four consecutive rows of one result column; as an operand it holds eight
// K positions of one row or column. So a result whose rows are the next contraction's index becomes that
// contraction's operand without leaving the lane, two 16-row results making one 32-wide K
// step (rounded to the plan's type on the way, as U and V are in the chains), provided the
// other operand orders its K the same way:
//   H    two results (rows b; rank 8: two a's of 8 rows each) make a K step of (a, b), the order
//        G1's fragments are packed in (trk_pack.hip)
//   Wt   results ft = 0, 1 (16 features (j,k) each) make a K step of 32: lane group g holds
//        features 4 g .. 4 g + 3 of both, and x is laid out in LDS in that order
//
// Work split: a workgroup owns TT tokens x (FC x SC) output pairs x all p. KW of its 4 or 8 waves
// split the feature chunks (their partial sums meet in LDS at the end), the others the pairs:
// KW = 4 or 8 with one or two pairs where token tiles are few and the chip has to be filled with
// narrow tiles, KW = 1 with up to 16 where it is full, as the waves then share x and G1's fragments.
// The steps (chunk of 32 features, digit i) run in lockstep over two LDS buffers. Four waves leave
// a SIMD one wave of up to 512 registers, whose tile amortises formation best (large calls); eight
// leave it two of half the size, and one issues while the other waits: 5120 -> 12288 R16 T=128 63 ->
// 59 us, 1920 -> 2880 R16 T=32 9.6 -> 8.0 us, R8 T=1023 31.5 -> 29 us.
//
// What bounds it: at KW = 1 matrix cores (2-3 times the dense product's work at rank 16: R^2 / TT
// of formation) and the waits between them; at KW = 4 and 8, where every wave reads its own x and
// all of G1's fragments, LDS as well. Counters at 14336 -> 4096, rank 16, 256 tokens, when that took
// 94 us: matrix cores busy 46 % of a CU's clocks, LDS 76 %, a third of that in bank conflicts of x's
// stores and of the join's reads of G3; with the offsets of x_at, the swap of x_swap and the pad P3K,
// each of which spreads the 16 lanes that one pass serves, 94 -> 90 us there, 5120 -> 12288 R16
// T=128 59 -> 55.6 us, 5120 -> 1024 R12 T=300 29.5 -> 27.4 us. Measured against the chains on the same
// card: 213 -> 90, 151 -> 55.6 and 74.8 -> 27.4 us; 17408 -> 5120 R16 T=2048 12660 -> 730 us (1.2
// PFLOP/s with the formation); 1920 -> 2880 R8 T=1023 50.7 -> 28.5 us, fp32 T=100 41.7 -> 37.3 us.
#include "trk_mfma_kernel.h"

namespace trk {
namespace {

using u32x4 = unsigned __attribute__((ext_vector_type(4)));
using u32x2 = unsigned __attribute__((ext_vector_type(2)));

template <KCfg C>
struct JoinGeo {
    static constexpr int R = C.R, R2 = R * R;
    static constexpr int nI = C.i0, nJ = C.i1, nK = C.i2, oP = C.o0, oQ = C.o1, oR = C.o2;
    static constexpr int IN = nI * nJ * nK, OUT = oP * oQ * oR, NJK = nJ * nK;
    static constexpr int EB = C.dt == TRK_DTYPE_F32 ? 4 : 2, VPE = 16 / EB;
    static constexpr int TT = C.TT, MT = TT / 16, FC = C.FC, SC = C.SC;
    static constexpr int NW = C.NW, NT = 64 * NW, KW = C.KS3, QW = NW / KW;
    static constexpr int WPC = C.NACC;            // workgroups per CU the registers leave room for
    static constexpr int NQ = FC * SC / QW;       // output pairs per wave
    static constexpr bool XS = KW == 1;           // the waves share x
    static constexpr int KS = R2 / 32;            // K steps of the formation
    static constexpr int NCH = cdiv(NJK, 32);     // chunks of 32 features
    static constexpr int NR = cdiv(NCH, KW);      // chunks a wave works through
    static constexpr bool PAD = NR * KW * 32 != NJK;  // some are empty, or end early: zeros
    static constexpr int NST = NR * nI;           // steps: (chunk, digit of i)
    static constexpr int FRAG = 512;              // elements of one operand fragment
    static constexpr int GPT = cdiv(KS * FRAG / VPE, NT);  // G1 vectors per thread and step
    // x of a step: TT rows of 32 KW features, loaded 16 bytes a lane, LPR lanes a row, so a wave
    // loads RPI rows at once, XN times; XPER of those until the rows repeat modulo 16
    static constexpr int LPR = KW * 32 * EB / 16, RPI = 64 / LPR, XN = cdiv(TT, NW * RPI);
    static constexpr int XPER = NW * RPI < 16 ? 16 / (NW * RPI) : 1;
    static constexpr int NRW = NQ < SC ? NQ : SC; // distinct r among a wave's pairs
    // H's MFMAs, one result (16 features) each: K = c alone where those lie in one j (rank 8: a
    // block diagonal of two a), else two j and c, NH of them for the j that a tile may span
    static constexpr bool SJ = nK % 16 == 0;
    static constexpr int span() {
        int worst = 1;
        for (int f = 0; f < NJK; f += 16) {
            const int last = f + 15 < NJK ? f + 15 : NJK - 1;
            worst = last / nK - f / nK + 1 > worst ? last / nK - f / nK + 1 : worst;
        }
        return worst;
    }
    static constexpr int NH = SJ ? 1 : cdiv(span(), 2);
    // packed section (trk_pack.hip): header (the output scale), then
    // J1[i][K step][lane][8], J2[q][j][b][c], J3[r][k][a][c]
    static constexpr int oJ1 = kJoinHeader / EB;
    static constexpr int oJ2 = oJ1 + nI * KS * FRAG;
    static constexpr int oJ3 = oJ2 + oQ * nJ * R2;
    // LDS, in elements: the workgroup's slices of G2 and G3 (rows of one k 16 bytes past
    // a multiple of the banks, which 8-byte reads of neighbouring k fill in order; 16-byte reads 32),
    // R^2 zeros, two steps of G1's fragments and of x; at the end the partial sums (KW > 1) or 64 tokens of y
    // replace them all
    static constexpr int P3K = R2 + (SJ ? 8 : 16);
    static constexpr int szJ2 = FC * nJ * R2, szJ3 = SC * nK * P3K, szG1 = KS * FRAG;
    // one step's x of one chunk: the rows loaded at once are stored without a branch (it would cut
    // the step's schedule in two: 5120 -> 17408 R16 T=160, TT = 160 over 8 waves, 112 -> 106 us), so
    // there is room for those past the tile
    static constexpr int XROWS = XN * NW * RPI > TT ? XN * NW * RPI : TT;
    // chunk c starts x_at(c) into a step's region: the 16 lanes that one pass of a store serves write
    // a row of four chunks (KW >= 4), and these offsets give their halves of 16 bytes different banks
    static constexpr int x_at(int c) {
        return c * (XROWS / 16 * FRAG) + (EB == 2 ? c % 2 * VPE + c / 2 * 4 * VPE : c * VPE);
    }
    static constexpr int szX = KW == 1 ? XROWS / 16 * FRAG : x_at(KW) + VPE;  // one step's x
    static constexpr int lJ3 = szJ2, lZ = lJ3 + szJ3, lG1 = lZ + R2, lX = lG1 + 2 * szG1;
    static constexpr int TILES = NQ * MT, TPW = cdiv(TILES, KW);  // y tiles, per storing wave
    // y through LDS (XS): [token][pair][p], a token's floats 4 words past a multiple of 64
    static constexpr int YG = MT < 4 ? MT : 4, YP = FC * SC * 16 + 4;
    static constexpr int RED_BYTES = KW > 1 ? NW * TILES * 1024 : YG * 16 * YP * 4;
    static constexpr int LDS_BYTES =
        (lX + 2 * szX) * EB > RED_BYTES ? (lX + 2 * szX) * EB : RED_BYTES;
    static constexpr int NBLK = cdiv(oQ, FC) * cdiv(oR, SC);

    static_assert(C.F == 1 && C.S == 2 && C.L == 0, "the joined family joins G2 and G3");
    static_assert(R == 8 || R == 16, "joined tiles are written for ring ranks 8 and 16");
    static_assert(oP <= 16 && C.LC == oP, "a joined tile holds all p in 16 columns");
    static_assert(NJK % 8 == 0 && NJK >= 32 && IN % VPE == 0, "x is read 8 features at a time");
    static_assert(nI % 2 == 0 && C.IC == 1, "steps of one digit of i, in pairs");
    static_assert(NQ % NRW == 0 && SC % NRW == 0, "a wave's pairs are whole rows or parts of one");
    static_assert(TT % 16 == 0 && FC * SC % QW == 0 && NW % KW == 0 && FC <= oQ && SC <= oR,
                  "joined tile");
    static_assert(LDS_BYTES <= 160 * 1024, "joined tile exceeds the 160 KB of LDS");
};

// One operand fragment from a fragment-ordered section, p at this lane's first 16 bytes:
// element u of lane l at l * 8 + u in 16 bits; in 32 bits as two planes of 4 ([u / 4][l][u % 4]),
// so that each read is 16 bytes a lane, contiguous.
template <class O>
__device__ __forceinline__ typename O::V8 join_read(const typename O::E *p) {
    if constexpr (sizeof(typename O::E) == 2) {
        return *reinterpret_cast<const typename O::V8 *>(p);
    } else {
        const f32x4 lo = *reinterpret_cast<const f32x4 *>(p);
        const f32x4 hi = *reinterpret_cast<const f32x4 *>(p + 256);
        return typename O::V8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    }
}

// A vector of consecutive elements at the alignment of its first 16 bytes.
template <class V, class E>
__device__ __forceinline__ V join_load(const E *p) {
    using VA = V __attribute__((aligned(sizeof(V) < 16 ? sizeof(V) : 16)));
    return *reinterpret_cast<const VA *>(p);
}

// Two results (rows 4g .. 4g+3 of one column each) as one K step of the next contraction.
template <class O>
__device__ __forceinline__ typename O::V8 join_pack(f32x4 lo, f32x4 hi) {
    using E = typename O::E;
    return typename O::V8{E(lo[0]), E(lo[1]), E(lo[2]), E(lo[3]),
                          E(hi[0]), E(hi[1]), E(hi[2]), E(hi[3])};
}

// Neighbouring r stored at once: a power of two up to `most`, dividing the `held` r a thread holds
// together, the workgroup's SC and the output mode (so that a run never crosses them).
constexpr int join_runs(int held, int sc, int oR, int most) {
    int run = 1;
    while (2 * run <= most && held % (2 * run) == 0 && sc % (2 * run) == 0 && oR % (2 * run) == 0) run *= 2;
    return run;
}

// Whether RUN neighbouring elements of y (and aux) may be accessed at once from a multiple of RUN.
template <int DT, bool EPI, int RUN>
__device__ __forceinline__ bool join_aligned(const void *y, int mode, const void *aux) {
    constexpr unsigned e = sizeof(typename Elem<DT>::T);
    const unsigned ye = EPI && (mode & kEpiKindMask) == TRK_EPI_F32 ? 4 : e;
    const unsigned ae = mode & kAuxF32 ? 4 : e;
    return !(reinterpret_cast<uintptr_t>(y) & (RUN * ye - 1)) &&
           !(EPI && aux && reinterpret_cast<uintptr_t>(aux) & (RUN * ae - 1));
}

// Elements o .. o + RUN - 1 of y through the epilogue. All of aux's are read, into a, before y's are
// written (they may be one buffer).
template <int DT, bool EPI, int RUN>
__device__ __forceinline__ void join_store(void *y, int mode, const void *aux, size_t o,
                                           const float *v, float *a, bool runs) {
    using T = typename Elem<DT>::T;
    using TV = T __attribute__((ext_vector_type(RUN)));
    using FV = float __attribute__((ext_vector_type(RUN)));
    const int kind = EPI ? mode & kEpiKindMask : TRK_EPI_STORE;
    if constexpr (EPI) {
        if (RUN > 1 && runs && (kind == TRK_EPI_ADD || kind == TRK_EPI_SILU_MUL)) {
            if (mode & kAuxF32) {
                const FV f = *reinterpret_cast<const FV *>(static_cast<const float *>(aux) + o);
#pragma unroll
                for (int n = 0; n < RUN; ++n) a[n] = f[n];
            } else {
                const TV f = *reinterpret_cast<const TV *>(static_cast<const T *>(aux) + o);
#pragma unroll
                for (int n = 0; n < RUN; ++n) a[n] = Elem<DT>::to_f32(f[n]);
            }
        } else {
#pragma unroll
            for (int n = 0; n < RUN; ++n) a[n] = epi_aux<DT>(aux, mode, o + n);
        }
    }
    if (RUN > 1 && runs) {
        if (EPI && kind == TRK_EPI_F32) {
            FV f;
#pragma unroll
            for (int n = 0; n < RUN; ++n) f[n] = v[n];
            *reinterpret_cast<FV *>(static_cast<float *>(y) + o) = f;
            return;
        }
        TV f;
#pragma unroll
        for (int n = 0; n < RUN; ++n) {
            float w = v[n];
            if constexpr (EPI) {
                if (kind == TRK_EPI_ADD) w = a[n] + v[n];
                if (kind == TRK_EPI_SILU_MUL) w = silu_f32(a[n]) * v[n];
            }
            f[n] = Elem<DT>::from_f32(w);
        }
        *reinterpret_cast<TV *>(static_cast<T *>(y) + o) = f;
        return;
    }
#pragma unroll
    for (int n = 0; n < RUN; ++n) {
        if constexpr (EPI)
            epi_put<DT>(y, mode, o + n, v[n], a[n]);
        else
            static_cast<T *>(y)[o + n] = Elem<DT>::from_f32(v[n]);
    }
}

// A 32-wide K step in its parts, so that independent chains can alternate between them: one MFMA
// in 16 bits; in 32 bits 8 of K 4 (Ops<F32>::k32 runs them back to back on one accumulator).
template <class O>
struct JoinMfma {
    static constexpr int N = 1;
    __device__ static Acc<32> part(typename O::V8 a, typename O::V8 b, Acc<32> c, int) {
        return O::k32(a, b, c);
    }
};
template <>
struct JoinMfma<Ops<TRK_DTYPE_F32>> {
    using O = Ops<TRK_DTYPE_F32>;
    static constexpr int N = 8;
    __device__ static Acc<32> part(O::V8 a, O::V8 b, Acc<32> c, int e) {
        return {__builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c.v, 0, 0, 0)};
    }
};

// Scheduling pattern of N instructions of class MASK, each followed by EACH MFMAs.
template <int MASK, int N, int EACH>
__device__ __forceinline__ void join_interleave() {
    if constexpr (N > 0) {
        __builtin_amdgcn_sched_group_barrier(MASK, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, EACH, 0);
        join_interleave<MASK, N - 1, EACH>();
    }
}

template <KCfg C, bool EPI, bool PAIR>
__device__ __forceinline__ void join_unit(const typename Ops<C.dt>::E *__restrict__ x,
                                          const typename Ops<C.dt>::E *__restrict__ packed0,
                                          const typename Ops<C.dt>::E *__restrict__ packed1,
                                          void *y, int T, int epi_mode, const void *aux, int unit,
                                          int tile_y, unsigned char *lds) {
    using G = JoinGeo<C>;
    using O = Ops<C.dt>;
    using E = typename O::E;
    using V8 = typename O::V8;
    constexpr int R = G::R;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lrow = lane & 15, lgrp = lane >> 4;
    const int kw = wave % G::KW, qw = wave / G::KW;
    constexpr int NRC = cdiv(G::oR, G::SC);
    const int q0 = unit / NRC * G::FC, r0 = unit % NRC * G::SC;
    const int t0 = tile_y * G::TT;
    // (the wave's pairs: nq -> pr = qw * NQ + nq -> (q0 + pr / SC, r0 + pr % SC))

    // x goes to LDS as [row][lane group][4 features of result 0, 4 of result 1], the eight K
    // positions of a lane group together, a region per chunk. All waves load it together, whole
    // cache lines at a time: with lanes in fragment order each lane touches a line of its own, and
    // with a wave loading its own chunk two waves fetch each line, half of it used (measured at
    // 14336 -> 4096 R16 T=256: x then took a third of the time). In 16 bits a lane's 16 bytes are
    // the features of two lane groups of one result; in 32 bits, of one. The lane groups of row w
    // sit at slots g ^ x_swap(w), so that the 32 lanes one LDS pass serves read 32 different
    // 16-byte units, and with shared x (a store's 16 lanes are then four rows, each writing the even or
    // the odd slots) so that rows two apart write different ones.
    // Byte offsets from the tile's first row (rows past the tile or the last token read the last one;
    // their results are not stored).
    auto x_swap = [](int row) { return row / 8 % 2 * 2 + (G::XS && G::EB == 2 ? row / 2 % 2 : 0); };
    const char *xt = reinterpret_cast<const char *>(x + size_t(t0) * G::IN);
    const int xc = lane % G::LPR, xw = wave * G::RPI + lane / G::LPR;  // 16 bytes of a row, row
    unsigned xoff[G::XN];
#pragma unroll
    for (int m = 0; m < G::XN; ++m)
        xoff[m] = unsigned(min(min(m * G::NW * G::RPI + xw, G::TT - 1), T - 1 - t0)) * G::IN * G::EB +
                  16 * xc;
    // The digits of i are walked from a start that differs between neighbouring units: x rows
    // a multiple of 4 KB apart keep one digit's features in one L2 channel, which every
    // workgroup of an XCD would otherwise read at once.
    const unsigned i0 = unsigned(unit) % G::nI;
    auto digit = [&](int st) { return int((i0 + unsigned(st)) % G::nI); };
    E *j2s = reinterpret_cast<E *>(lds), *j3s = j2s + G::lJ3, *zeros = j2s + G::lZ;
    E *g1s = j2s + G::lG1;
    // fragment reads: one address register per region, everything else in the instruction's
    // offset field (the regions start past its 64 KB)
    int lane_g1 = G::lG1 + lane * G::VPE;
    int lane_x = G::lX + G::x_at(kw) + (lrow * 4 + (lgrp ^ x_swap(lrow))) * G::VPE;
    int put_x[G::XPER];
#pragma unroll
    for (int m = 0; m < G::XPER; ++m) {
        const int row = m * G::NW * G::RPI + xw, w = row % 16;
        // (16 bits: groups 2 (s % 2) and the next, result s / 2, which x_swap leaves neighbours)
        constexpr int SPC = G::LPR / G::KW;  // lanes of a row per chunk
        const int sl = xc % SPC;
        put_x[m] = G::lX + G::x_at(xc / SPC) + row / 16 * G::FRAG + w * 4 * G::VPE +
                   (G::EB == 2 ? ((2 * (sl % 2)) ^ x_swap(w)) * 8 + sl / 2 * 4
                               : sl / 4 * 256 + (sl % 4 ^ x_swap(w)) * 4);
        asm("" : "+v"(put_x[m]));
    }
    // (shared x: where a row's odd lane groups go, on the side of the even ones that x_swap says)
    int put_x2 = put_x[0] + (x_swap(xw % 16) % 2 ? -8 : 8);
    asm("" : "+v"(lane_g1), "+v"(lane_x), "+v"(put_x2));

    f32x4 gate[PAIR ? G::TPW : 1];
#pragma unroll 1
    for (int pass = 0; pass < (PAIR ? 2 : 1); ++pass) {
        const E *pk = PAIR && pass ? packed1 : packed0;
        const float scale = *reinterpret_cast<const float *>(pk);
        f32x4 acc[G::NQ][G::MT];
#pragma unroll
        for (int n = 0; n < G::NQ; ++n)
#pragma unroll
            for (int m = 0; m < G::MT; ++m) acc[n][m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

        // one step's G1 fragments: global -> registers -> LDS
        u32x4 gr[2][G::GPT];
        auto load_g1 = [&](int st, int set) TRK_INLINE {
            const u32x4 *src = reinterpret_cast<const u32x4 *>(pk + G::oJ1 + digit(st) * G::szG1);
#pragma unroll
            for (int v = 0; v < G::GPT; ++v) {
                const int i = tid + v * G::NT;
                if (G::szG1 / G::VPE % G::NT == 0 || i < G::szG1 / G::VPE) gr[set][v] = src[i];
            }
        };
        auto store_g1 = [&](int buf) TRK_INLINE {
            u32x4 *dst = reinterpret_cast<u32x4 *>(g1s + buf * G::szG1);
#pragma unroll
            for (int v = 0; v < G::GPT; ++v) {
                const int i = tid + v * G::NT;
                if (G::szG1 / G::VPE % G::NT == 0 || i < G::szG1 / G::VPE) dst[i] = gr[buf][v];
            }
        };
        // x of a step, global -> registers -> LDS: the features of the waves' chunks at digit i
        // (features past the last are zero, and so are whole chunks past the last)
        u32x4 xr[2][G::XN];
        auto chunk_of = [&](int st) { return int(unsigned(st) / G::nI) * G::KW; };
        auto absent = [&](int st) {
            return G::PAD && chunk_of(st) * 32 + xc * (16 / G::EB) >= G::NJK;
        };
        auto load_x = [&](int st, int set) TRK_INLINE {
            const char *base = xt + (digit(st) * G::NJK + chunk_of(st) * 32) * G::EB;
#pragma unroll
            for (int m = 0; m < G::XN; ++m)
                xr[set][m] = *reinterpret_cast<const u32x4 *>(base + xoff[m] - (absent(st) ? 16 * xc : 0));
        };
        auto store_x = [&](int st, int set, int buf) TRK_INLINE {  // step st's, which load_x read
#pragma unroll
            for (int m = 0; m < G::XN; ++m) {
                E *dst = j2s + put_x[m % G::XPER] + buf * G::szX +
                         m / G::XPER * (G::NW * G::RPI * G::XPER / 16) * G::FRAG;
                const u32x4 v = absent(st) ? u32x4{0, 0, 0, 0} : xr[set][m];
                if constexpr (G::EB == 2) {
                    *reinterpret_cast<u32x2 *>(dst) = u32x2{v[0], v[1]};
                    E *dst2 = G::XS ? j2s + put_x2 + buf * G::szX + m * (G::NW * G::RPI / 16) * G::FRAG
                                    : dst + 8;
                    *reinterpret_cast<u32x2 *>(dst2) = u32x2{v[2], v[3]};
                } else {
                    *reinterpret_cast<u32x4 *>(dst) = v;
                }
            }
        };

        // prologue: the slices of G2 and G3, and the first steps' G1 and x, all in flight before
        // the first is stored
        if (PAIR && pass) __syncthreads();  // the first pass is done with the LDS
        constexpr int N2 = G::szJ2 / G::VPE, N3 = G::SC * G::nK * G::R2 / G::VPE;
        u32x4 v2[cdiv(N2, G::NT)], v3[cdiv(N3, G::NT)];
#pragma unroll
        for (int k = 0; k < cdiv(N2, G::NT); ++k) {
            constexpr int PER = G::nJ * G::R2 / G::VPE;
            const int v = min(tid + k * G::NT, N2 - 1), q = min(q0 + v / PER, G::oQ - 1);
            v2[k] = reinterpret_cast<const u32x4 *>(pk + G::oJ2 + q * G::nJ * G::R2)[v % PER];
        }
#pragma unroll
        for (int k = 0; k < cdiv(N3, G::NT); ++k) {
            constexpr int PER = G::nK * G::R2 / G::VPE;
            const int v = min(tid + k * G::NT, N3 - 1), r = min(r0 + v / PER, G::oR - 1);
            v3[k] = reinterpret_cast<const u32x4 *>(pk + G::oJ3 + r * G::nK * G::R2)[v % PER];
        }
        load_g1(0, 0);
        load_g1(1, 1);
        load_x(0, 0);
        load_x(min(1, G::NST - 1), 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < cdiv(N2, G::NT); ++k)
            reinterpret_cast<u32x4 *>(j2s)[min(tid + k * G::NT, N2 - 1)] = v2[k];
#pragma unroll
        for (int k = 0; k < cdiv(N3, G::NT); ++k) {
            constexpr int ROW = G::R2 / G::VPE;
            const int v = min(tid + k * G::NT, N3 - 1);
            reinterpret_cast<u32x4 *>(j3s)[v / ROW * (G::P3K / G::VPE) + v % ROW] = v3[k];
        }
        if (tid < G::R2 / G::VPE) reinterpret_cast<u32x4 *>(zeros)[tid] = u32x4{0, 0, 0, 0};
        store_g1(0);
        store_g1(1);
        store_x(0, 0, 0);
        load_g1(2, 0);
        load_g1(3, 1);
        load_x(min(2, G::NST - 1), 0);
        __syncthreads();
        V8 gf[G::KS], h[G::NQ][2][G::KS];
#pragma unroll
        for (int s = 0; s < G::KS; ++s) gf[s] = join_read<O>(j2s + lane_g1 + s * G::FRAG);
        __syncthreads();  // step 0 rewrites that buffer

        // H: the joined slice of a chunk's 32 features, as the formation's operands
        auto join = [&](int ch) TRK_INLINE {
            // Operands: A rows b (rank 8: (a', b), block diagonal in a'), B columns the features; K
            // = c, or (j of two, c). Lane groups hold 4 (SJ) or 8 of K.
            using A = std::conditional_t<G::SJ, typename O::V4, V8>;
            constexpr int KL = G::SJ ? 4 : 8;
            const int jl = G::SJ ? 0 : R == 8 ? lgrp & 1 : lgrp >> 1;  // this group's j of the two
            const int cl = G::SJ ? KL * lgrp % R : R == 8 ? 0 : 8 * (lgrp & 1);  // its first c
            const int al = R == 8 ? lgrp >> 1 : 0;                  // rank 8: its a of the two
            constexpr int AD = R == 8 ? 2 : 1;              // a's per result
            constexpr int NB = 2 * G::KS < 8 ? 2 * G::KS : 8;  // results of a pair per block
            constexpr int NBK = 2 * G::KS / NB;             // blocks per ft
            const int rw = qw * G::NQ % G::SC;
            A a2[2][G::NQ][G::NH];
            const E *b3[2];
            int jn[2], jb[2];
#pragma unroll
            for (int ft = 0; ft < 2; ++ft) {
                jb[ft] = (ch * 32 + 16 * ft) / G::nK;
#pragma unroll
                for (int n = 0; n < G::NQ; ++n)
#pragma unroll
                    for (int m = 0; m < G::NH; ++m) {
                        const int fq = (qw * G::NQ + n) / G::SC;
                        const int j = min(jb[ft] + m * 2 + jl, G::nJ - 1);
                        a2[ft][n][m] = join_load<A>(j2s + ((fq * G::nJ + j) * R + lrow % R) * R + cl);
                        if (R == 8 && lrow / 8 != al) a2[ft][n][m] = A{};
                    }
                // this lane's feature: its j, its k. Columns past the last feature, and with one MFMA
                // per result the lanes of the other j, read zeros.
                const int f = ch * 32 + 16 * ft + lrow;
                jn[ft] = f / G::nK;
                b3[ft] = j3s + (rw * G::nK + f % G::nK) * G::P3K + al * R + cl;
                if ((G::PAD && f >= G::NJK) ||
                    (!G::SJ && G::NH == 1 && jn[ft] != jb[ft] + jl))
                    b3[ft] = nullptr;
            }
            // block k of 2 NBK: its operands are read while block k - 1's MFMAs run
            A b[2][G::NRW][NB];
            auto read_b = [&](int k) TRK_INLINE {
#pragma unroll
                for (int n = 0; n < G::NRW; ++n)
#pragma unroll
                    for (int v = 0; v < NB; ++v) {
                        const int o = (k % NBK * NB + v) * AD * R;
                        const E *p = b3[k / NBK];
                        b[k & 1][n][v] = join_load<A>((p ? p + n * (G::nK * G::P3K) : zeros) + o);
                    }
            };
            read_b(0);
#pragma unroll
            for (int k = 0; k < 2 * NBK; ++k) {
                const int ft = k / NBK;
                if (k + 1 < 2 * NBK) read_b(k + 1);
                __builtin_amdgcn_sched_barrier(0);
                f32x4 d[G::NQ][NB];
#pragma unroll
                for (int m = 0; m < G::NH; ++m)
#pragma unroll
                    for (int v = 0; v < NB; ++v)
#pragma unroll
                        for (int n = 0; n < G::NQ; ++n) {
                            A bm = b[k & 1][n % G::NRW][v];
                            if (G::NH > 1 && jn[ft] != jb[ft] + m * 2 + jl) bm = A{};
                            const f32x4 t = m ? d[n][v] : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                            if constexpr (G::SJ)
                                d[n][v] = O::k16(a2[ft][n][m], bm, Acc<16>{t}).v;
                            else
                                d[n][v] = O::k32(a2[ft][n][m], bm, Acc<32>{t}).v;
                        }
#pragma unroll
                for (int n = 0; n < G::NQ; ++n)
#pragma unroll
                    for (int v = 0; v < NB; v += 2)
                        h[n][ft][(k % NBK * NB + v) / 2] = join_pack<O>(d[n][v], d[n][v + 1]);
            }
        };
        // Step st (of parity P): the weight tiles of (chunk, digit) and their products with x.
        // G1's fragments arrived in registers during step st - 1; this step reads those of
        // st + 1 from LDS, writes those of st + 2 there (the buffer every wave has read by the
        // last barrier) and starts the loads of st + 4's, two steps before their store; x goes
        // the same way, st + 1's to LDS and st + 3's from memory. The scheduling barriers keep every read a block of MFMAs ahead of
        // its use: with one or two waves a SIMD nothing else covers its latency.
        auto step = [&](auto parity, int st) TRK_INLINE {
            constexpr int P = decltype(parity)::value;
            V8 xl[G::MT];
#pragma unroll
            for (int m = 0; m < G::MT; ++m)
                xl[m] = join_read<O>(j2s + lane_x + P * G::szX + m * G::FRAG);
            Acc<32> w[G::NQ][2];
#pragma unroll
            for (int n = 0; n < G::NQ; ++n)
#pragma unroll
                for (int ft = 0; ft < 2; ++ft) w[n][ft].v = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < G::KS; ++s)
#pragma unroll
                for (int e = 0; e < JoinMfma<O>::N; ++e)
#pragma unroll
                    for (int n = 0; n < G::NQ; ++n)
#pragma unroll
                        for (int ft = 0; ft < 2; ++ft)
                            w[n][ft] = JoinMfma<O>::part(h[n][ft][s], gf[s], w[n][ft], e);
            store_g1(P);
            load_g1(st + 4, P);
            store_x(min(st + 1, G::NST - 1), 1 - P, 1 - P);
            load_x(min(st + 3, G::NST - 1), 1 - P);
            // one memory operation per few of the formation's MFMAs: x's reads, then the stores,
            // then the loads (in a block of their own they held the MFMAs up: their issue alone
            // took a sixth of a step)
            constexpr int RD = G::MT * G::EB / 2, WR = G::GPT + G::XN, LD = G::GPT + G::XN;
            constexpr int MF = 2 * G::NQ * G::KS * (G::EB == 2 ? 1 : 8);
            constexpr int EACH = MF / (RD + WR + LD) > 0 ? MF / (RD + WR + LD) : 1;
            join_interleave<0x100, RD, EACH>();
            join_interleave<0x200, WR, EACH>();
            join_interleave<0x020, LD, EACH>();
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < G::KS; ++s)
                gf[s] = join_read<O>(j2s + lane_g1 + (1 - P) * G::szG1 + s * G::FRAG);
            V8 wb[G::NQ];
#pragma unroll
            for (int n = 0; n < G::NQ; ++n) wb[n] = join_pack<O>(w[n][0].v, w[n][1].v);
            // (in groups of 4 tiles: 32-bit x in flight takes twice the registers)
            constexpr int MG = JoinMfma<O>::N == 1 ? G::MT : 4;
#pragma unroll
            for (int m0 = 0; m0 < G::MT; m0 += MG)
#pragma unroll
                for (int e = 0; e < JoinMfma<O>::N; ++e)
#pragma unroll
                    for (int m = m0; m < m0 + MG && m < G::MT; ++m)
#pragma unroll
                        for (int n = 0; n < G::NQ; ++n)
                            acc[n][m] = JoinMfma<O>::part(xl[m], wb[n], Acc<32>{acc[n][m]}, e).v;
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
        };
#pragma unroll 1
        for (int rd = 0; rd < G::NR; ++rd) {
            join(rd * G::KW + kw);
#pragma unroll 1
            for (int ii = 0; ii < G::nI; ii += 2) {
                step(std::integral_constant<int, 0>{}, rd * G::nI + ii);
                step(std::integral_constant<int, 1>{}, rd * G::nI + ii + 1);
            }
        }
        // the KW waves' partial sums meet in LDS; each wave adds and keeps its share of the
        // tiles (tile = mt * NQ + nq), in wave order
        f32x4 out[G::TPW];
        if constexpr (G::KW > 1) {
            f32x4 *red = reinterpret_cast<f32x4 *>(lds);
#pragma unroll
            for (int n = 0; n < G::NQ; ++n)
#pragma unroll
                for (int m = 0; m < G::MT; ++m)
                    red[(wave * G::TILES + m * G::NQ + n) * 64 + lane] = acc[n][m];
            __syncthreads();
#pragma unroll
            for (int t = 0; t < G::TPW; ++t) {
                const int tile = kw * G::TPW + t;
                out[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                if (G::TILES % G::KW == 0 || tile < G::TILES)
#pragma unroll
                    for (int w = 0; w < G::KW; ++w)
                        out[t] += red[((qw * G::KW + w) * G::TILES + tile) * 64 + lane];
            }
        } else {
#pragma unroll
            for (int t = 0; t < G::TPW; ++t) out[t] = acc[t % G::NQ][t / G::NQ];
        }
#pragma unroll
        for (int t = 0; t < G::TPW; ++t) out[t] *= scale;
        if (PAIR && pass == 0) {
#pragma unroll
            for (int t = 0; t < G::TPW; ++t) gate[t] = out[t];
            continue;
        }
        if constexpr (PAIR)
#pragma unroll
            for (int t = 0; t < G::TPW; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) out[t][e] = silu_f32(gate[t][e]) * out[t][e];
        // y[t][p][q][r], RUN neighbouring r in one store where y and aux are aligned for it (every
        // store is a transaction of its own: a lane's neighbours hold other p, far apart in y)
        constexpr int kRuns = join_runs(G::XS ? G::SC : G::NQ, G::SC, G::oR, 16 / G::EB);
        if constexpr (G::XS) {
            // the waves' pairs meet in LDS, YG token tiles at a time: a thread then stores all r of
            // a (token, p) (measured at 5120 -> 12288 R16 T=128: 2-byte stores took 11 of 71 us)
            constexpr int RUN = kRuns;
            const bool runs = RUN > 1 && join_aligned<C.dt, EPI, RUN>(y, epi_mode, PAIR ? nullptr : aux);
            float *ys = reinterpret_cast<float *>(lds);
#pragma unroll
            for (int m0 = 0; m0 < G::MT; m0 += G::YG) {
                if (m0) __syncthreads();
#pragma unroll
                for (int m = m0; m < m0 + G::YG && m < G::MT; ++m)
#pragma unroll
                    for (int n = 0; n < G::NQ; ++n)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            ys[((m - m0) * 16 + 4 * lgrp + e) * G::YP + (qw * G::NQ + n) * 16 + lrow] =
                                out[m * G::NQ + n][e];
                __syncthreads();
                constexpr int ITEMS = G::YG * 256;
#pragma unroll 1
                for (int i = tid; i < ITEMS; i += G::NT) {
                    const int p = i % 16, tl = i / 16, tok = t0 + m0 * 16 + tl;
                    if (p >= G::oP || tok >= T || m0 * 16 + tl >= G::TT) continue;
#pragma unroll
                    for (int k = 0; k < G::FC * G::SC; k += RUN) {
                        const int q = q0 + k / G::SC, r = r0 + k % G::SC;
                        if (q >= G::oQ || r >= G::oR) continue;
                        float v[RUN], a[RUN];
#pragma unroll
                        for (int n = 0; n < RUN; ++n) v[n] = ys[tl * G::YP + (k + n) * 16 + p];
                        join_store<C.dt, EPI && !PAIR, RUN>(
                            y, epi_mode, aux, size_t(tok) * G::OUT + (p * G::oQ + q) * G::oR + r, v, a, runs);
                    }
                }
            }
        } else {
            constexpr int RUN = G::TPW % kRuns == 0 && G::TILES % G::KW == 0 ? kRuns : 1;
            const bool runs = RUN > 1 && join_aligned<C.dt, EPI, RUN>(y, epi_mode, PAIR ? nullptr : aux);
#pragma unroll
            for (int t = 0; t < G::TPW; t += RUN) {
                const int tile = kw * G::TPW + t;
                if (G::TILES % G::KW != 0 && tile >= G::TILES) break;
                const int mt = tile / G::NQ, pr = qw * G::NQ + tile % G::NQ;
                const int q = q0 + pr / G::SC, r = r0 + pr % G::SC;
                if (lrow >= G::oP || q >= G::oQ || r >= G::oR) continue;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int tok = t0 + mt * 16 + 4 * lgrp + e;
                    if (tok >= T) continue;
                    float v[RUN], a[RUN];
#pragma unroll
                    for (int n = 0; n < RUN; ++n) v[n] = out[t + n][e];
                    join_store<C.dt, EPI && !PAIR, RUN>(
                        y, epi_mode, aux, size_t(tok) * G::OUT + (lrow * G::oQ + q) * G::oR + r, v, a, runs);
                }
            }
        }
    }
}

// Workgroup -> (unit, token tile), over the whole launch: each XCD takes one contiguous range,
// so neighbouring output pairs, which share lines of y, are written through one L2.
template <KCfg C>
__device__ __forceinline__ int2 join_unit_of(int bx, int by) {
    constexpr int NBLK = JoinGeo<C>::NBLK;
    const int n = NBLK * int(gridDim.y), lin = by * NBLK + bx;
    const int xcd = lin % 8, base = n / 8, rem = n % 8;
    const int g = xcd * base + (xcd < rem ? xcd : rem) + lin / 8;
    return {g % NBLK, g / NBLK};
}

template <KCfg C, bool EPI>
__global__ void __launch_bounds__(JoinGeo<C>::NT, JoinGeo<C>::WPC * JoinGeo<C>::NW / 4)
    ring3_join_kernel(const typename Ops<C.dt>::E *__restrict__ x,
                      const typename Ops<C.dt>::E *__restrict__ packed, void *y, int T,
                      int epi_mode, const void *aux) {  // aux may equal y
    __shared__ __attribute__((aligned(16))) unsigned char lds[JoinGeo<C>::LDS_BYTES];
    const int2 u = join_unit_of<C>(blockIdx.x, blockIdx.y);
    join_unit<C, EPI, false>(x, packed, nullptr, y, T, epi_mode, aux, u.x, u.y, lds);
}

template <KCfg C>
__global__ void __launch_bounds__(JoinGeo<C>::NT, JoinGeo<C>::WPC * JoinGeo<C>::NW / 4)
    ring3_join_pair_kernel(const typename Ops<C.dt>::E *__restrict__ x,
                           const typename Ops<C.dt>::E *__restrict__ packed_g,
                           const typename Ops<C.dt>::E *__restrict__ packed_u, void *y, int T) {
    __shared__ __attribute__((aligned(16))) unsigned char lds[JoinGeo<C>::LDS_BYTES];
    const int2 u = join_unit_of<C>(blockIdx.x, blockIdx.y);
    join_unit<C, true, true>(x, packed_g, packed_u, y, T, TRK_EPI_SILU_MUL, nullptr, u.x, u.y, lds);
}

template <KCfg C>
int launch_join(const Plan &plan, const Variant &v, const void *packed, const void *x, void *y,
                int tokens, Epi epi, hipStream_t stream) {
    using G = JoinGeo<C>;
    using E = typename Ops<C.dt>::E;
    const E *pk = reinterpret_cast<const E *>(static_cast<const char *>(packed) +
                                              plan.chains[v.chain].offF);
    constexpr int per_launch = 65535 * G::TT;  // the grid's y limit, as launch_mfma
    const size_t y_elem = (epi.mode & kEpiKindMask) == TRK_EPI_F32 ? 4 : sizeof(E);
    const size_t aux_elem = (epi.mode & kAuxF32) ? 4 : sizeof(E);
    for (int t0 = 0; t0 < tokens; t0 += per_launch) {
        int n = tokens - t0 < per_launch ? tokens - t0 : per_launch;
        const E *xe = static_cast<const E *>(x) + size_t(t0) * G::IN;
        void *yc = static_cast<char *>(y) + size_t(t0) * G::OUT * y_elem;
        const void *ac =
            epi.aux ? static_cast<const char *>(epi.aux) + size_t(t0) * G::OUT * aux_elem : nullptr;
        int mode = epi.mode;
        void *args[] = {&xe, &pk, &yc, &n, &mode, &ac};
        const void *fn = epi.mode == TRK_EPI_STORE
                             ? reinterpret_cast<const void *>(&ring3_join_kernel<C, false>)
                             : reinterpret_cast<const void *>(&ring3_join_kernel<C, true>);
        const int st = check_hip(hipLaunchKernel(fn, dim3(G::NBLK, (n + G::TT - 1) / G::TT),
                                                 dim3(G::NT), args, 0, stream),
                                 "trk_forward: joined kernel launch");
        if (st != TRK_OK) return st;
    }
    return TRK_OK;
}

template <KCfg C>
int launch_join_pair(const Plan &plan, const Variant &v, const void *packed_g,
                     const void *packed_u, const void *x, void *y, int tokens,
                     hipStream_t stream) {
    using G = JoinGeo<C>;
    using E = typename Ops<C.dt>::E;
    const size_t off = plan.chains[v.chain].offF;
    const E *pg = reinterpret_cast<const E *>(static_cast<const char *>(packed_g) + off);
    const E *pu = reinterpret_cast<const E *>(static_cast<const char *>(packed_u) + off);
    constexpr int per_launch = 65535 * G::TT;
    for (int t0 = 0; t0 < tokens; t0 += per_launch) {
        int n = tokens - t0 < per_launch ? tokens - t0 : per_launch;
        const E *xe = static_cast<const E *>(x) + size_t(t0) * G::IN;
        void *yc = static_cast<void *>(static_cast<E *>(y) + size_t(t0) * G::OUT);
        void *args[] = {&xe, &pg, &pu, &yc, &n};
        const int st = check_hip(hipLaunchKernel(reinterpret_cast<const void *>(&ring3_join_pair_kernel<C>),
                                                 dim3(G::NBLK, (n + G::TT - 1) / G::TT), dim3(G::NT),
                                                 args, 0, stream),
                                 "trk_forward_swiglu: joined kernel launch");
        if (st != TRK_OK) return st;
    }
    return TRK_OK;
}

#define TRK_ENTRY_JOIN(CFG, TMIN, TMAX) \
    {CFG, TMIN, TMAX, JoinGeo<CFG>::LDS_BYTES, launch_join<CFG>, nullptr},
#define TRK_ENTRY_JOIN_PAIR(CFG, TMIN, TMAX) \
    {CFG, TMIN, TMAX, JoinGeo<CFG>::LDS_BYTES, launch_join<CFG>, launch_join_pair<CFG>},

}  // namespace
}  // namespace trk
