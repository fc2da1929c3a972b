// Packing of the three cores into the per-chain sections of the packed buffer.
//
// Replaces pack_cores (src/factorized_inference/tr_kernel.py:86-99): same idea (the same
// values re-laid out for the kernels, zero padding only, no expansion and no dense W), own
// layouts. For each chain (contraction order F, S, L) of the plan:
//   Fk[f][r1][r2][KF]  = Fc[r1][f][iF][r2]   for iF < nF, else 0
//   Sk[s][r3][K2]      = Sc[r2][s][iS][r3]   at k = (r2/sg)*sg*nS + iS*sg + r2%sg < nS*R,
//                                            else 0
//   Lk[iL][l][K]       = Lc[r3][l][iL][r1]   at K = (r3/lg)*lg*R + r1*lg + r3%lg
// (sg = lg = R: the natural orders k = iS*R + r2, K = r1*R + r3). A chain with sfrag stores
// Sk in the order the register-resident 32x32x16 A fragments are loaded: for each tile of 32
// rows (s, r3) and each step of 16 k, the 64 lanes' 8-element pieces one after another
// (lane = 32 * (k % 16 / 8) + row % 32), rows past oS*R zero. Only the sections a chain owns
// are written; the others are shared with an earlier chain of the same order.
// where a chain core Xc[in][o][i][out] is the core G[in][o][i][out] of a forward order and
// G[out][o][i][in] of a backward one. Bits are copied, so the dtype does not matter beyond
// its width.
#include <algorithm>

#include "trk_internal.h"
#include "trk_types.h"

namespace trk {
namespace {

// index of G[alpha][o][i][beta] in a core of shape [R][O][I][R]
__device__ inline size_t core_index(int alpha, int o, int i, int beta, int O, int I, int R) {
    return ((size_t(alpha) * O + o) * I + i) * R + beta;
}

struct PackArgs {
    int R, Rc, forward;  // kernel rank; rank of the cores read (ring indices >= Rc pack zero)
    int nF, nS, nL, oF, oS, oL, KF, K2, sg, lg, sfrag;
    size_t nFk, nSk, nLk;  // element counts of the three sections
};

// N: 32 bits where the chain's sections have fewer than 2^31 elements (the index arithmetic is a
// chain of divisions, several times as long in 64 bits)
template <typename W, typename N>
__global__ void __launch_bounds__(256) pack_chain_kernel(const W *__restrict__ gF,
                                                         const W *__restrict__ gS,
                                                         const W *__restrict__ gL,
                                                         W *__restrict__ Fk, W *__restrict__ Sk,
                                                         W *__restrict__ Lk, PackArgs a) {
    const N nFk = N(a.nFk), nSk = N(a.nSk), total = N(a.nFk + a.nSk + a.nLk);
    const int R = a.R;
    for (N d = blockIdx.x * N(blockDim.x) + threadIdx.x; d < total; d += N(gridDim.x) * blockDim.x) {
        if (d < nFk) {
            const int iF = int(d % a.KF);
            N rest = d / a.KF;
            const int r2 = int(rest % R);
            rest /= R;
            const int r1 = int(rest % R);
            const int f = int(rest / R);
            W v = W(0);
            if (iF < a.nF && r1 < a.Rc && r2 < a.Rc)
                v = gF[a.forward ? core_index(r1, f, iF, r2, a.oF, a.nF, a.Rc)
                                 : core_index(r2, f, iF, r1, a.oF, a.nF, a.Rc)];
            Fk[d] = v;
        } else if (d < nFk + nSk) {
            const N e = d - nFk;
            int k, row;
            if (a.sfrag) {  // [tile][k / 16][lane][8]
                const int lane = int(e / 8 % 64), ks = a.K2 / 16;
                const N rest = e / 512;
                k = int(rest % ks) * 16 + lane / 32 * 8 + int(e % 8);
                row = int(rest / ks) * 32 + lane % 32;
            } else {
                k = int(e % a.K2);
                row = int(e / a.K2);
            }
            const int r3 = row % R, s = row / R;
            W v = W(0);
            if (k < a.nS * R && s < a.oS) {
                const int span = a.sg * a.nS, rem = k % span;
                const int iS = rem / a.sg, r2 = k / span * a.sg + rem % a.sg;
                if (r2 < a.Rc && r3 < a.Rc)
                    v = gS[a.forward ? core_index(r2, s, iS, r3, a.oS, a.nS, a.Rc)
                                     : core_index(r3, s, iS, r2, a.oS, a.nS, a.Rc)];
            }
            Sk[e] = v;
        } else {
            const N e = d - nFk - nSk;
            const int kk = int(e % N(R * R)), span = a.lg * R, rem = kk % span;
            const int r1 = rem / a.lg, r3 = kk / span * a.lg + rem % a.lg;
            N rest = e / N(R * R);
            const int l = int(rest % a.oL);
            const int iL = int(rest / a.oL);
            W v = W(0);
            if (r1 < a.Rc && r3 < a.Rc)
                v = gL[a.forward ? core_index(r3, l, iL, r1, a.oL, a.nL, a.Rc)
                                 : core_index(r1, l, iL, r3, a.oL, a.nL, a.Rc)];
            Lk[e] = v;
        }
    }
}

template <typename W>
int pack_all(const Plan &plan, const void *const g[3], void *packed, hipStream_t stream) {
    char *base = static_cast<char *>(packed);
    for (int ci = 0; ci < plan.nchains; ++ci) {
        const Chain &c = plan.chains[ci];
        if (c.join) continue;
        PackArgs a;
        a.R = c.R;
        a.Rc = plan.core_rank;
        a.forward = c.forward;
        a.nF = c.nF;
        a.nS = c.nS;
        a.nL = c.nL;
        a.oF = c.oF;
        a.oS = c.oS;
        a.oL = c.oL;
        a.KF = c.KF;
        a.K2 = c.K2;
        a.sg = c.sg;
        a.lg = c.lg;
        a.sfrag = c.sfrag;
        a.nFk = c.ownF ? size_t(c.oF) * c.R * c.R * c.KF : 0;
        a.nSk = c.ownS ? size_t(c.sfrag ? (c.oS * c.R + 31) / 32 * 32 : c.oS * c.R) * c.K2 : 0;
        a.nLk = c.ownL ? size_t(c.nL) * c.oL * c.R * c.R : 0;
        const size_t total = a.nFk + a.nSk + a.nLk;
        if (total == 0) continue;
        const int blocks = int(std::min<size_t>((total + 255) / 256, 4096));
        hipLaunchKernelGGL((total >> 31 ? &pack_chain_kernel<W, size_t> : &pack_chain_kernel<W, unsigned>),
                           dim3(blocks), dim3(256), 0, stream,
                           static_cast<const W *>(g[c.order[0]]),
                           static_cast<const W *>(g[c.order[1]]),
                           static_cast<const W *>(g[c.order[2]]),
                           reinterpret_cast<W *>(base + c.offF),
                           reinterpret_cast<W *>(base + c.offS),
                           reinterpret_cast<W *>(base + c.offL), a);
        const int st = check_hip(hipGetLastError(), "trk_pack: launch");
        if (st != TRK_OK) return st;
    }
    return TRK_OK;
}

// The joined-core section (trk_join_kernel.h): [header][J1][J2][J3].
//   J1[i][step][lane][8] = G1[a,p,i,b] as the formation's B fragments: column p = lane % 16 (zero
//                          at or past oP), K position 8 g + u of lane group g = lane / 16 being
//                          (a, b) in the order two results of the join (rows 4 g + u % 4) make a
//                          K step; fp32 stores u in two planes of four ([u / 4][lane][u % 4])
//   J2[q][j][b][c] = G2[b,q,j,c]
//   J3[r][k][a][c] = G3[c,r,k,a]
// fp16 cores are scaled by a power of two that brings the largest magnitude of each into [1/2, 1),
// which changes no bits but the exponent (values more than 2^13 below the largest become
// subnormal), and the header's first float is the factor that undoes it on the fp32 sums:
// products of two and three cores are formed in the cores' type, and cores far from 1 would leave
// fp16's range there. The header's next 3 x kPeaks floats are the largest magnitudes of the
// cores' parts (infinite where a part holds an infinity or a NaN), and the word kJoinUneven says
// whether a core is too uneven for one scale (join_spread_kernel). bf16 and fp32 have the range.
struct JoinArgs {
    int R, Rc, nI, nJ, nK, oP, oQ, oR;
    unsigned nJ1, nJ2, nJ3;  // (plan_join_chain keeps the section below 2^31 elements)
};

constexpr int kPeaks = 16;  // workgroups per core that look for its largest magnitude
static_assert(1 + 3 * kPeaks <= kJoinUneven && (kJoinUneven + 1) * 4 <= kJoinHeader,
              "the peaks and the verdict fit the header");

template <int DT>
__global__ void __launch_bounds__(1024) join_peak_kernel(
    const typename Elem<DT>::T *__restrict__ g1, const typename Elem<DT>::T *__restrict__ g2,
    const typename Elem<DT>::T *__restrict__ g3, size_t n1, size_t n2, size_t n3, float *peaks) {
    const typename Elem<DT>::T *g = blockIdx.y == 0 ? g1 : blockIdx.y == 1 ? g2 : g3;
    const size_t n = blockIdx.y == 0 ? n1 : blockIdx.y == 1 ? n2 : n3;
    float m = 0.0f;
#pragma unroll 8
    for (size_t i = blockIdx.x * 1024 + threadIdx.x; i < n; i += 1024 * kPeaks) {
        const float v = fabsf(Elem<DT>::to_f32(g[i]));
        m = v <= m ? m : v <= 3.4028234e38f ? v : INFINITY;
    }
    __shared__ float part[1024];
    part[threadIdx.x] = m;
    __syncthreads();
    for (int w = 512; w > 0; w /= 2) {
        if (threadIdx.x < w) part[threadIdx.x] = fmaxf(part[threadIdx.x], part[threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x == 0) peaks[blockIdx.y * kPeaks + blockIdx.x] = part[0];
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0)  // join_spread_kernel may raise it
        reinterpret_cast<unsigned *>(peaks - 1)[kJoinUneven] = 0;
}

__device__ inline float join_peak(const float *peaks) {
    float m = 0.0f;
    for (int i = 0; i < kPeaks; ++i) m = fmaxf(m, peaks[i]);
    return m;
}

// The power of two just above the largest of a core's peaks (0 if that is 0 or not finite).
__device__ inline int join_exponent(const float *peaks) {
    const float m = join_peak(peaks);
    int e = 0;
    if (m > 0.0f && m <= 3.4028234e38f) frexpf(m, &e);
    return e;
}

// Whether one scale per core keeps the joined kernel's fp16 intermediates (products of two and of
// three scaled cores) out of fp16's subnormals, where they would lose bits that the chains, which
// round only sums that x is part of, keep. One workgroup looks at one slice (one index of one of a
// core's four modes). The core is uneven if the mean magnitude of a slice's nonzero values is
// below 1/16 of the core's peak, or more than a quarter of them lie below 1/64 of it. Values of
// an even core then average 2^-5 at least after the scaling, H 2^-8.5 and W 2^-10 at rank 8 (the
// fewest terms): 4 bits above the subnormals. Normal, uniform and Laplace values pass (means of
// 1/6, 1/2 and 1/12 of the peak of 10^5 values), digits whose sizes differ by 3 in all three cores
// just so. In a model of both kernels' roundings every set of cores that passes has the
// chains' error (2.9e-4), and the first to lose a tenth more is far past the bound.
constexpr float kJoinMean = 16.0f, kJoinSmall = 64.0f;
constexpr unsigned kJoinSmallShare = 4;

__global__ void __launch_bounds__(1024) join_spread_kernel(const _Float16 *__restrict__ g1,
                                                           const _Float16 *__restrict__ g2,
                                                           const _Float16 *__restrict__ g3,
                                                           float *header, JoinArgs a) {
    const int k = blockIdx.y;
    const _Float16 *g = k == 0 ? g1 : k == 1 ? g2 : g3;
    const unsigned dims[4] = {unsigned(a.Rc), unsigned(k == 0 ? a.oP : k == 1 ? a.oQ : a.oR),
                              unsigned(k == 0 ? a.nI : k == 1 ? a.nJ : a.nK), unsigned(a.Rc)};
    unsigned slice = blockIdx.x, mode = 0;
    while (mode < 4 && slice >= dims[mode]) slice -= dims[mode++];
    if (mode == 4) return;  // (the grid is as wide as the core with the most slices)
    unsigned inner = 1, all = dims[0] * dims[1] * dims[2] * dims[3];
    for (unsigned m = mode + 1; m < 4; ++m) inner *= dims[m];
    const unsigned n = all / dims[mode];
    const float peak = join_peak(header + 1 + k * kPeaks);
    float sum = 0.0f;
    unsigned nonzero = 0, small = 0;
#pragma unroll 8
    for (unsigned e = threadIdx.x; e < n; e += 1024) {
        const float v = fabsf(float(g[(e / inner * dims[mode] + slice) * inner + e % inner]));
        sum += v;
        nonzero += v != 0.0f;
        small += v != 0.0f && v * kJoinSmall < peak;
    }
    __shared__ float sums[16];
    __shared__ unsigned counts[16], smalls[16];
    for (int w = 32; w > 0; w /= 2) {
        sum += __shfl_xor(sum, w);
        nonzero += __shfl_xor(nonzero, w);
        small += __shfl_xor(small, w);
    }
    if (threadIdx.x % 64 == 0) {
        sums[threadIdx.x / 64] = sum;
        counts[threadIdx.x / 64] = nonzero;
        smalls[threadIdx.x / 64] = small;
    }
    __syncthreads();
    if (threadIdx.x) return;
    for (int w = 1; w < 16; ++w) {
        sum += sums[w];
        nonzero += counts[w];
        small += smalls[w];
    }
    if (nonzero && (!(peak <= 3.4028234e38f) || sum * kJoinMean < peak * nonzero ||
                    small * kJoinSmallShare > nonzero))
        atomicOr(reinterpret_cast<unsigned *>(header) + kJoinUneven, 1u);
}

// The verdict to pinned host memory. (With a 4-byte copy in its place and 256 threads a slice in
// join_spread_kernel, preparing 1920 -> 2880 took 74 us at rank 8 and 80 at rank 16; 66 and 71 now.)
__global__ void join_verdict_kernel(const unsigned *__restrict__ header, unsigned *host) {
    *host = header[kJoinUneven];
}

template <int DT>
__global__ void __launch_bounds__(256) join_pack_kernel(
    const typename Elem<DT>::T *__restrict__ g1, const typename Elem<DT>::T *__restrict__ g2,
    const typename Elem<DT>::T *__restrict__ g3, char *__restrict__ out, JoinArgs a) {
    using E = Elem<DT>;
    using T = typename E::T;
    int exponents[3] = {0, 0, 0};
    if constexpr (DT == TRK_DTYPE_F16)
        for (int k = 0; k < 3; ++k)
            exponents[k] = join_exponent(reinterpret_cast<const float *>(out) + 1 + k * kPeaks);
    const int R = a.R, R2 = R * R;
    T *dst = reinterpret_cast<T *>(out + kJoinHeader);
    const unsigned total = a.nJ1 + a.nJ2 + a.nJ3;
    if (blockIdx.x == 0 && threadIdx.x == 0)
        *reinterpret_cast<float *>(out) = ldexpf(1.0f, exponents[0] + exponents[1] + exponents[2]);
    for (unsigned d = blockIdx.x * blockDim.x + threadIdx.x; d < total; d += gridDim.x * blockDim.x) {
        float v = 0.0f;
        int core = 0;
        if (d < a.nJ1) {
            const unsigned e = d;
            const int in = int(e % 512), s = int(e / 512 % (R2 / 32)), i = int(e / 512 / (R2 / 32));
            const int lane = sizeof(T) == 2 ? in / 8 : in % 256 / 4;
            const int u = sizeof(T) == 2 ? in % 8 : in / 256 * 4 + in % 4;
            const int p = lane % 16, g = lane / 16;
            const int ca = R == 8 ? 4 * s + u / 4 * 2 + g / 2 : 2 * s + u / 4;
            const int cb = R == 8 ? 4 * (g % 2) + u % 4 : 4 * g + u % 4;
            if (p < a.oP && ca < a.Rc && cb < a.Rc)
                v = E::to_f32(g1[core_index(ca, p, i, cb, a.oP, a.nI, a.Rc)]);
        } else if (d < a.nJ1 + a.nJ2) {
            const unsigned e = d - a.nJ1;
            const int cc = int(e % R), cb = int(e / R % R), j = int(e / R2 % a.nJ);
            const int q = int(e / R2 / a.nJ);
            core = 1;
            if (cb < a.Rc && cc < a.Rc)
                v = E::to_f32(g2[core_index(cb, q, j, cc, a.oQ, a.nJ, a.Rc)]);
        } else {
            const unsigned e = d - a.nJ1 - a.nJ2;
            const int cc = int(e % R), ca = int(e / R % R), k = int(e / R2 % a.nK);
            const int r = int(e / R2 / a.nK);
            core = 2;
            if (ca < a.Rc && cc < a.Rc)
                v = E::to_f32(g3[core_index(cc, r, k, ca, a.oR, a.nK, a.Rc)]);
        }
        dst[d] = E::from_f32(ldexpf(v, core == 0   ? -exponents[0]
                                       : core == 1 ? -exponents[1]
                                                   : -exponents[2]));
    }
}

template <int DT>
int pack_join(const Plan &plan, const Chain &c, const void *const g[3], void *packed,
              hipStream_t stream) {
    using T = typename Elem<DT>::T;
    char *out = static_cast<char *>(packed) + c.offF;
    const unsigned R2 = c.R * c.R;
    const T *t[3] = {static_cast<const T *>(g[0]), static_cast<const T *>(g[1]),
                     static_cast<const T *>(g[2])};
    JoinArgs a{c.R, plan.core_rank,
               plan.in_modes[0], plan.in_modes[1], plan.in_modes[2],
               plan.out_modes[0], plan.out_modes[1], plan.out_modes[2],
               R2 * 16 * plan.in_modes[0], R2 * plan.in_modes[1] * plan.out_modes[1],
               R2 * plan.in_modes[2] * plan.out_modes[2]};
    if constexpr (DT == TRK_DTYPE_F16) {
        size_t n[3];
        for (int k = 0; k < 3; ++k)
            n[k] = size_t(plan.core_rank) * plan.core_rank * plan.in_modes[k] * plan.out_modes[k];
        int slices = 0;
        for (int k = 0; k < 3; ++k)
            slices = std::max(slices, 2 * plan.core_rank + plan.in_modes[k] + plan.out_modes[k]);
        float *header = reinterpret_cast<float *>(out);
        hipLaunchKernelGGL(join_peak_kernel<DT>, dim3(kPeaks, 3), dim3(1024), 0, stream, t[0], t[1],
                           t[2], n[0], n[1], n[2], header + 1);
        hipLaunchKernelGGL(join_spread_kernel, dim3(slices, 3), dim3(1024), 0, stream,
                           static_cast<const _Float16 *>(g[0]), static_cast<const _Float16 *>(g[1]),
                           static_cast<const _Float16 *>(g[2]), header, a);
    }
    const unsigned total = a.nJ1 + a.nJ2 + a.nJ3;
    hipLaunchKernelGGL(join_pack_kernel<DT>, dim3(std::min(total / 256 + 1, 4096u)), dim3(256), 0,
                       stream, t[0], t[1], t[2], out, a);
    return check_hip(hipGetLastError(), "trk_pack: launch");
}

}  // namespace

int launch_join_verdict(const void *section, unsigned *host, hipStream_t stream) {
    hipLaunchKernelGGL(join_verdict_kernel, dim3(1), dim3(1), 0, stream,
                       static_cast<const unsigned *>(section), host);
    return check_hip(hipGetLastError(), "trk_plan_admit: launch");
}

int launch_pack(const Plan &plan, const void *g1, const void *g2, const void *g3, void *packed,
                hipStream_t stream) {
    const void *g[3] = {g1, g2, g3};
    for (int ci = 0; ci < plan.nchains; ++ci) {
        const Chain &c = plan.chains[ci];
        if (!c.join) continue;
        const int st = plan.dtype == TRK_DTYPE_F16    ? pack_join<TRK_DTYPE_F16>(plan, c, g, packed, stream)
                       : plan.dtype == TRK_DTYPE_BF16 ? pack_join<TRK_DTYPE_BF16>(plan, c, g, packed, stream)
                                                      : pack_join<TRK_DTYPE_F32>(plan, c, g, packed, stream);
        if (st != TRK_OK) return st;
    }
    if (plan.elem == 4) return pack_all<uint32_t>(plan, g, packed, stream);
    return pack_all<uint16_t>(plan, g, packed, stream);
}

}  // namespace trk
