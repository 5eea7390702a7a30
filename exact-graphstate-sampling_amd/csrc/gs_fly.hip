// Butterfly sweeps (gs_fly.h): NS steps of a run on each group of 2^D entries a thread holds (D = NS, or NS + 1 when the
// norms of the step after them are summed too).  A single step moves the table once per step at the HBM rate with its
// FP64 work a quarter of that time, so sweeps of more steps move it less:
//   chain mode (weights known): two, three or four steps per read and write of the table.  Complex64 width 29: 8.3 ms per
//   string with pairs of steps only, 7.5 ms with up to three, 6.8 ms with up to four (208 VGPRs, two waves per SIMD, and
//   FP64 work as long as the traffic); complex128 width 21: 97, 71 and 62 us.
//   sampled and forced complex128 strings: steps k and k+1 per read and write, the write folding in step k+2's norms; step
//   k+1's decision comes before from a read-only pass that applies step k in registers (WRITE false) and sums step k+1's
//   norms: three passes over the table per two steps instead of four (width 23 1.68 -> 1.47 ms per sample, width 26 6.76
//   -> 5.88).  Complex64 strings gain 3-7 % from it at most (their forced ones lose 20 %: 16 FP64 products more per
//   entry), and their norms would be summed in another order, which moves the rounding of stored values.
// Values between the steps are rounded to the storage type as they would be in memory.  Slot indices are uniform over
// the lanes of a wave, only signs differ, so a step's route is a uniform branch.
#include "gs_chain.h"
#include "gs_fly.h"

namespace gs {

namespace {

enum { kNormNone = 0, kNormGram = 1, kNormDirect = 2 };

// Step i on the group's entries.  p: parities of the thread's base, its slot indices the same over the wave; pe: of the
// entries relative to it; prun: of the run's second element.  Sums: the step's written norm (chain mode), or the last
// step's written and stored norms.
template <int ROUTE, int I, class S, int VR, int NE, int NA, int NORM, bool LAST>
__device__ __forceinline__ void fly_level(uint32_t par, uint32_t p, uint32_t prun, const uint32_t (&pe)[NE],
                                          const double2 (&w)[2], S (&v)[NE][VR], double (&acc)[NA]) {
#pragma unroll
    for (int e = 0; e < NE; e++) {
        if ((e >> I) & 1) continue;
        const uint32_t J = uint32_t(__builtin_amdgcn_readfirstlane(int(p ^ pe[e])) >> (4 + I)) & 1;
#pragma unroll
        for (int x = 0; x < VR; x++) {
            double2 ylo, yhi;
            fly_pair<ROUTE>(par, J, ((p ^ pe[e] ^ (x ? prun : 0)) >> I) & 1, Cx<S>::widen(v[e][x]),
                            Cx<S>::widen(v[e | (1 << I)][x]), w[0], w[1], ylo, yhi);
            v[e][x] = Cx<S>::narrow(ylo);
            v[e | (1 << I)][x] = Cx<S>::narrow(yhi);
            if constexpr (NORM == kNormNone) {
                add_norm(acc[I], ylo);
                add_norm(acc[I], yhi);
            } else if constexpr (LAST) {
                add_norm(acc[0], ylo);
                add_norm(acc[0], yhi);
                add_norm(acc[1], Cx<S>::widen(v[e][x]));
                add_norm(acc[1], Cx<S>::widen(v[e | (1 << I)][x]));
            }
        }
    }
}

// Norms of step I (not applied) from the group's values: direct branch norms, or the Gram matrix G00, G11, Re, Im G01.
template <int ROUTE, int I, class S, int VR, int NE, int NA, int NORM>
__device__ __forceinline__ void fly_norms(uint32_t par, uint32_t p, uint32_t prun, const uint32_t (&pe)[NE],
                                          const double2 (&M)[2][2], const S (&v)[NE][VR], double (&acc)[NA]) {
#pragma unroll
    for (int e = 0; e < NE; e++) {
        if ((e >> I) & 1) continue;
        const uint32_t J = uint32_t(__builtin_amdgcn_readfirstlane(int(p ^ pe[e])) >> (4 + I)) & 1;
#pragma unroll
        for (int x = 0; x < VR; x++) {
            const double2 lo = Cx<S>::widen(v[e][x]), hi = Cx<S>::widen(v[e | (1 << I)][x]);
            const uint32_t sg = ((p ^ pe[e] ^ (x ? prun : 0)) >> I) & 1;
            const uint32_t slo = sg ^ (J ? par : 0), shi = sg ^ (J ? 0 : par);
            auto flip = [](double a, uint32_t s) {
                return __hiloint2double(__double2hiint(a) ^ int(s << 31), __double2loint(a));
            };
            if constexpr (NORM == kNormDirect) {
#pragma unroll
                for (int b = 0; b < 2; b++) {
                    double2 ylo, yhi;
                    fly_pair<ROUTE>(par, J, sg, lo, hi, M[b][0], M[b][1], ylo, yhi);
                    add_norm(acc[2 + b], ylo);
                    add_norm(acc[2 + b], yhi);
                }
            } else if constexpr (ROUTE == kRouteMixA) {
                add_norm(acc[2], lo);
                add_norm(acc[2], hi);
                const double re = fma(lo.x, hi.x, lo.y * hi.y), im = fma(lo.y, hi.x, -lo.x * hi.y);
                acc[4] += flip(re, shi) + flip(re, slo);
                acc[5] += flip(im, shi) - flip(im, slo);
            } else if constexpr (ROUTE == kRouteMixB) {
                const double nl = norm2(lo), nh = norm2(hi);
                acc[2] += nl + nh;
                acc[4] += flip(nl, slo) + flip(nh, shi);
            } else {
                add_norm(acc[2], cadd(lo, hi));
                add_norm(acc[3], cadd(lo, flip_if(hi, par)));
            }
        }
    }
}

}  // namespace

template <class S, int NS, int NORM, bool WRITE>
__global__ __launch_bounds__(kThreads) void fly_kernel(const FlyDesc* __restrict__ fp, S* __restrict__ mem,
                                                       double* __restrict__ part, Ctl* __restrict__ ctl, Epi epi) {
    constexpr int D = NS + (NORM ? 1 : 0), NE = 1 << D, VR = 16 / int(sizeof(S)), LR = VR == 2 ? 1 : 0;
    constexpr int NA = NORM == kNormNone ? NS : NORM == kNormGram ? 6 : 4;
    const FlyDesc& f = *fp;
    mem += uint64_t(blockIdx.y) * epi.slot_entries;   // this block's string
    part += size_t(blockIdx.y) * epi.slot_part;
    ctl += blockIdx.y;
    if (ctl->dead) return;
    const int k0 = epi.k - (NORM && WRITE ? NS - 1 : 0);      // first step
    double2 w[NS][2];
    w[0][0] = make_double2(ctl->w[0], ctl->w[1]);
    w[0][1] = make_double2(ctl->w[2], ctl->w[3]);
    if constexpr (NORM != kNormNone && NS == 2) {
        w[1][0] = make_double2(ctl->w2[0], ctl->w2[1]);
        w[1][1] = make_double2(ctl->w2[2], ctl->w2[3]);
    } else {
#pragma unroll
        for (int i = 1; i < NS; i++) {
            const KStep& n = epi.plain[k0 + i];
            const int b = __builtin_amdgcn_readfirstlane(
                epi.forced[size_t(blockIdx.y) * size_t(epi.ns) + size_t(k0 + i)]);
            w[i][0] = make_double2(n.mre[b][0], n.mim[b][0]);
            w[i][1] = make_double2(n.mre[b][1], n.mim[b][1]);
        }
    }
    double2 M[2][2];
    if constexpr (NORM == kNormDirect) {
        const KStep& n = epi.plain[k0 + NS];
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int x = 0; x < 2; x++) M[b][x] = make_double2(n.mre[b][x], n.mim[b][x]);
    }
    int route[D];
    uint32_t par[D];
#pragma unroll
    for (int i = 0; i < D; i++) {
        route[i] = int(uniform_byte(f.route[i]));
        par[i] = uniform_byte(f.par[i]);
    }
    uint64_t de[NE];                                   // the group's entries relative to its base
    uint32_t pe[NE];
#pragma unroll
    for (int e = 0; e < NE; e++) {
        de[e] = 0;
        pe[e] = 0;
#pragma unroll
        for (int i = 0; i < D; i++)
            if ((e >> i) & 1) {
                de[e] ^= f.dir[i];
                pe[e] ^= uniform_byte(f.dn[i]);
            }
    }
    const int tid = threadIdx.x;
    uint64_t a = 0;
    uint32_t p = uniform_byte(f.cn);
#pragma unroll
    for (int b = 0; b < 8; b++)
        if ((tid >> b) & 1) {
            a ^= f.cols[LR + b];
            p ^= uniform_byte(f.pn[LR + b]);
        }
    const unsigned bid = f.xcd && f.lg_grid >= 3 ? (blockIdx.x >> 3) | ((blockIdx.x & 7u) << (f.lg_grid - 3))
                                                 : blockIdx.x;
    for (int b = 0; b < f.lg_grid; b++)
        if ((bid >> b) & 1) {
            a ^= f.cols[LR + 8 + b];
            p ^= f.pn[LR + 8 + b];
        }
    const uint32_t prun = LR ? uniform_byte(f.pn[0]) : 0;
    double acc[NA];
#pragma unroll
    for (int q = 0; q < NA; q++) acc[q] = 0;
    for (int it = 0; it < (1 << f.lg_iter); it++) {
        if (it > 0) {                                  // Gray code: one coordinate changes
            const int j = LR + 8 + f.lg_grid + __builtin_ctz(unsigned(it));
            a ^= f.cols[j];
            p ^= uniform_byte(f.pn[j]);
        }
        S v[NE][VR];
#pragma unroll
        for (int e = 0; e < NE; e++) Run<S, VR>::load(mem, (a ^ de[e]) & ~uint64_t(VR - 1), v[e]);
#pragma unroll
        for (int e = 0; e < NE; e++) permute<S, VR>(v[e], unsigned(de[e]) & (VR - 1));     // a has no run bit
        fly_each([&](auto i) {
            constexpr int I = decltype(i)::value;
            fly_route_of(route[I], [&](auto r) {
                fly_level<decltype(r)::value, I, S, VR, NE, NA, NORM, I == NS - 1>(par[I], p, prun, pe, w[I], v, acc);
            });
        }, std::make_integer_sequence<int, NS>{});
        if constexpr (NORM != kNormNone)               // norms of the step after them, from the rounded values
            fly_route_of(route[NS], [&](auto r) {
                fly_norms<decltype(r)::value, NS, S, VR, NE, NA, NORM>(par[NS], p, prun, pe, M, v, acc);
            });
        if constexpr (WRITE) {
#pragma unroll
            for (int e = 0; e < NE; e++) {
                permute<S, VR>(v[e], unsigned(de[e]) & (VR - 1));
                Run<S, VR>::store(mem, (a ^ de[e]) & ~uint64_t(VR - 1), v[e]);
            }
        }
    }
    if constexpr (NORM == kNormGram)
        if (route[NS] != kRouteSplit) acc[3] = acc[2];
    sweep_epilogue<NA, true>(acc, part, ctl, epi, NORM == kNormGram ? kWriteGram : NORM == kNormDirect ? kWriteDirect : kWrite);
}

namespace {
template <class S>
void* fly_for(int ns) {
    return ns == 4   ? reinterpret_cast<void*>(&fly_kernel<S, 4, kNormNone, true>)
           : ns == 3 ? reinterpret_cast<void*>(&fly_kernel<S, 3, kNormNone, true>)
                     : reinterpret_cast<void*>(&fly_kernel<S, 2, kNormNone, true>);
}
}  // namespace

// Chain mode: ns (2, 3 or 4) steps; storage 0 = c64 / 1 = c128.
void* fly_kernel_ptr(int storage, int ns) { return storage == 0 ? fly_for<float2>(ns) : fly_for<double2>(ns); }

// c128, norm 1 Gram / 2 direct: two steps written with the third one's norms, or (write false) the read-only pass before.
void* fly_norm_kernel_ptr(int norm, bool write) {
    if (write)
        return norm == kNormGram ? reinterpret_cast<void*>(&fly_kernel<double2, 2, kNormGram, true>)
                                 : reinterpret_cast<void*>(&fly_kernel<double2, 2, kNormDirect, true>);
    return norm == kNormGram ? reinterpret_cast<void*>(&fly_kernel<double2, 1, kNormGram, false>)
                             : reinterpret_cast<void*>(&fly_kernel<double2, 1, kNormDirect, false>);
}

}  // namespace gs
