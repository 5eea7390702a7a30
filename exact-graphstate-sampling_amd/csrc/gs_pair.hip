// Two steps per sweep of the in-place arena, for the modes whose weights are known beforehand (chain mode: no scale, every
// bit forced).  A chain step alone is one read and one write of the table at the HBM rate; two steps in one sweep move
// the same bytes once (see gs_pair.h).  A thread owns one aligned 16-byte run per slot (VR super-cosets, the unit bit 0
// their first coordinate); the 8 coordinates of the threads, like the run's, never change step k+1's slot index, so all
// routing is uniform and only signs differ between lanes.  The table between the steps is rounded to the storage type
// in registers: the stored tables are those of single steps bit for bit, the norms up to the order of their FP64 sums.
// Measured on chain strings, one step against two per sweep: width 29 complex64 15.4 -> 8.3 ms, width 26 4.2 -> 2.55 ms,
// width 24 0.73 -> 0.58 ms, width 20 complex128 184 -> 90 us (12 together).
#include "gs_chain.h"
#include "gs_pair.h"
#include "gs_pstep.h"

namespace gs {

template <class S, int NQ, int NI, int MO, bool DEG>
__global__ __launch_bounds__(kThreads) void pair_sweep_kernel(const PStep* __restrict__ pp, S* __restrict__ mem,
                                                              double* __restrict__ part, Ctl* __restrict__ ctl,
                                                              Epi epi) {
    constexpr int NU = DEG ? 1 : MO, VR = 16 / int(sizeof(S)), LR = VR == 2 ? 1 : 0;
    const PStep& s = *pp;
    const PairDesc& P = s.d;
    mem += uint64_t(blockIdx.y) * epi.slot_entries;   // this block's string
    part += size_t(blockIdx.y) * epi.slot_part;
    ctl += blockIdx.y;
    if (ctl->dead) return;
    const double2 w0 = make_double2(ctl->w[0], ctl->w[1]), w1 = make_double2(ctl->w[2], ctl->w[3]);
    const KStep& n = epi.plain[epi.k + 1];
    const int b1 = __builtin_amdgcn_readfirstlane(epi.forced[size_t(blockIdx.y) * size_t(epi.ns) + epi.k + 1]);
    const double2 x0 = make_double2(n.mre[b1][0], n.mim[b1][0]), x1 = make_double2(n.mre[b1][1], n.mim[b1][1]);
    const PairRegs r(P, PairSteps{s.off, s.g1, s.m1, s.t0m, s.t1m, s.parm, s.u0m, s.u1m, s.uparm});
    const int tid = threadIdx.x;
    uint64_t a_tb = 0;
    uint32_t p_tb = 0, ph_b = 0;
#pragma unroll
    for (int b = 0; b < 8; b++)
        if ((tid >> b) & 1) {
            a_tb ^= P.cols[LR + b];
            p_tb ^= P.pn[LR + b];
        }
    const unsigned bid = s.xcd && s.lg_grid >= 3 ? (blockIdx.x >> 3) | ((blockIdx.x & 7u) << (s.lg_grid - 3))
                                                 : blockIdx.x;
    for (int b = 0; b < s.lg_grid; b++)
        if ((bid >> b) & 1) {
            a_tb ^= P.cols[LR + 8 + b];
            p_tb ^= P.pn[LR + 8 + b];
            ph_b ^= P.pn[LR + 8 + b];
        }
    const int jit = LR + 8 + s.lg_grid;
    const uint32_t p_run = LR ? P.pn[0] : 0;          // parities of the run's second super-coset
    double acc[2] = {0, 0};
    for (int it = 0; it < (1 << s.lg_iter); it++) {
        if (it > 0) {                                 // Gray code: one coordinate changes
            const int j = jit + __builtin_ctz(unsigned(it));
            a_tb ^= P.cols[j];
            p_tb ^= P.pn[j];
            ph_b ^= P.pn[j];
        }
        const uint32_t ph = __builtin_amdgcn_readfirstlane(ph_b);
        S v[NI][NQ][VR];
#pragma unroll
        for (int i = 0; i < NI; i++)
#pragma unroll
            for (int q = 0; q < NQ; q++)
                Run<S, VR>::load(mem, (a_tb ^ r.lab[i] ^ r.off[q]) & ~uint64_t(VR - 1), v[i][q]);
        S f[NU][2][VR];
#pragma unroll
        for (int i = 0; i < NI; i++)
#pragma unroll
            for (int q = 0; q < NQ; q++) permute<S, VR>(v[i][q], unsigned(a_tb ^ r.lab[i] ^ r.off[q]) & (VR - 1));
#pragma unroll
        for (int x = 0; x < VR; x++) {
            const uint32_t pa = p_tb ^ (x ? p_run : 0);
            double2 e[NI][MO];
#pragma unroll
            for (int i = 0; i < NI; i++) {
                S vi[NQ];
#pragma unroll
                for (int q = 0; q < NQ; q++) vi[q] = v[i][q][x];
                double2 A[2][2];
                pair_route0<S, NQ>(r, vi, pa, i, A);
#pragma unroll
                for (int t = 0; t < MO; t++) {
                    const double2 o = cfma(w0, A[t][0], cmul(w1, A[t][1]));
                    add_norm(acc[0], o);
                    e[i][t] = Cx<S>::widen(Cx<S>::narrow(o));
                }
            }
#pragma unroll
            for (int c = 0; c < NU; c++) {
                double2 A[2][2];
                pair_route1<NI, MO, DEG>(r, e, pa, ph, c, A);
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    const double2 o = cfma(x0, A[t][0], cmul(x1, A[t][1]));
                    if (t == 0 || r.m1 == 2) add_norm(acc[1], o);
                    f[c][t][x] = Cx<S>::narrow(o);
                }
            }
        }
#pragma unroll
        for (int c = 0; c < NU; c++)
#pragma unroll
            for (int t = 0; t < 2; t++) {
                if (t == 1 && r.m1 != 2) break;
                const uint64_t at = r.out(a_tb, ph, c) ^ (t ? r.g1 : 0);
                permute<S, VR>(f[c][t], unsigned(at) & (VR - 1));
                Run<S, VR>::store(mem, at & ~uint64_t(VR - 1), f[c][t]);
            }
    }
    sweep_epilogue<2, true>(acc, part, ctl, epi, kWrite);
}

namespace {

template <class S, int NQ>
void* by_kind(int ni, int mo, int deg) {
#define GS_PK(a, b, c) \
    if (ni == a && mo == b && deg == c) return reinterpret_cast<void*>(&pair_sweep_kernel<S, NQ, a, b, c>);
    GS_PK(1, 1, 0) GS_PK(1, 2, 0) GS_PK(1, 2, 1) GS_PK(2, 1, 0) GS_PK(2, 2, 0) GS_PK(2, 2, 1) GS_PK(4, 1, 0) GS_PK(4, 2, 0)
#undef GS_PK
    return nullptr;
}

template <class S>
void* by_slots(int nq, int ni, int mo, int deg) {
    return nq == 1 ? by_kind<S, 1>(ni, mo, deg) : nq == 2 ? by_kind<S, 2>(ni, mo, deg) : by_kind<S, 4>(ni, mo, deg);
}

}  // namespace

// Sweep of a pair (storage 0 = c64 / 1 = c128; the slots of step k and the kind of pair); nullptr when not built.
void* pair_sweep_kernel_ptr(int storage, int nq, int ni, int mo, int deg) {
    return storage == 0 ? by_slots<float2>(nq, ni, mo, deg) : by_slots<double2>(nq, ni, mo, deg);
}

}  // namespace gs
