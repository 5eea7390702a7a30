// Runs of small steps in one block per string.
//
// The head and tail of a plan are steps of a few thousand cosets and less, where a sweep costs far less than a launch;
// one block runs such a run step after step -- norm pass, decision, write pass, bookkeeping -- with the run's table in
// LDS: the arena slots a run touches span a subspace of at most 64 KB, or the whole arena where that fits (build_small in
// gs_engine.hip), and the host gives every step's
// columns, offsets and g as indices into that subspace.  The arithmetic per coset is the sweep kernels' (FP64 routed slot
// sums, one rounding per store), the chain logic theirs too (gsamp2.cpp:46-49, :67, :80-95).
//
// What bounds it is latency: a step has little to compute and two sums over the cosets that the next pass needs.  So
// the chain state lives in registers of every thread (each makes the decision itself, no broadcast), sums go through
// lane swaps and DPP inside a wave and one barrier across waves, steps of at most 64 cosets run on the first wave with no
// barrier at all (narrow_steps), every descriptor, bit and uniform is in LDS before the first step, and the logarithms,
// which no decision needs, are taken for all steps at once at the end.  A version with the table in the arena, state
// changes by one thread and two barriers per pass took 4.6 us per step; with one code for all steps it was 2.0 us, and
// this one takes 1.3 us (the n = 24 plan, 24 steps, complex64: 115 -> 49.5 -> 33.6 us).
#include "gs_math.h"
#include "gs_wave.h"

namespace gs {

namespace {

constexpr int kWavesS = kSmallThreads / 64;
static_assert(kSmallMaxNk < 15, "narrow_steps keeps an index and a sign in 16 bits");

// A step of at most 64 cosets, as the first wave reads it: offsets two to a word, g, and kind | m << 5 | par << 8 |
// growth << 12 | next step's growth << 13 | nk << 16.
struct NStep {
    uint32_t o01, o23, g, bits;
};

struct Shared {                       // after the table in LDS
    SStep s[kSmallSteps];
    NStep n[kSmallSteps];
    double coef[kSmallSteps][2][4];   // per branch |m0|^2, |m1|^2, Re and Im of m0 conj(m1)
    uint16_t word[kSmallSteps][64];   // per lane: index of its coset's base, its sign in bit 15
    double U[kSmallSteps];
    double pfac[kSmallSteps], plog[kSmallSteps];      // factors of Pr, and their log2 at the end of the run
    double sfac[kSmallSteps], slog[kSmallSteps];      // table norms of the rescalings (kRun), and their log2
    double cond[kSmallSteps];
    double sum[2][kWavesS][4];
    Ctl c;
    int np, nsf, kdone;
    int8_t forced[kSmallSteps], bits[kSmallSteps];
};

// Chain state of a run, the same in every thread that runs the step.
struct State {
    double prev, nstored;
    double2 w0, w1;
    double sc;
    int bv, dead, qidx;
    int np, nsf;                      // entries of pfac, sfac
    int buf;                          // buffer of the next sum across waves (the last one may still be read)
    bool neglog;                      // a zero-probability branch: log2 Pr = -inf
};

// Sums of a pass over the threads that run it, in every one of them.  nw: waves with cosets (the others' sums are zeros);
// across waves lane q adds up value q, in wave order.
template <bool WIDE, int NQ>
__device__ __forceinline__ void pass_sum(Shared& sh, int& buf, const double (&v)[4], double (&out)[4], int nw) {
    const int lane = threadIdx.x & 63;
    const double r = NQ == 4 ? sum4(v) : NQ == 2 ? sum2(v) : wave_sum(v[0]);
    if constexpr (WIDE) {
        const int wave = threadIdx.x >> 6, row = lane >> 4;
        if ((lane & 15) == 0) sh.sum[buf][wave][NQ == 4 ? (row >> 1) | (row & 1) << 1 : row >> 1] = r;   // see sum2, sum4
        __syncthreads();
        double x = sh.sum[buf][0][lane & 3];
#pragma unroll
        for (int w = 1; w < kWavesS; w++) {
            if (w >= nw) break;
            x += sh.sum[buf][w][lane & 3];
        }
        buf ^= 1;
#pragma unroll
        for (int q = 0; q < NQ; q++) out[q] = lane_value(x, q);
    } else {
#pragma unroll
        for (int q = 0; q < NQ; q++) out[q] = lane_value(r, NQ == 4 ? 32 * (q & 1) + 16 * (q >> 1) : 32 * q);
    }
}

// Routed slot sums A[tau][x] of the coset at a (sign pc), slots in ascending order; kind: slots * 4 + Route, uniform.
template <class S, int NTQ, int ROUTE>
__device__ __forceinline__ void slot_sums(const S* tab, uint32_t a, const uint32_t (&off)[4], uint32_t pc, uint32_t par,
                                          double2 (&A)[2][2]) {
    S v[NTQ];
#pragma unroll
    for (int j = 0; j < NTQ; j++) v[j] = tab[a ^ off[j]];
    A[0][0] = A[0][1] = A[1][0] = A[1][1] = make_double2(-0.0, -0.0);
#pragma unroll
    for (int j = 0; j < NTQ; j++) {
        const double2 w = Cx<S>::widen(v[j]);
        const int neg = int((pc ^ (par >> j)) << 31);
        const double2 ws = make_double2(__hiloint2double(__double2hiint(w.x) ^ neg, __double2loint(w.x)),
                                        __hiloint2double(__double2hiint(w.y) ^ neg, __double2loint(w.y)));
        constexpr bool MIX = ROUTE == kRouteMixA || ROUTE == kRouteMixB;
        const int t0 = MIX ? j & 1 : 0;
        const int t1 = ROUTE == kRoute1 ? 0 : ROUTE == kRouteSplit ? 1 : ROUTE == kRouteMixA ? 1 - (j & 1) : (j & 1);
        A[t0][0] = cadd(A[t0][0], w);
        A[t1][1] = cadd(A[t1][1], ws);
    }
}
template <class S>
__device__ __forceinline__ void slot_sums_of(int kind, const S* tab, uint32_t a, const uint32_t (&off)[4], uint32_t pc,
                                             uint32_t par, double2 (&A)[2][2]) {
    switch (kind) {
        case 1 * 4 + kRoute1: slot_sums<S, 1, kRoute1>(tab, a, off, pc, par, A); break;
        case 1 * 4 + kRouteSplit: slot_sums<S, 1, kRouteSplit>(tab, a, off, pc, par, A); break;
        case 2 * 4 + kRoute1: slot_sums<S, 2, kRoute1>(tab, a, off, pc, par, A); break;
        case 2 * 4 + kRouteSplit: slot_sums<S, 2, kRouteSplit>(tab, a, off, pc, par, A); break;
        case 2 * 4 + kRouteMixA: slot_sums<S, 2, kRouteMixA>(tab, a, off, pc, par, A); break;
        case 2 * 4 + kRouteMixB: slot_sums<S, 2, kRouteMixB>(tab, a, off, pc, par, A); break;
        case 4 * 4 + kRoute1: slot_sums<S, 4, kRoute1>(tab, a, off, pc, par, A); break;
        case 4 * 4 + kRouteSplit: slot_sums<S, 4, kRouteSplit>(tab, a, off, pc, par, A); break;
        case 4 * 4 + kRouteMixA: slot_sums<S, 4, kRouteMixA>(tab, a, off, pc, par, A); break;
        default: slot_sums<S, 4, kRouteMixB>(tab, a, off, pc, par, A); break;
    }
}

// One step on one wave (at most 64 cosets) or on the whole block.  last: the run's last step, whose outputs go to the
// arena.  A thread with one coset keeps its slot sums from the norm pass for the write.
template <class S, bool WIDE>
__device__ __forceinline__ void small_step(Shared& sh, S* tab, S* mem, const KStep* plain, const Epi& e, State& st, int k,
                                           int k0, bool decided, bool last) {
    const SStep& s = sh.s[k - k0];
    const int t = threadIdx.x;
    constexpr int T = WIDE ? kSmallThreads : 64;
    constexpr int LT = WIDE ? 9 : 6;
    auto uni = [](uint32_t v) { return uint32_t(__builtin_amdgcn_readfirstlane(int(v))); };
    const int nk = int(uni(uint32_t(s.nk))), m = int(uni(uint32_t(s.m))), kind = int(uni(uint32_t(s.kind)));
    const uint32_t par = uni(s.par), rho = uni(s.rho), g = uni(s.g);
    uint32_t off[4];
#pragma unroll
    for (int j = 0; j < 4; j++) off[j] = uni(s.off[j]);
    uint32_t bt = 0;
#pragma unroll
    for (int j = 0; j < LT; j++)                               // columns beyond nk are 0
        bt ^= ((t >> j) & 1) ? s.cols[j] : 0;
    double2 M[2][2];
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
        for (int x = 0; x < 2; x++) M[b][x] = make_double2(s.mre[b][x], s.mim[b][x]);
    const uint32_t n = 1u << nk;
    const bool one = !WIDE || n <= uint32_t(T);
    const int nw = n >= uint32_t(T) ? kWavesS : int(n >> 6);    // only the wide path asks
    // index of coset c (c = t mod T) and its routed slot sums
    auto index_of = [&](uint32_t c) {
        uint32_t a = bt;
        if constexpr (WIDE)
#pragma unroll
            for (int j = LT; j < kSmallMaxNk; j++) a ^= ((c >> j) & 1) ? s.cols[j] : 0;
        return a;
    };
    double2 A[2][2];
    auto sums = [&](uint32_t a, uint32_t c) { slot_sums_of<S>(kind, tab, a, off, uint32_t(__popc(c & rho)) & 1, par, A); };
    bool have = false;                                         // A holds the sums of this thread's only coset
    // Norms the decision needs: none when it is forced or made without them (chain1, forced hybrid steps) or follows
    // from the stored norm (growth steps), direct branch norms for a forced string, else the Gram matrix.
    if (!decided) {
        int bv = e.forced ? int(sh.forced[k - k0]) : -1;
        const bool need_p = e.mode == kChain || (e.mode == kRun && bv < 0);
        const int growth = int(uni(uint32_t(s.growth)));
        double n2[2] = {0, 0};
        if (need_p && growth) {
#pragma unroll
            for (int b = 0; b < 2; b++) n2[b] = (norm2(M[b][0]) + norm2(M[b][1])) * st.nstored;
        } else if (need_p) {
            double acc[4] = {0, 0, 0, 0}, red[4];
            const bool direct = e.mode == kChain && e.forced;
            for (uint32_t c = t; c < n; c += T) {
                sums(index_of(c), c);
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const double2 a = A[q][0], b = A[q][1];
                    if (direct) {
                        add_norm(acc[0], cfma(M[0][0], a, cmul(M[0][1], b)));
                        add_norm(acc[1], cfma(M[1][0], a, cmul(M[1][1], b)));
                    } else {
                        add_norm(acc[0], a);
                        add_norm(acc[1], b);
                        acc[2] = fma(a.x, b.x, fma(a.y, b.y, acc[2]));
                        acc[3] = fma(a.y, b.x, fma(-a.x, b.y, acc[3]));
                    }
                }
            }
            have = one;
            if (direct) pass_sum<WIDE, 2>(sh, st.buf, acc, red, nw);
            else pass_sum<WIDE, 4>(sh, st.buf, acc, red, nw);
#pragma unroll
            for (int b = 0; b < 2; b++) {
                const double2 m0 = M[b][0], m1 = M[b][1];
                const double pr = m0.x * m1.x + m0.y * m1.y, pi = m0.y * m1.x - m0.x * m1.y;   // m0 conj(m1)
                n2[b] = direct ? red[b] : norm2(m0) * red[0] + norm2(m1) * red[1] + 2 * (pr * red[2] - pi * red[3]);
            }
        }
        double sc = 1.0;
        if (e.mode == kChain) {
            double both = 1.0 / sqrt((t & 1) ? n2[1] : n2[0]);  // lane 0: branch 0, lane 1: branch 1
            double p1 = n2[1] / (n2[0] + n2[1]);
            here(both);                                         // the two beside each other
            here(p1);
            if (bv < 0) bv = sh.U[k - k0] < p1;
            const double pb = bv ? p1 : 1 - p1;
            if (pb <= 0) {
                st.neglog = true;
                st.dead = 1;
                return;
            }
            if (t == 0) sh.pfac[st.np] = pb;
            st.np++;
            sc = lane_value(both, __builtin_amdgcn_readfirstlane(bv));
        } else if (e.mode == kRun) {
            sc = 1.0 / sqrt(st.prev);
            if (bv < 0) bv = sh.U[st.qidx++] < n2[1] / (n2[0] + n2[1]);
        }
        bv = __builtin_amdgcn_readfirstlane(bv);
        if (t == 0) sh.bits[k - k0] = int8_t(bv);
        st.bv = bv;
        st.sc = sc;
        const double2 m0 = bv ? M[1][0] : M[0][0], m1 = bv ? M[1][1] : M[0][1];
        st.w0 = make_double2(m0.x * sc, m0.y * sc);
        st.w1 = make_double2(m1.x * sc, m1.y * sc);
    }
    double acc[4] = {0, 0, 0, 0}, red[4];
    for (uint32_t c = t; c < n; c += T) {
        const uint32_t a = index_of(c);
        if (!have) sums(a, c);
        uint64_t pa = 0;
        if (last)
            for (int j = 0; j < nk; j++)
                if ((c >> j) & 1) pa ^= plain[k].cols[j];
#pragma unroll
        for (int q = 0; q < 2; q++) {
            if (q >= m) break;
            const double2 v = cfma(st.w0, A[q][0], cmul(st.w1, A[q][1]));
            const S sv = Cx<S>::narrow(v);
            if (last) mem[q ? pa ^ plain[k].g : pa] = sv;
            else tab[q ? a ^ g : a] = sv;
            add_norm(acc[0], v);
            add_norm(acc[1], Cx<S>::widen(sv));
        }
    }
    if constexpr (!WIDE) wave_fence();
    // the written norm is used outside the renormalised chain, the stored one by a growth step or after the run
    const bool stored = e.mode != kChain1 && (last || uni(uint32_t(sh.s[k + 1 - k0].growth)) != 0);
    if (e.mode == kChain && !stored) {
        if constexpr (WIDE) __syncthreads();
        return;
    }
    if (stored) pass_sum<WIDE, 2>(sh, st.buf, acc, red, nw);
    else pass_sum<WIDE, 1>(sh, st.buf, acc, red, nw);
    if (stored) st.nstored = red[1];
    const double nb = red[0];
    if (e.mode == kChain1) {                                   // gsamp2.cpp:67
        if (t == 0) sh.cond[k - k0] = nb / (2 * st.prev);
        st.prev = nb;
        if (nb <= 0) st.dead = 1;
    } else if (e.mode == kRun) {                               // gsamp2.cpp:93-95
        const double cd = nb / 2;
        if (t == 0) {
            sh.sfac[st.nsf] = st.prev;
            sh.cond[k - k0] = cd;
            sh.pfac[st.np] = cd;
        }
        st.nsf++;
        st.prev = nb;
        if (nb <= 0) st.dead = 1;
        else st.np++;
    }
    if (e.mode != kChain && nb <= 0) st.neglog = true;
}

// Steps from k on while they have at most 64 cosets (before step `to`), on the first wave alone; returns the step it
// stopped at.  The chain from one step to the next is all latency -- slots from LDS, sums over the wave, a square root and
// a division, the outputs -- so everything else is out of it: bases and signs of every lane were computed for all steps
// at once, the next step's are fetched during this one, four sums share one butterfly, and both branches' scales are
// taken on two lanes while p1 is divided.
template <class S, int MODE>
__device__ __forceinline__ int narrow_steps(Shared& sh, S* tab, bool forced, State& st, int k, int k0, int to) {
    const int t = threadIdx.x;
    auto uni = [](uint32_t v) { return uint32_t(__builtin_amdgcn_readfirstlane(int(v))); };
    NStep nx = sh.n[k - k0];
    uint32_t word = sh.word[k - k0][t];
    while (k < to) {
        const uint32_t o01 = uni(nx.o01), o23 = uni(nx.o23), g = uni(nx.g), bits = uni(nx.bits);
        const uint32_t a = word & 0x7fffu, pc = word >> 15;
        const uint32_t off[4] = {o01 & 0xffffu, o01 >> 16, o23 & 0xffffu, o23 >> 16};
        const int i = k - k0, m = int(bits >> 5) & 3;
        const bool on = uint32_t(t) < (1u << (bits >> 16));
        double2 A[2][2];
        if (on) slot_sums_of<S>(int(bits & 31), tab, a, off, pc, (bits >> 8) & 15, A);
        else A[0][0] = A[0][1] = A[1][0] = A[1][1] = make_double2(0, 0);
        if (k + 1 < to) {
            nx = sh.n[i + 1];
            word = sh.word[i + 1][t];
        }
        const SStep& s = sh.s[i];
        const double2 M[2][2] = {{make_double2(s.mre[0][0], s.mim[0][0]), make_double2(s.mre[0][1], s.mim[0][1])},
                                 {make_double2(s.mre[1][0], s.mim[1][0]), make_double2(s.mre[1][1], s.mim[1][1])}};
        int bv = forced ? int(sh.forced[i]) : -1;
        double u = MODE == kChain ? sh.U[i] : MODE == kRun ? sh.U[st.qidx] : 0;
        double cf[2][4];
        if constexpr (MODE != kChain1) {
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int j = 0; j < 4; j++) cf[b][j] = sh.coef[i][b][j];
        }
        bv = __builtin_amdgcn_readfirstlane(bv);
        const bool growth = (bits >> 12) & 1;
        double sc = 1.0;
        if constexpr (MODE == kRun) sc = 1.0 / sqrt(st.prev);
        if (MODE == kChain || (MODE == kRun && bv < 0)) {
            double n2[2];
            if (growth) {
#pragma unroll
                for (int b = 0; b < 2; b++) n2[b] = (cf[b][0] + cf[b][1]) * st.nstored;
            } else if (MODE == kChain && forced) {
                double acc[4] = {0, 0, 0, 0};
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    if (q >= m) break;
                    add_norm(acc[0], cfma(M[0][0], A[q][0], cmul(M[0][1], A[q][1])));
                    add_norm(acc[1], cfma(M[1][0], A[q][0], cmul(M[1][1], A[q][1])));
                }
                const double r = sum2(acc);
                n2[0] = lane_value(r, 0);
                n2[1] = lane_value(r, 32);
            } else {
                double acc[4] = {0, 0, 0, 0};
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    if (q >= m) break;
                    const double2 x = A[q][0], y = A[q][1];
                    add_norm(acc[0], x);
                    add_norm(acc[1], y);
                    acc[2] = fma(x.x, y.x, fma(x.y, y.y, acc[2]));
                    acc[3] = fma(x.y, y.x, fma(-x.x, y.y, acc[3]));
                }
                const double r = sum4(acc);
                const double r0 = lane_value(r, 0), r1 = lane_value(r, 32), r2 = lane_value(r, 16), r3 = lane_value(r, 48);
#pragma unroll
                for (int b = 0; b < 2; b++) n2[b] = cf[b][0] * r0 + cf[b][1] * r1 + 2 * (cf[b][2] * r2 - cf[b][3] * r3);
            }
            double p1 = n2[1] / (n2[0] + n2[1]);
            if constexpr (MODE == kChain) {
                double both = 1.0 / sqrt((t & 1) ? n2[1] : n2[0]);   // lane 0: branch 0, lane 1: branch 1
                here(both);
                here(p1);
                if (bv < 0) bv = __builtin_amdgcn_readfirstlane(int(u < p1));
                const double pb = bv ? p1 : 1 - p1;
                if (__builtin_amdgcn_readfirstlane(int(pb <= 0))) {
                    st.neglog = true;
                    st.dead = 1;
                    return k;
                }
                if (t == 0) sh.pfac[st.np] = pb;
                st.np++;
                sc = lane_value(both, bv);
            } else {
                bv = __builtin_amdgcn_readfirstlane(int(u < p1));
                st.qidx++;
            }
        }
        if (t == 0) sh.bits[i] = int8_t(bv);
        st.bv = bv;
        st.sc = sc;
        const double2 m0 = bv ? M[1][0] : M[0][0], m1 = bv ? M[1][1] : M[0][1];
        st.w0 = make_double2(m0.x * sc, m0.y * sc);
        st.w1 = make_double2(m1.x * sc, m1.y * sc);
        double acc[4] = {0, 0, 0, 0};
        if (on) {
#pragma unroll
            for (int q = 0; q < 2; q++) {
                if (q >= m) break;
                const double2 v = cfma(st.w0, A[q][0], cmul(st.w1, A[q][1]));
                const S sv = Cx<S>::narrow(v);
                tab[q ? a ^ g : a] = sv;
                add_norm(acc[0], v);
                add_norm(acc[1], Cx<S>::widen(sv));
            }
        }
        wave_fence();
        k++;
        const bool stored = MODE != kChain1 && ((bits >> 13) & 1);
        if (MODE == kChain && !stored) continue;
        double nb;
        if (stored) {
            const double r = sum2(acc);
            nb = lane_value(r, 0);
            st.nstored = lane_value(r, 32);
        } else {
            nb = wave_sum(acc[0]);
        }
        if constexpr (MODE == kChain1) {                       // gsamp2.cpp:67
            if (t == 0) sh.cond[i] = nb / (2 * st.prev);
            st.prev = nb;
        } else if constexpr (MODE == kRun) {                   // gsamp2.cpp:93-95
            const double cd = nb / 2;
            if (t == 0) {
                sh.sfac[st.nsf] = st.prev;
                sh.cond[i] = cd;
                sh.pfac[st.np] = cd;
            }
            st.nsf++;
            st.prev = nb;
            if (!__builtin_amdgcn_readfirstlane(int(nb <= 0))) st.np++;
        }
        if (MODE != kChain && __builtin_amdgcn_readfirstlane(int(nb <= 0))) {
            st.dead = 1;
            st.neglog = true;
            return k - 1;
        }
    }
    return k;
}

// Steps k0 .. k1-1 of one chain, one block per string.  start: the chain begins here (table 1, fresh state); decided0:
// step k0's decision was already made (by the previous write's fused norms).
template <class S>
__global__ __launch_bounds__(kSmallThreads) void small_run_kernel(const SStep* __restrict__ steps,
                                                                  const KStep* __restrict__ plain, S* __restrict__ mem,
                                                                  Ctl* __restrict__ ctl, Epi epi, int k0, int k1,
                                                                  int decided0, int start, int tab_bytes) {
    extern __shared__ __align__(16) unsigned char lds[];
    S* tab = reinterpret_cast<S*>(lds);
    Shared& sh = *reinterpret_cast<Shared*>(lds + tab_bytes);
    const Epi e = slot_epi(epi);
    mem += uint64_t(blockIdx.y) * epi.slot_entries;
    ctl += blockIdx.y;
    const int t = threadIdx.x, steps_n = k1 - k0;
    State st{};
    st.prev = st.nstored = 1;
    double logp0 = 0, logscale0 = 0;
    if (!start) {
        const Ctl c = *ctl;
        if (c.dead) return;
        st.prev = c.prev;
        st.nstored = c.nstored;
        st.w0 = make_double2(c.w[0], c.w[1]);
        st.w1 = make_double2(c.w[2], c.w[3]);
        st.sc = c.sc;
        st.bv = c.bv;
        st.qidx = c.qidx;
        logp0 = c.logp;
        logscale0 = c.logscale;
    }
    const int q0 = st.qidx;                                    // kRun draws one uniform per sampled step
    {
        const uint32_t* from = reinterpret_cast<const uint32_t*>(steps + k0);
        uint32_t* to = reinterpret_cast<uint32_t*>(sh.s);
        for (int i = t; i < steps_n * int(sizeof(SStep) / 4); i += kSmallThreads) to[i] = from[i];
        if (t < steps_n) {
            if (e.forced) sh.forced[t] = e.forced[k0 + t];
            if (t == 0) sh.bits[0] = int8_t(st.bv);            // a step decided before the run keeps its bit
            if (!e.forced || e.mode == kRun) sh.U[t] = e.U[(e.mode == kRun ? q0 : k0) + t];
        }
    }
    st.qidx = 0;
    if (start && t == 0) tab[0] = Cx<S>::narrow(make_double2(1.0, 0.0));
    __syncthreads();
    for (int i = t >> 6; i < steps_n; i += kWavesS) {
        const SStep& s = sh.s[i];
        if (s.nk > 6) continue;
        const int lane = t & 63;
        uint32_t a = 0;
#pragma unroll
        for (int j = 0; j < 6; j++) a ^= ((lane >> j) & 1) ? s.cols[j] : 0;
        sh.word[i][lane] = uint16_t(a | (uint32_t(__popc(uint32_t(lane) & s.rho)) & 1) << 15);
        if (lane < 2) {
            const double2 m0 = make_double2(s.mre[lane][0], s.mim[lane][0]), m1 = make_double2(s.mre[lane][1], s.mim[lane][1]);
            sh.coef[i][lane][0] = norm2(m0);
            sh.coef[i][lane][1] = norm2(m1);
            sh.coef[i][lane][2] = m0.x * m1.x + m0.y * m1.y;   // m0 conj(m1)
            sh.coef[i][lane][3] = m0.y * m1.x - m0.x * m1.y;
        }
        if (lane == 0) {
            const uint32_t next = i + 1 < steps_n ? uint32_t(sh.s[i + 1].growth != 0) : 1u;
            sh.n[i] = NStep{s.off[0] | s.off[1] << 16, s.off[2] | s.off[3] << 16, s.g,
                            uint32_t(s.kind) | uint32_t(s.m) << 5 | s.par << 8 | uint32_t(s.growth != 0) << 12 | next << 13 |
                                uint32_t(s.nk) << 16};
        }
    }
    __syncthreads();
    if (!start) {
        const SStep& s = sh.s[0];
        const KStep& p = plain[k0];
        for (int i = t; i < (s.ntq << s.nk); i += kSmallThreads) {     // the live slots of step k0
            const int c = i & ((1 << s.nk) - 1), j = i >> s.nk;
            uint64_t pa = p.off[j];
            uint32_t a = s.off[j];
            for (int b = 0; b < s.nk; b++)
                if ((c >> b) & 1) {
                    pa ^= p.cols[b];
                    a ^= s.cols[b];
                }
            tab[a] = mem[pa];
        }
        __syncthreads();
    }
    int k = k0;
    bool decided = decided0 != 0;
    while (k < k1 && !st.dead) {
        if (sh.s[k - k0].nk > 6) {
            small_step<S, true>(sh, tab, mem, plain, e, st, k, k0, decided, k + 1 == k1);
            decided = false;
            if (!st.dead) k++;
            continue;
        }
        int to = k;                                            // steps of one wave
        while (to < k1 && sh.s[to - k0].nk <= 6) to++;
        if (t < 64) {
            while (k < to && !st.dead) {
                const int stop = to == k1 ? k1 - 1 : to;       // the run's last step writes to the arena
                if (decided || k >= stop) {
                    small_step<S, false>(sh, tab, mem, plain, e, st, k, k0, decided, k + 1 == k1);
                    decided = false;
                    if (!st.dead) k++;
                } else if (e.mode == kChain) {
                    k = narrow_steps<S, kChain>(sh, tab, e.forced != nullptr, st, k, k0, stop);
                } else if (e.mode == kChain1) {
                    k = narrow_steps<S, kChain1>(sh, tab, true, st, k, k0, stop);
                } else {
                    k = narrow_steps<S, kRun>(sh, tab, e.forced != nullptr, st, k, k0, stop);
                }
            }
            if (t == 0) {
                Ctl c{};
                c.prev = st.prev;
                c.nstored = st.nstored;
                c.qidx = st.qidx;
                c.dead = st.dead;
                c.bv = st.bv;
                c.sc = st.sc;
                c.w[0] = st.w0.x; c.w[1] = st.w0.y; c.w[2] = st.w1.x; c.w[3] = st.w1.y;
                sh.c = c;
                sh.np = st.np;
                sh.nsf = st.nsf;
                sh.kdone = k;
            }
        }
        __syncthreads();
        if (t >= 64) {
            st.prev = sh.c.prev;
            st.nstored = sh.c.nstored;
            st.qidx = sh.c.qidx;
            st.dead = sh.c.dead;
            st.np = sh.np;
            st.nsf = sh.nsf;
            k = sh.kdone;
        }
        decided = false;
    }
    __syncthreads();
    // k = the step that met a zero branch, or k1.  log2 of every factor, then their sum in step order.
    if (t < st.np) sh.plog[t] = log2(sh.pfac[t]);
    if (t >= 64 && t - 64 < st.nsf) sh.slog[t - 64] = log2(sh.sfac[t - 64]);
    __syncthreads();
    if (t < k - k0) {
        e.bits[k0 + t] = sh.bits[t];
        if (e.mode != kChain) e.cond[k0 + t] = sh.cond[t];
    }
    // a zero branch leaves zero conditionals (and a run's remaining bits as forced, or 0) from its step on; in chain mode
    // the string ends where it is
    if (st.dead && e.mode != kChain) {
        const int end = e.mode == kChain1 ? e.ns : e.k1;
        for (int q = k + t; q < end; q += kSmallThreads) {
            e.cond[q] = 0;
            if (e.mode == kRun) e.bits[q] = e.forced[q] < 0 ? 0 : e.forced[q];
        }
    }
    if (t != 0) return;
    Ctl c{};
    c.logp = logp0;
    for (int i = 0; i < st.np; i++) c.logp += sh.plog[i];
    c.logscale = logscale0;
    for (int i = 0; i < st.nsf; i++) c.logscale += 0.5 * sh.slog[i];
    if (st.neglog) c.logp = -INFINITY;
    c.prev = st.prev;
    c.nstored = st.nstored;
    c.sc = st.sc;
    c.w[0] = st.w0.x; c.w[1] = st.w0.y; c.w[2] = st.w1.x; c.w[3] = st.w1.y;
    c.bv = st.bv;
    c.dead = st.dead;
    c.qidx = q0 + st.qidx;
    if (c.dead || k1 == e.k1) {
        if (e.mode == kChain1 && !c.dead) c.logp = log2(c.prev) - e.ns;
        e.out[0] = c.logp;
        e.out[1] = c.logscale;
        e.out[2] = c.prev;
        e.out[3] = c.dead;
    }
    *ctl = c;
}

}  // namespace

size_t small_run_lds(size_t tab_bytes) { return tab_bytes + sizeof(Shared); }
void* small_run_kernel_ptr(int storage) {
    return storage == 0 ? reinterpret_cast<void*>(&small_run_kernel<float2>)
                        : reinterpret_cast<void*>(&small_run_kernel<double2>);
}

}  // namespace gs
