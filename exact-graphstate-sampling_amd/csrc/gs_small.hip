// Runs of small steps in one block per string.
//
// The head and tail of a plan are steps of a few thousand cosets and less, where a sweep costs far less than a launch;
// one block runs such a run step after step -- norm pass, decision, write pass, bookkeeping -- with the run's table in
// LDS: the arena slots a run touches span a subspace of at most 2^kSmallTab entries, and the host gives every step's
// columns, offsets and g as indices into that subspace.  The arithmetic per coset is the sweep kernels' (FP64 routed slot
// sums, one rounding per store), the chain logic theirs too (gsamp2.cpp:46-49, :67, :80-95).
//
// What bounds it is latency: a step has little to compute and two sums over the cosets that the next pass needs.  So
// the chain state lives in registers of every thread (each makes the decision itself, no broadcast), sums go through
// DPP inside a wave and one barrier across waves, steps of at most 64 cosets run on the first wave with no barrier at
// all, every descriptor, bit and uniform is in LDS before the first step, and the logarithms, which no decision needs,
// are taken for all steps at once at the end.  A version with the table in the arena, state changes by one thread and
// two barriers per pass took 4.6 us per step; this one takes 2.0 us
// (the n = 24 plan, 24 steps, complex64: 115 -> 49.5 us).
#include "gs_math.h"
#include "gs_wave.h"

namespace gs {

namespace {

constexpr int kWavesS = kSmallThreads / 64;

struct Shared {                       // after the table in LDS
    SStep s[kSmallSteps];
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

// Sums of a pass over the threads that run it, in every one of them.
template <bool WIDE, int NQ>
__device__ __forceinline__ void pass_sum(Shared& sh, int& buf, const double (&v)[4], double (&out)[4]) {
    double r[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) r[q] = wave_sum(v[q]);
    if constexpr (WIDE) {
        const int wave = threadIdx.x >> 6;
        if ((threadIdx.x & 63) == 0)
#pragma unroll
            for (int q = 0; q < NQ; q++) sh.sum[buf][wave][q] = r[q];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            double x = sh.sum[buf][0][q];
#pragma unroll
            for (int w = 1; w < kWavesS; w++) x += sh.sum[buf][w][q];
            r[q] = x;
        }
        buf ^= 1;
    }
#pragma unroll
    for (int q = 0; q < NQ; q++) out[q] = r[q];
}

// One step on one wave (at most 64 cosets) or on the whole block.  last: the run's last step, whose outputs go to the
// arena.
template <class S, bool WIDE>
__device__ __forceinline__ void small_step(Shared& sh, S* tab, S* mem, const KStep* plain, const Epi& e, State& st, int k,
                                           int k0, bool decided, bool last) {
    const SStep& s = sh.s[k - k0];
    const int t = threadIdx.x;
    constexpr int T = WIDE ? kSmallThreads : 64;
    constexpr int LT = WIDE ? 9 : 6;
    const int nk = __builtin_amdgcn_readfirstlane(s.nk), ntq = __builtin_amdgcn_readfirstlane(s.ntq);
    const int m = __builtin_amdgcn_readfirstlane(s.m);
    const uint32_t route = __builtin_amdgcn_readfirstlane(int(s.route));   // t0 | t1 << 4 | par << 8, a bit per offset
    const uint32_t rho = s.rho, g = s.g;
    uint32_t off[4];
#pragma unroll
    for (int j = 0; j < 4; j++) off[j] = s.off[j];
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
    // index of coset c (c = t mod T) and its routed slot sums
    auto index_of = [&](uint32_t c) {
        uint32_t a = bt;
        if constexpr (WIDE)
#pragma unroll
            for (int j = LT; j < kSmallMaxNk; j++) a ^= ((c >> j) & 1) ? s.cols[j] : 0;
        return a;
    };
    auto sums = [&](uint32_t a, uint32_t c, double2 (&A)[2][2]) {
        S v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = tab[a ^ off[j]];    // offsets beyond ntq repeat the first
        const uint32_t pc = __popc(c & rho) & 1;
        A[0][0] = A[0][1] = A[1][0] = A[1][1] = make_double2(-0.0, -0.0);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (j >= ntq) break;
            const double2 w = Cx<S>::widen(v[j]);
            const int neg = int((pc ^ (route >> (8 + j))) << 31);
            const double2 ws = make_double2(__hiloint2double(__double2hiint(w.x) ^ neg, __double2loint(w.x)),
                                            __hiloint2double(__double2hiint(w.y) ^ neg, __double2loint(w.y)));
            if ((route >> j) & 1) A[1][0] = cadd(A[1][0], w); else A[0][0] = cadd(A[0][0], w);       // uniform branches
            if ((route >> (4 + j)) & 1) A[1][1] = cadd(A[1][1], ws); else A[0][1] = cadd(A[0][1], ws);
        }
    };
    // Norms the decision needs: none when it is forced or made without them (chain1, forced hybrid steps) or follows
    // from the stored norm (growth steps), direct branch norms for a forced string, else the Gram matrix.
    if (!decided) {
        int bv = e.forced ? int(sh.forced[k - k0]) : -1;
        const bool need_p = e.mode == kChain || (e.mode == kRun && bv < 0);
        const int growth = __builtin_amdgcn_readfirstlane(s.growth);
        double n2[2] = {0, 0};
        if (need_p && growth) {
#pragma unroll
            for (int b = 0; b < 2; b++) n2[b] = (norm2(M[b][0]) + norm2(M[b][1])) * st.nstored;
        } else if (need_p) {
            double acc[4] = {0, 0, 0, 0}, red[4];
            const bool direct = e.mode == kChain && e.forced;
            for (uint32_t c = t; c < n; c += T) {
                double2 A[2][2];
                sums(index_of(c), c, A);
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
            pass_sum<WIDE, 4>(sh, st.buf, acc, red);
#pragma unroll
            for (int b = 0; b < 2; b++) {
                const double2 m0 = M[b][0], m1 = M[b][1];
                const double pr = m0.x * m1.x + m0.y * m1.y, pi = m0.y * m1.x - m0.x * m1.y;   // m0 conj(m1)
                n2[b] = direct ? red[b] : norm2(m0) * red[0] + norm2(m1) * red[1] + 2 * (pr * red[2] - pi * red[3]);
            }
        }
        double sc = 1.0;
        if (e.mode == kChain) {
            const double p1 = n2[1] / (n2[0] + n2[1]);
            if (bv < 0) bv = sh.U[k - k0] < p1;
            const double pb = bv ? p1 : 1 - p1;
            if (pb <= 0) {
                st.neglog = true;
                st.dead = 1;
                return;
            }
            if (t == 0) sh.pfac[st.np] = pb;
            st.np++;
            sc = 1.0 / sqrt(bv ? n2[1] : n2[0]);
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
        double2 A[2][2];
        const uint32_t a = index_of(c);
        sums(a, c, A);
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
    pass_sum<WIDE, 2>(sh, st.buf, acc, red);
    st.nstored = red[1];
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
    if (start) {
        if (t == 0) tab[0] = Cx<S>::narrow(make_double2(1.0, 0.0));
        __syncthreads();
    } else {
        __syncthreads();
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
            for (; k < to && !st.dead;) {
                small_step<S, false>(sh, tab, mem, plain, e, st, k, k0, decided, k + 1 == k1);
                decided = false;
                if (!st.dead) k++;
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
