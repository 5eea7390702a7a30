// The other kernels of the engines: reductions after a sweep, one-thread chain kernels, runs of diagonal steps; and the
// table of all of them the engines launch from.
#include "gs_sweep.h"

namespace gs {

void* sweep_kernel_c64(int lr, int vg, int ntq, int route, int sweep, int route2);
void* sweep_kernel_c128(int lr, int vg, int ntq, int route, int sweep, int route2);

// Reduction and chain logic of a sweep whose blocks left their partials (one block per string, launched after the
// sweep).
template <int NQ>
__global__ __launch_bounds__(kThreads) void sweep_reduce_kernel(const double* __restrict__ part, unsigned nblk,
                                                                Ctl* __restrict__ ctl, Epi e, int sweep) {
    ctl += blockIdx.y;
    part += size_t(blockIdx.y) * e.slot_part;
    if (ctl->dead) return;
    __shared__ double sh[kThreads / 64][NQ];
    const int t = threadIdx.x;
    reduce_partials<NQ>(sh, part, nblk, t, false);
    if (t != 0) return;
    double red[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) red[q] = sh[0][q];
    chain_step<NQ, true>(red, ctl, slot_epi(e), sweep);
}

// The same for many blocks, in the same order: thread t of the one-block kernel sums partials t, t + 256, ...; here a
// wave does that for one quantity and 64 of the t, and the last of the 4 NQ waves adds up and runs the chain.  One block
// reads the 64-byte partials of 2^14 blocks in 28.7 us, bound by the loads one CU has in flight; the waves in 10.2 us.
template <int NQ>
__global__ __launch_bounds__(64) void wide_reduce_kernel(double* __restrict__ part, unsigned nblk, Ctl* __restrict__ ctl,
                                                         Epi e, int sweep) {
    constexpr int NW = kThreads / 64, U = 16;
    ctl += blockIdx.y;
    part += size_t(blockIdx.y) * e.slot_part;
    if (ctl->dead) return;
    const int lane = threadIdx.x, q = int(blockIdx.x) % NQ, w = int(blockIdx.x) / NQ;
    double r = 0;
    for (unsigned i = unsigned(w * 64 + lane); i < nblk; i += U * kThreads) {
        double v[U];
#pragma unroll
        for (int u = 0; u < U; u++)
            v[u] = part[size_t(min(i + unsigned(u) * kThreads, nblk - 1)) * kPartStride + q];
#pragma unroll
        for (int u = 0; u < U; u++)
            if (i + unsigned(u) * kThreads < nblk) r += v[u];
    }
    for (int o = 32; o > 0; o >>= 1) r += __shfl_xor(r, o, 64);
    // the wave's sum in the last, unused double of partial w * NQ + q; published before the counter is raised
    auto slot = [&](int i) { return reinterpret_cast<unsigned long long*>(part + size_t(i) * kPartStride + kPartStride - 1); };
    int last = 0;
    if (lane == 0) {
        unsigned long long old = __hip_atomic_exchange(slot(w * NQ + q), (unsigned long long)__double_as_longlong(r),
                                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" : "+v"(old) : : "memory");
        last = __hip_atomic_fetch_add(e.counter + blockIdx.y, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
               unsigned(NW * NQ - 1);
    }
    if (!__shfl(last, 0, 64)) return;
    __atomic_thread_fence(__ATOMIC_ACQUIRE);
    double v = 0;
    if (lane < NW * NQ)
        v = __longlong_as_double((long long)__hip_atomic_load(slot(lane), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    double red[NQ];
#pragma unroll
    for (int k = 0; k < NQ; k++) {
        red[k] = __shfl(v, k, 64);
#pragma unroll
        for (int j = 1; j < NW; j++) red[k] += __shfl(v, j * NQ + k, 64);
    }
    if (lane != 0) return;
    chain_step<NQ, true>(red, ctl, slot_epi(e), sweep);
    __hip_atomic_store(e.counter + blockIdx.y, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------------------------------------------------------
// single-thread chain kernels

__global__ void decide_kernel(Ctl* ctl, Epi e, int k) {
    Ctl& c = ctl[blockIdx.y];
    if (!c.dead) decide(c, slot_epi(e), k, -1, nullptr);
}

__global__ void publish_kernel(Ctl* ctl, Epi e) { publish(ctl[blockIdx.y], slot_epi(e)); }

// ---------------------------------------------------------------------------------------------------------------
// Runs of diagonal steps (RStep).  Pass 1 sums |v|^2 of the run's table per sign pattern sigma, pass 2 multiplies every
// entry by the product factor of its pattern; between them one block reduces the sums and makes the run's j decisions
// with the chain functions above, from the exact norms of each step's two branches:
//   n_b(step i) = sum_sigma H[sigma] |F_{i-1}(sigma)|^2 |M_b0 + (-1)^{sigma_i} M_b1|^2,
//   F_i(sigma) = F_{i-1}(sigma) (w0_i + (-1)^{sigma_i} w1_i),  (w0, w1) = the decided row of M_i times the step's scale,
// which is what the per-step sweeps compute one step at a time (the values are rounded to the storage type once per
// run instead of once per step).  All sums are in a fixed order: results are bitwise reproducible.

// Thread and block parts of a run pass: base address and sigma of the thread's coordinate origin.
__device__ __forceinline__ void run_origin(const RStep& r, uint64_t& a, int& sg, bool& active) {
    const int tid = threadIdx.x;
    a = 0;
    sg = r.kappa;
#pragma unroll
    for (int b = 0; b < 8; b++)
        if ((tid >> b) & 1) {
            a ^= r.cols[1 + b];
            sg ^= r.sig[1 + b];
        }
    active = r.nk >= 9 || (uint64_t(tid) << 1) < (uint64_t(1) << r.nk);
    const unsigned bid = r.xcd && r.lg_grid >= 3 ? (blockIdx.x >> 3) | ((blockIdx.x & 7u) << (r.lg_grid - 3))
                                                 : blockIdx.x;
    for (int b = 0; b < r.lg_grid; b++)
        if ((bid >> b) & 1) {
            a ^= r.cols[9 + b];
            sg ^= r.sig[9 + b];
        }
}

// Pass 1: per block, the sum of |v|^2 per pattern (2^j bins; threads own bins and scan the block's values in a fixed
// order) into hpart[block][kRunBins].
template <class S>
__global__ __launch_bounds__(kThreads) void run_hist_kernel(const RStep* __restrict__ rp, const S* __restrict__ mem,
                                                           double* __restrict__ hpart, const Ctl* __restrict__ ctl) {
    if (ctl->dead) return;
    const RStep& r = *rp;
    uint64_t a_tb;
    int sg;
    bool active;
    run_origin(r, a_tb, sg, active);
    const int jit = 9 + r.lg_grid;
    const int niter = 1 << r.lg_iter;
    __shared__ double sw[4 * kThreads];
    __shared__ int ss[4 * kThreads];
    const int t = threadIdx.x;
    int nv = 2;                                     // values per thread
    if (r.pair) {
        // tile pairs (a, a ^ gc): the pairing coordinate may change sigma, so the second tile's values go to their
        // own two patterns
        const uint64_t gc = r.cols[jit];
        const int sgp = r.sig[jit];
        double acc[4] = {0, 0, 0, 0};
        uint64_t a_it = 0;
        for (int i = 0; i < (niter >> 1); i++) {
            if (i > 0) a_it ^= r.cols[jit + 1 + __builtin_ctz(unsigned(i))];
            if (!active) continue;
            S e[2], h[2];
            Run<S, 2>::load(mem, a_tb ^ a_it, e);
            Run<S, 2>::load(mem, a_tb ^ a_it ^ gc, h);
            add_norm(acc[0], Cx<S>::widen(e[0]));
            add_norm(acc[1], Cx<S>::widen(e[1]));
            add_norm(acc[2], Cx<S>::widen(h[0]));
            add_norm(acc[3], Cx<S>::widen(h[1]));
        }
        for (int q = 0; q < 4; q++) {
            sw[4 * t + q] = acc[q];
            ss[4 * t + q] = sg ^ ((q & 1) ? r.sig[0] : 0) ^ ((q & 2) ? sgp : 0);
        }
        nv = 4;
    } else {
        double acc0 = 0, acc1 = 0;
        uint64_t a_it = 0;
        for (int it = 0; it < niter; it++) {
            if (it > 0) a_it ^= r.cols[jit + __builtin_ctz(unsigned(it))];
            if (!active) continue;
            S e[2];
            Run<S, 2>::load(mem, a_tb ^ a_it, e);
            add_norm(acc0, Cx<S>::widen(e[0]));
            add_norm(acc1, Cx<S>::widen(e[1]));
        }
        sw[2 * t] = acc0;
        sw[2 * t + 1] = acc1;
        ss[2 * t] = sg;
        ss[2 * t + 1] = sg ^ r.sig[0];
    }
    __syncthreads();
    double h = 0;
    for (int q = 0; q < nv * kThreads; q++)
        if (ss[q] == t) h += sw[q];
    hpart[size_t(blockIdx.x) * kRunBins + t] = h;
}

// First stage of the reduction: chunk g sums the pattern sums of blocks [g nblk / G, (g + 1) nblk / G) in order.
__global__ __launch_bounds__(kRunBins) void run_chunk_kernel(const double* __restrict__ hpart, unsigned nblk,
                                                            double* __restrict__ chunk, const Ctl* __restrict__ ctl) {
    if (ctl->dead) return;
    const unsigned G = gridDim.x, g = blockIdx.x, t = threadIdx.x;
    const unsigned b0 = unsigned((uint64_t(g) * nblk) / G), b1 = unsigned((uint64_t(g + 1) * nblk) / G);
    double h = 0;
    for (unsigned b = b0; b < b1; b++) h += hpart[size_t(b) * kRunBins + t];
    chunk[size_t(g) * kRunBins + t] = h;
}

// The run's decisions and bookkeeping (one block of kRunBins threads, thread t = pattern t), then the product factors
// F_j(sigma) for pass 2.  Each step: the branch norms by a fixed-order block sum, decide() (forced bit, or U < p1),
// the written norm nb, finish_write(); the stored norm of pass 2 replaces nb as the growth-step norm afterwards.
__global__ __launch_bounds__(kRunBins) void run_decide_kernel(const RStep* __restrict__ rp,
                                                             const double* __restrict__ chunk, unsigned G,
                                                             Ctl* __restrict__ ctl, Epi e, double2* __restrict__ fac) {
    Ctl& c = *ctl;
    if (c.dead) return;
    const RStep& r = *rp;
    const int t = threadIdx.x;
    __shared__ double sh[kRunBins / 64][2];
    __shared__ int s_dead;
    double H = 0;
    for (unsigned g = 0; g < G; g++) H += chunk[size_t(g) * kRunBins + t];
    double2 F = make_double2(1.0, 0.0);
    double W = H;                                              // H |F|^2
    if (t == 0) s_dead = 0;
    for (int i = 0; i < r.j; i++) {
        const int k = r.k0 + i;
        const int s = (t >> i) & 1;
        double nb2[2];
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const double2 m0 = make_double2(r.mre[i][b][0], r.mim[i][b][0]);
            const double2 m1 = make_double2(r.mre[i][b][1], r.mim[i][b][1]);
            nb2[b] = W * norm2(cadd(m0, negate_if(m1, s)));
        }
        block_tree_sum<2, kRunBins>(sh, nb2, t);
        if (t == 0) {
            const double red[2] = {sh[0][0], sh[0][1]};
            decide(c, e, k, kDirect, red);
            s_dead = c.dead;
        }
        __syncthreads();
        if (s_dead) return;
        const double2 w0 = make_double2(c.w[0], c.w[1]), w1 = make_double2(c.w[2], c.w[3]);
        F = cmul(F, cadd(w0, negate_if(w1, s)));
        W = H * norm2(F);
        const double one[2] = {W, 0.0};
        block_tree_sum<2, kRunBins>(sh, one, t);
        if (t == 0) {
            finish_write(c, e, k, sh[0][0], sh[0][0]);
            if (!c.dead && k + 1 == e.k1) publish(c, e);
            s_dead = c.dead;
        }
        __syncthreads();
        if (s_dead) return;
    }
    fac[t] = F;
}

// Next-step slot index (bit 0) and sign (bit 1) parities of coordinate c of a paired run.
__device__ __forceinline__ int run_pn(const RStep& r, int c) {
    return int((r.phim >> c) & 1) | (int((r.num >> c) & 1) << 1);
}

// Pass 2: every entry times its pattern's factor (FP64, one rounding), in place; the stored table's norm goes to the
// chain state (role kRoleStored).  GRAM (paired runs): the pass also sums the next step's Gram matrix from the values
// it stores -- run element e at address a pairs with element e ^ peps at a ^ gc, the two slots of one next-step coset
// -- and the chain decides that step (role kRoleStoredGram).
template <class S, bool GRAM, int ROUTE2>
__global__ __launch_bounds__(kThreads) void run_apply_kernel(const RStep* __restrict__ rp, S* __restrict__ mem,
                                                            const double2* __restrict__ fac, double* __restrict__ part,
                                                            Ctl* __restrict__ ctl, Epi epi) {
    constexpr int NA = GRAM ? 5 : 1;
    if (ctl->dead) return;
    const RStep& r = *rp;
    uint64_t a_tb;
    int sg;
    bool active;
    run_origin(r, a_tb, sg, active);
    const double2 f0 = fac[sg], f1 = fac[sg ^ r.sig[0]];
    const int jit = 9 + r.lg_grid;
    const int niter = 1 << r.lg_iter;
    double acc[NA];
#pragma unroll
    for (int q = 0; q < NA; q++) acc[q] = 0;
    if (GRAM || r.pair) {
        const uint64_t gc = r.cols[jit];
        const int sgp = r.sig[jit];
        const double2 g0 = fac[sg ^ sgp], g1 = fac[sg ^ sgp ^ r.sig[0]];
        int pn_tb = 0;                              // next-step parities of the thread's and block's coordinates
        if constexpr (GRAM) {
            const int tid = threadIdx.x;
#pragma unroll
            for (int b = 0; b < 8; b++)
                if ((tid >> b) & 1) pn_tb ^= run_pn(r, 1 + b);
            const unsigned bid = r.xcd && r.lg_grid >= 3 ? (blockIdx.x >> 3) | ((blockIdx.x & 7u) << (r.lg_grid - 3))
                                                         : blockIdx.x;
            for (int b = 0; b < r.lg_grid; b++)
                if ((bid >> b) & 1) pn_tb ^= run_pn(r, 9 + b);
        }
        const int pn0 = run_pn(r, 0), peps = r.peps;
        double gi[kgCount];
#pragma unroll
        for (int q = 0; q < kgCount; q++) gi[q] = 0;
        uint64_t a_it = 0;
        int pn_it = 0;
        for (int i = 0; i < (niter >> 1); i++) {
            if (i > 0) {
                const int c = jit + 1 + __builtin_ctz(unsigned(i));
                a_it ^= r.cols[c];
                if constexpr (GRAM) pn_it ^= run_pn(r, c);
            }
            if (!active) continue;
            const uint64_t a = a_tb ^ a_it, b = a ^ gc;
            S e[2], h[2];
            Run<S, 2>::load(mem, a, e);
            Run<S, 2>::load(mem, b, h);
            e[0] = Cx<S>::narrow(cmul(Cx<S>::widen(e[0]), f0));
            e[1] = Cx<S>::narrow(cmul(Cx<S>::widen(e[1]), f1));
            h[0] = Cx<S>::narrow(cmul(Cx<S>::widen(h[0]), g0));
            h[1] = Cx<S>::narrow(cmul(Cx<S>::widen(h[1]), g1));
            Run<S, 2>::store(mem, a, e);
            Run<S, 2>::store(mem, b, h);
            add_norm(acc[0], Cx<S>::widen(e[0]));
            add_norm(acc[0], Cx<S>::widen(e[1]));
            add_norm(acc[0], Cx<S>::widen(h[0]));
            add_norm(acc[0], Cx<S>::widen(h[1]));
            if constexpr (GRAM) {
#pragma unroll
                for (int el = 0; el < 2; el++) {
                    const int pe = pn_tb ^ pn_it ^ (el ? pn0 : 0);      // parities of element el's address
                    const S vb = (el ^ peps) ? h[1] : h[0];
                    gram_invariants<ROUTE2>(Cx<S>::widen(e[el]), Cx<S>::widen(vb), uint32_t(pe & 1),
                                            uint32_t((pe >> 1) & 1), gi);
                }
            }
        }
        if constexpr (GRAM) gram_assemble<ROUTE2>(gi, r.par2, acc + 1);
        sweep_epilogue<NA>(acc, part, ctl, epi, kWrite);
        return;
    }
    uint64_t a_it = 0;
    for (int it = 0; it < niter; it++) {
        if (it > 0) a_it ^= r.cols[jit + __builtin_ctz(unsigned(it))];
        if (!active) continue;
        const uint64_t a = a_tb ^ a_it;
        S e[2];
        Run<S, 2>::load(mem, a, e);
        e[0] = Cx<S>::narrow(cmul(Cx<S>::widen(e[0]), f0));
        e[1] = Cx<S>::narrow(cmul(Cx<S>::widen(e[1]), f1));
        Run<S, 2>::store(mem, a, e);
        add_norm(acc[0], Cx<S>::widen(e[0]));
        add_norm(acc[0], Cx<S>::widen(e[1]));
    }
    sweep_epilogue<NA>(acc, part, ctl, epi, kWrite);
}

// ---------------------------------------------------------------------------------------------------------------
// dispatch table

// Kernel for (storage 0 = c64 / 1 = c128, log2 run, vg, ntq, route, sweep, next route); nullptr when not built.
void* sweep_kernel_for(int storage, int lr, int vg, int ntq, int route, int sweep, int route2) {
    return storage == 0 ? sweep_kernel_c64(lr, vg, ntq, route, sweep, route2)
                        : sweep_kernel_c128(lr, vg, ntq, route, sweep, route2);
}

// log2 run length of the plain layout per storage, and of the fused layout (which adds the pairing coordinate).
// Runs of 2 for both storages: complex64 plain sweeps measured faster with runs of 2 than of 4 (c2: 4.58 -> 4.47 ms
// per sample; the 2^25-coset plain write 222 -> 200 us) and slower with runs of 1.
int plain_lr(int) { return 1; }
int fused_lr(int storage) { return storage == 0 ? 1 : 0; }

void* decide_kernel_ptr() { return reinterpret_cast<void*>(&decide_kernel); }
template <int NQ>
hipError_t reduce_for(double* part, unsigned nblk, Ctl* ctl, const Epi& epi, int sweep, unsigned strings, hipStream_t stream) {
    Epi e = epi;
    void* args[] = {&part, &nblk, &ctl, &e, &sweep};
    if (nblk >= unsigned(kWideReduce))
        return hipLaunchKernel(reinterpret_cast<void*>(&wide_reduce_kernel<NQ>), dim3(kThreads / 64 * NQ, strings), dim3(64),
                               args, 0, stream);
    return hipLaunchKernel(reinterpret_cast<void*>(&sweep_reduce_kernel<NQ>), dim3(1, strings), dim3(kThreads), args, 0,
                           stream);
}
// Reduction of nq partial sums per block after a sweep of nblk blocks and strings (Gram 4, direct 2, write 2, write +
// Gram 6, write + direct 4; a product pass 1, with the next step's Gram 5; chain-mode sweeps one per step).
hipError_t launch_reduce(int nq, double* part, unsigned nblk, Ctl* ctl, const Epi& epi, int sweep, unsigned strings,
                         hipStream_t stream) {
    switch (nq) {
        case 1: return reduce_for<1>(part, nblk, ctl, epi, sweep, strings, stream);
        case 2: return reduce_for<2>(part, nblk, ctl, epi, sweep, strings, stream);
        case 3: return reduce_for<3>(part, nblk, ctl, epi, sweep, strings, stream);
        case 4: return reduce_for<4>(part, nblk, ctl, epi, sweep, strings, stream);
        case 5: return reduce_for<5>(part, nblk, ctl, epi, sweep, strings, stream);
        case 6: return reduce_for<6>(part, nblk, ctl, epi, sweep, strings, stream);
    }
    return hipErrorInvalidValue;
}
void* publish_kernel_ptr() { return reinterpret_cast<void*>(&publish_kernel); }
void* run_hist_kernel_ptr(int storage) {
    return storage == 0 ? reinterpret_cast<void*>(&run_hist_kernel<float2>)
                        : reinterpret_cast<void*>(&run_hist_kernel<double2>);
}
void* run_apply_kernel_ptr(int storage) {
    return storage == 0 ? reinterpret_cast<void*>(&run_apply_kernel<float2, false, kRoute1>)
                        : reinterpret_cast<void*>(&run_apply_kernel<double2, false, kRoute1>);
}
// The product pass of a paired run that also sums the next step's Gram matrix (next route route2).
template <class S>
void* run_apply_gram_for(int route2) {
    switch (route2) {
        case kRoute1: return reinterpret_cast<void*>(&run_apply_kernel<S, true, kRoute1>);
        case kRouteSplit: return reinterpret_cast<void*>(&run_apply_kernel<S, true, kRouteSplit>);
        case kRouteMixA: return reinterpret_cast<void*>(&run_apply_kernel<S, true, kRouteMixA>);
        case kRouteMixB: return reinterpret_cast<void*>(&run_apply_kernel<S, true, kRouteMixB>);
    }
    return nullptr;
}
void* run_apply_gram_kernel_ptr(int storage, int route2) {
    return storage == 0 ? run_apply_gram_for<float2>(route2) : run_apply_gram_for<double2>(route2);
}
void* run_chunk_kernel_ptr() { return reinterpret_cast<void*>(&run_chunk_kernel); }
void* run_decide_kernel_ptr() { return reinterpret_cast<void*>(&run_decide_kernel); }

}  // namespace gs
