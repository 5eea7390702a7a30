// Chain logic of the sweeps (one thread), and the end of a sweep: block sums, partials, the chain's next state.
#pragma once
#include "gs_math.h"

namespace gs {

__device__ __forceinline__ double2 step_m(const KStep& s, int b, int x) {
    return make_double2(s.mre[b][x], s.mim[b][x]);
}

__device__ void publish(Ctl& c, const Epi& e) {
    if (e.mode == kChain1 && !c.dead) c.logp = log2(c.prev) - e.ns;
    if (e.quiet) return;
    e.out[0] = c.logp;
    e.out[1] = c.logscale;
    e.out[2] = c.prev;
    e.out[3] = c.dead;
}

// Bookkeeping of the write of step k (norm nb of the written FP64 values, nst of the rounded stored values).
__device__ void finish_write(Ctl& c, const Epi& e, int k, double nb, double nst) {
    c.nstored = nst;
    if (e.mode == kChain1) {                                   // gsamp2.cpp:67
        if (!e.quiet) e.cond[k] = nb / (2 * c.prev);
        c.prev = nb;
        if (nb <= 0) {
            if (!e.quiet)
                for (int q = k; q < e.ns; q++) e.cond[q] = 0;
            c.logp = -INFINITY;
            c.dead = 1;
        }
    } else if (e.mode == kRun) {                               // gsamp2.cpp:93-95
        c.logscale += 0.5 * log2(c.prev);
        const double cd = nb / 2;
        if (!e.quiet) e.cond[k] = cd;
        c.prev = nb;
        if (nb <= 0) {
            if (!e.quiet)
                for (int q = k; q < e.k1; q++) {
                    e.cond[q] = 0;
                    e.bits[q] = e.forced[q] < 0 ? 0 : e.forced[q];
                }
            c.logp = -INFINITY;
            c.dead = 1;
        } else {
            c.logp += log2(cd);
        }
    }
    if (c.dead) publish(c, e);
}

// Decision of step k from its norms: norm == kGram (red = G00, G11, Re G01, Im G01), kDirect (red = n0, n1), or -1
// (no norms: forced step, chain1, or a growth step whose norms follow from the stored table's norm).
__device__ void decide(Ctl& c, const Epi& e, int k, int norm, const double* red) {
    const KStep& s = e.plain[k];
    int bv = e.forced ? e.forced[k] : -1;
    double sc = 1.0;
    const bool need_p = (e.mode == kChain) || (e.mode == kRun && bv < 0);
    double n0 = 0, n1 = 0;
    if (need_p) {
        for (int b = 0; b < 2; b++) {
            const double2 m0 = step_m(s, b, 0), m1 = step_m(s, b, 1);
            double nbv;
            if (norm == kGram) {
                const double pr = m0.x * m1.x + m0.y * m1.y, pi = m0.y * m1.x - m0.x * m1.y;   // m0 conj(m1)
                nbv = norm2(m0) * red[0] + norm2(m1) * red[1] + 2 * (pr * red[2] - pi * red[3]);
            } else if (norm == kDirect) {
                nbv = red[b];
            } else {
                nbv = (norm2(m0) + norm2(m1)) * c.nstored;
            }
            (b ? n1 : n0) = nbv;
        }
    }
    if (e.mode == kChain) {                                    // gsamp2.cpp:46-49
        const double p1 = n1 / (n0 + n1);
        if (bv < 0) bv = e.U[k] < p1;
        const double pb = bv ? p1 : 1 - p1;
        if (pb <= 0) {
            c.logp = -INFINITY;
            c.dead = 1;
            publish(c, e);
            return;
        }
        c.logp += log2(pb);
        sc = 1.0 / sqrt(bv ? n1 : n0);
    } else if (e.mode == kChain1) {
        sc = 1.0;
    } else {                                                   // gsamp2.cpp:80-87
        sc = 1.0 / sqrt(c.prev);
        if (bv < 0) bv = e.U[c.qidx++] < n1 / (n0 + n1);
    }
    if (!e.quiet) e.bits[k] = int8_t(bv);
    c.bv = bv;
    c.sc = sc;
    const double2 m0 = step_m(s, bv, 0), m1 = step_m(s, bv, 1);
    c.w[0] = m0.x * sc;
    c.w[1] = m0.y * sc;
    c.w[2] = m1.x * sc;
    c.w[3] = m1.y * sc;
}

// Block-wide sum of v[NQ] over the NT threads in a fixed order (a butterfly inside each 64-lane wave, then the wave
// sums in wave order by one thread: two barriers instead of a log2(NT)-level tree); the result is in sh[0][*].
template <int NQ, int NT = kThreads>
__device__ __forceinline__ void block_tree_sum(double (&sh)[NT / 64][NQ], const double (&v)[NQ], int t) {
    double r[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        r[q] = v[q];
        for (int o = 32; o > 0; o >>= 1) r[q] += __shfl_xor(r[q], o, 64);
    }
    if ((t & 63) == 0)
#pragma unroll
        for (int q = 0; q < NQ; q++) sh[t >> 6][q] = r[q];
    __syncthreads();
    if (t == 0)
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            double x = sh[0][q];
            for (int w = 1; w < NT / 64; w++) x += sh[w][q];
            sh[0][q] = x;
        }
    __syncthreads();
}

// Chain logic after a sweep, from its reduced sums (one thread).  MULTI: the sweep may be one of several steps (the others
// are spared the code, which costs them registers and scratch: 6 hybrid strings of 60 steps, 712 us with it, 650 without).
template <int NQ, bool MULTI = false>
__device__ void chain_step(const double (&red)[NQ], Ctl* ctl, const Epi& e, int sweep) {
    Ctl& c = *ctl;
    if constexpr (NQ == 1) {            // one sum: the product pass of a run (role kRoleStored), the stored norm
        c.nstored = red[0];
        return;
    } else if constexpr (NQ == 5) {     // a product pass that also summed the next step's Gram (kRoleStoredGram)
        c.nstored = red[0];
        if (!c.dead) decide(c, e, e.k + 1, kGram, red + 1);
        return;
    } else if (e.role == kRoleNorm) {
        decide(c, e, e.k, sweep, red);
    } else if (MULTI && NQ <= 4 && e.role == kRolePair) {
#pragma unroll
        for (int i = 0; i < NQ; i++) {
            if (c.dead) break;
            if (i) decide(c, e, e.k + i, -1, nullptr);
            finish_write(c, e, e.k + i, red[i], red[i]);
        }
        if (!c.dead) {
            if (e.k + NQ == e.k1) publish(c, e);
            else if (e.next == kNextDecide) decide(c, e, e.k + NQ, -1, nullptr);
        }
    } else if (MULTI && (NQ == 4 || NQ == 6) && e.role == kRolePeek) {
        double w[4];
#pragma unroll
        for (int q = 0; q < 4; q++) w[q] = c.w[q];
        finish_write(c, e, e.k, red[0], red[1]);
        if (!c.dead) decide(c, e, e.k + 1, NQ == 6 ? kGram : kDirect, red + 2);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            c.w2[q] = c.w[q];
            c.w[q] = w[q];
        }
    } else {
        finish_write(c, e, e.k, red[0], red[1]);
        if (!c.dead) {
            if (e.k + 1 == e.k1) publish(c, e);
            else if (e.next == kNextDecide) decide(c, e, e.k + 1, -1, nullptr);
            else if (e.next == kNextFusedGram) decide(c, e, e.k + 1, kGram, red + 2);
            else if (e.next == kNextFusedDirect) decide(c, e, e.k + 1, kDirect, red + 2);
        }
    }
}

// Fixed-order sum of the first NQ values of nblk block partials by one block; the result is in sh[0][*].
template <int NQ>
__device__ __forceinline__ void reduce_partials(double (&sh)[kThreads / 64][NQ], const double* part, unsigned nblk,
                                                int t, bool atomic_loads) {
    double r[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) r[q] = 0;
    for (unsigned i = t; i < nblk; i += kThreads)
#pragma unroll
        for (int q = 0; q < NQ; q++)
            r[q] += atomic_loads ? __hip_atomic_load(part + size_t(i) * kPartStride + q, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT)
                                 : part[size_t(i) * kPartStride + q];
    block_tree_sum<NQ>(sh, r, t);
}

// End of a sweep block: the block's sums go to its partial slot.  Launches of at most kFenceBlocks blocks finish in
// the kernel: the last block of a string to arrive (agent-scope counter) reduces and runs the chain; a string's only
// block does so at once.  Larger launches end here and sweep_reduce_kernel follows on the stream: an agent-scope
// release per block writes back the XCD's L2 each time (tens of ns per block), which a launch boundary does once.
template <int NQ, bool MULTI = false>
__device__ void sweep_epilogue(double (&acc)[NQ], double* part, Ctl* ctl, const Epi& e, int sweep) {
    // block sum (wave butterfly, then the 4 waves in order)
#pragma unroll
    for (int q = 0; q < NQ; q++)
        for (int o = 32; o > 0; o >>= 1) acc[q] += __shfl_xor(acc[q], o, 64);
    __shared__ double sh[kThreads / 64][NQ];
    __shared__ int s_last;
    const int t = threadIdx.x;
    const unsigned nblk = gridDim.x;
    const bool inkernel = reduces_in_kernel(nblk, gridDim.y);
    if ((t & 63) == 0)
#pragma unroll
        for (int q = 0; q < NQ; q++) sh[t >> 6][q] = acc[q];
    __syncthreads();
    if (t == 0) {
        double* mine = part + size_t(blockIdx.x) * kPartStride;
        double red[NQ];
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            double v = sh[0][q];
#pragma unroll
            for (int w = 1; w < kThreads / 64; w++) v += sh[w][q];
            red[q] = v;
        }
        if (nblk == 1) {
            chain_step<NQ, MULTI>(red, ctl, slot_epi(e), sweep);
        } else {
#pragma unroll
            for (int q = 0; q < NQ; q++) {
                if (inkernel) __hip_atomic_store(mine + q, red[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                else mine[q] = red[q];
            }
        }
        if (inkernel && nblk > 1) {
            const unsigned done = __hip_atomic_fetch_add(e.counter + blockIdx.y, 1u, __ATOMIC_ACQ_REL,
                                                         __HIP_MEMORY_SCOPE_AGENT);
            s_last = done == nblk - 1;
        }
    }
    if (!inkernel || nblk == 1) return;
    __syncthreads();
    if (!s_last) return;
    __atomic_thread_fence(__ATOMIC_ACQUIRE);
    reduce_partials<NQ>(sh, part, nblk, t, true);
    if (t != 0) return;
    double red[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) red[q] = sh[0][q];
    chain_step<NQ, MULTI>(red, ctl, slot_epi(e), sweep);
    __hip_atomic_store(e.counter + blockIdx.y, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace gs
