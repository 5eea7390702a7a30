// Sweep kernels of the in-place cut-rank dynamic program on CDNA4 (gfx950).
//
// One step reads, for every coset representative c < 2^nk, the ntq live slots base(c) ^ off_j (base is GF(2)-linear
// in c: XOR of the coordinate columns selected by the bits of c) and produces for each measured bit b and output tau
//   out[b][tau] = sum_{terms} M[b][x] (-1)^{x (parity(c & rhoc) ^ par_j)} mem[base(c) ^ off_j]
// (gsamp2.cpp:32-38).  The sums are regrouped as out[b][tau] = M[b][0] A[tau][0] + M[b][1] A[tau][1] with A[tau][x]
// the signed slot sums routed to (tau, x); all arithmetic is FP64, the arena is complex<float> (c64) or
// complex<double> (c128), and a store rounds once (gsamp2.cpp:35, :52).
//
// Sweeps (template SWEEP):
//   kGram        per block, the 2x2 Gram matrix G[x][x'] = sum_c sum_tau A[tau][x] conj(A[tau][x']); the branch norms
//                n_b = sum_{x,x'} M[b][x] conj(M[b][x']) G[x][x'] follow without recomputing both branches;
//   kDirect      per block, n_0 and n_1 summed directly as |out[b][tau]|^2 (full relative precision for forced
//                strings, the reference's norm pass);
//   kWrite       stores out[bv][tau] * sc in place (tau 0 at base, tau 1 at base ^ g) and returns the FP64 norm of the
//                written values and of the rounded stored values;
//   kWriteGram / kWriteDirect  kWrite, plus the Gram matrix / direct norms of the NEXT step computed from the values
//                just stored: the thread's cosets are chosen to span the next step's pairing vector, so both slots of
//                each next-step coset are in the thread's registers.  This removes the next step's norm pass (one
//                read of the table per sampled step).
//
// Layout.  A block of 256 threads handles a tile of 256 * V cosets per iteration; thread t owns the V = VR * VG
// cosets whose low coordinates run over 0..V-1.  Coordinates 0..log2(VR)-1 have unit physical columns, so the VR
// cosets' slots are one aligned run (a 16-byte vector access); with VG = 2, coordinate log2(VR) has an arbitrary
// column Gamma (a second run).  XOR with low offset bits permutes a run; the permutation is undone in registers.
// Each thread writes exactly the slots it read (or fresh slots of a growth step): race free in place.
//
// Tiles are enumerated in Gray-code order inside a block, so the next tile XORs one column into the base address and
// flips the parity bits by one mask: O(1) scalar work per tile.
//
// Chain logic.  The block partial sums of a sweep are reduced in a fixed order and the chain runs on the device: the
// bookkeeping of a write (chain1 / run_steps conditionals, the stored table's norm) and the decision of the next step
// (forced, or U_k < p1 with U_k drawn on the host: gsamp2.cpp:47, :86, :108 draw one uniform per sampled step from a
// stream that does not depend on p1).  Sweeps of a few blocks reduce in their last block (agent-scope counter);
// larger ones are followed by a one-block reduction kernel.  No host round trip.
//
// Arithmetic per coset.  The sign of an x = 1 term is (-1)^{pc} sigma_j with pc = parity(c & rhoc) (per coset) and
// sigma_j = (-1)^{par_j} (per step), so A[tau][1] = (-1)^{pc} sigma_{j0} B_tau with B_tau = sum_j sigma_{j0} sigma_j
// slot_j: sigma_{j0} goes into the step's coefficient and (-1)^{pc} flips the fresh product M_b1 B_tau (one XOR per
// component).  The fused sweeps reduce the next step's Gram matrix from per-route invariants of each next-step coset
// (a, b): |a|^2 + |b|^2, Re/Im a conj(b), |a|^2 - |b|^2, with the per-coset signs applied to scalars.
#pragma once
#include "gs_chain.h"

namespace gs {

__device__ __forceinline__ double2 negate_if(double2 a, int s) {
    const unsigned long long m = (unsigned long long)(s & 1) << 63;
    return make_double2(__longlong_as_double(__double_as_longlong(a.x) ^ m),
                        __longlong_as_double(__double_as_longlong(a.y) ^ m));
}
// output index of offset j's x = 0 / x = 1 term under each canonical route
template <int ROUTE>
__device__ __host__ constexpr int tau_x0(int j) {
    return ROUTE == kRouteMixA || ROUTE == kRouteMixB ? (j & 1) : 0;
}
template <int ROUTE>
__device__ __host__ constexpr int tau_x1(int j) {
    return ROUTE == kRoute1 ? 0 : ROUTE == kRouteSplit ? 1 : ROUTE == kRouteMixA ? 1 - (j & 1) : (j & 1);
}

// Accumulate the routed signed slot sums of one coset: A[tau][x] += slot values (sign (-1)^{pc ^ par_j} on x = 1).
// The sums start from -0.0, the additive identity (x + -0.0 == x for every x), so a sum of one term compiles to no
// addition at all.
template <int ROUTE, int NTQ, int MO>
__device__ __forceinline__ void route_terms(double2 (&A)[MO][2], const double2 (&w)[NTQ], int pc, uint32_t parmask) {
#pragma unroll
    for (int t = 0; t < MO; t++) A[t][0] = A[t][1] = make_double2(-0.0, -0.0);
#pragma unroll
    for (int j = 0; j < NTQ; j++) {
        A[tau_x0<ROUTE>(j)][0] = cadd(A[tau_x0<ROUTE>(j)][0], w[j]);
        A[tau_x1<ROUTE>(j)][1] = cadd(A[tau_x1<ROUTE>(j)][1], negate_if(w[j], pc ^ int(parmask >> j)));
    }
}

template <int MO>
__device__ __forceinline__ void gram_acc(const double2 (&A)[MO][2], double* acc) {
#pragma unroll
    for (int t = 0; t < MO; t++) {
        const double2 a = A[t][0], b = A[t][1];
        add_norm(acc[0], a);
        add_norm(acc[1], b);
        acc[2] = fma(a.x, b.x, fma(a.y, b.y, acc[2]));      // Re a conj(b)
        acc[3] = fma(a.y, b.x, fma(-a.x, b.y, acc[3]));     // Im a conj(b)
    }
}

template <int MO>
__device__ __forceinline__ void direct_acc(const double2 (&A)[MO][2], const double2 (&M)[2][2], double* acc) {
#pragma unroll
    for (int t = 0; t < MO; t++) {
        add_norm(acc[0], cfma(M[0][0], A[t][0], cmul(M[0][1], A[t][1])));
        add_norm(acc[1], cfma(M[1][0], A[t][0], cmul(M[1][1], A[t][1])));
    }
}

// (-1)^s v for s in {0, 1} (sign bit flip)
__device__ __forceinline__ double flip(double v, uint32_t s) {
    return __hiloint2double(__double2hiint(v) ^ int(s << 31), __double2loint(v));
}
__device__ __forceinline__ double2 flip2(double2 v, uint32_t s) { return make_double2(flip(v.x, s), flip(v.y, s)); }

// First offset routed to (tau, x = 1), or -1.
template <int ROUTE, int NTQ>
__device__ __host__ constexpr int first_x1(int tau) {
    for (int j = 0; j < NTQ; j++)
        if (tau_x1<ROUTE>(j) == tau) return j;
    return -1;
}

// Per-launch write coefficients: w1t[tau] = sigma_{j0(tau)} w1 and rho[j] = sigma_{j0} sigma_j (j0 = first_x1 of
// offset j's x = 1 output).
template <int ROUTE, int NTQ, int MO>
__device__ __forceinline__ void write_coefs(double2 w1, uint32_t parmask, double2 (&w1t)[MO], double (&rho)[NTQ]) {
#pragma unroll
    for (int t = 0; t < MO; t++) {
        const int j0 = first_x1<ROUTE, NTQ>(t);
        w1t[t] = j0 >= 0 ? flip2(w1, (parmask >> j0) & 1) : w1;
    }
#pragma unroll
    for (int j = 0; j < NTQ; j++) {
        const int j0 = first_x1<ROUTE, NTQ>(tau_x1<ROUTE>(j));
        rho[j] = flip(1.0, ((parmask >> j) ^ (parmask >> j0)) & 1);
    }
}

// Output tau of one coset: w0 A[tau][0] + (-1)^pc w1t[tau] B_tau (the slot sums in offset order, as route_terms).
template <int ROUTE, int NTQ, int MO>
__device__ __forceinline__ double2 write_out(int t, const double2 (&x)[NTQ], uint32_t pc, double2 w0,
                                             const double2 (&w1t)[MO], const double (&rho)[NTQ]) {
    double2 a = make_double2(0, 0), b = a;
    bool h0 = false, h1 = false;
#pragma unroll
    for (int j = 0; j < NTQ; j++) {
        if (tau_x0<ROUTE>(j) == t) {
            a = h0 ? cadd(a, x[j]) : x[j];
            h0 = true;
        }
        if (tau_x1<ROUTE>(j) == t) {
            b = h1 ? make_double2(fma(rho[j], x[j].x, b.x), fma(rho[j], x[j].y, b.y)) : x[j];
            h1 = true;
        }
    }
    if (!h1) return cmul(w0, a);
    const double2 p = flip2(cmul(w1t[t], b), pc);
    return h0 ? cfma(w0, a, p) : p;
}

// Next-step Gram invariants of one coset (va, vb) in coset order; J swaps the roles of the two slots, sg is the
// coset's sign bit.  Accumulators: N = sum |va|^2 + |vb|^2, R = sum Re va conj(vb), SR = sum (-1)^sg Re, SI = sum
// (-1)^{sg ^ J} Im, SN = sum (-1)^sg N, SD = sum (-1)^{sg ^ J} (|va|^2 - |vb|^2).
enum { kgN, kgR, kgSR, kgSI, kgSN, kgSD, kgCount };
template <int ROUTE2>
__device__ __forceinline__ void gram_invariants(double2 va, double2 vb, uint32_t J, uint32_t sg, double (&g)[kgCount]) {
    if constexpr (ROUTE2 == kRouteSplit || ROUTE2 == kRouteMixA) {
        add_norm(g[kgN], va);
        add_norm(g[kgN], vb);
    } else {
        const double na = norm2(va), nb = norm2(vb);
        g[kgN] += na + nb;
        g[kgSN] += flip(na + nb, sg);
        g[kgSD] += flip(na - nb, sg ^ J);
    }
    if constexpr (ROUTE2 == kRouteSplit) {
        g[kgR] = fma(va.x, vb.x, fma(va.y, vb.y, g[kgR]));
    } else if constexpr (ROUTE2 == kRouteMixA || ROUTE2 == kRoute1) {
        const double re = fma(va.x, vb.x, va.y * vb.y), im = fma(va.y, vb.x, -va.x * vb.y);
        if constexpr (ROUTE2 == kRoute1) g[kgR] += re;
        g[kgSR] += flip(re, sg);
        g[kgSI] += flip(im, sg ^ J);
    }
}

// G00, G11, Re G01, Im G01 of the next step from the invariants (sigma1 = (-1)^{par} of its second slot).
template <int ROUTE2>
__device__ __forceinline__ void gram_assemble(const double (&g)[kgCount], int par, double* G) {
    const double s1 = par ? -1.0 : 1.0;
    if constexpr (ROUTE2 == kRouteSplit) {
        G[0] = g[kgN] + 2 * g[kgR];
        G[1] = g[kgN] + 2 * s1 * g[kgR];
        G[2] = 0;
        G[3] = 0;
    } else if constexpr (ROUTE2 == kRouteMixA) {
        G[0] = G[1] = g[kgN];
        G[2] = (1 + s1) * g[kgSR];
        G[3] = (s1 - 1) * g[kgSI];
    } else if constexpr (ROUTE2 == kRouteMixB) {
        G[0] = G[1] = g[kgN];
        G[2] = par ? g[kgSD] : g[kgSN];
        G[3] = 0;
    } else {
        G[0] = g[kgN] + 2 * g[kgR];
        G[1] = g[kgN] + 2 * s1 * g[kgR];
        G[2] = (par ? g[kgSD] : g[kgSN]) + (1 + s1) * g[kgSR];
        G[3] = (s1 - 1) * g[kgSI];
    }
}

// The chain step of block partials a previous sweep left unreduced, run at the start of the next sweep by every block
// (fixed-order sums: every block computes the same state); thread 0 of block 0 alone writes the string's outputs and
// stores the state at epi.ctl_out.  cl receives the state in every thread.
template <int NQ>
__device__ void pending_reduce_step(Ctl& cl, const Ctl* ctl, const Epi& epi, Ctl* shc) {
    __shared__ double sh[kThreads / 64][NQ];
    const int t = threadIdx.x;
    reduce_partials<NQ>(sh, epi.pend_part + size_t(blockIdx.y) * epi.slot_part, epi.pend_nblk, t, false);
    if (t == 0) {
        Ctl c = *ctl;
        if (!c.dead) {
            double red[NQ];
#pragma unroll
            for (int q = 0; q < NQ; q++) red[q] = sh[0][q];
            Epi ep = slot_epi(epi);
            ep.k = epi.pend_k;
            ep.role = epi.pend_role;
            ep.next = epi.pend_next;
            ep.quiet = blockIdx.x != 0;
            chain_step<NQ>(red, &c, ep, epi.pend_sweep);
        }
        *shc = c;
        if (blockIdx.x == 0) epi.ctl_out[blockIdx.y] = c;
    }
    __syncthreads();
    cl = *shc;
}

__device__ void pending_step(Ctl& cl, const Ctl* ctl, const Epi& epi) {
    __shared__ Ctl shc;
    if (epi.pend_nq == 2) pending_reduce_step<2>(cl, ctl, epi, &shc);
    else if (epi.pend_nq == 4) pending_reduce_step<4>(cl, ctl, epi, &shc);
    else pending_reduce_step<6>(cl, ctl, epi, &shc);
}

// ---------------------------------------------------------------------------------------------------------------
// the sweep

template <class S, int VR, int VG, int NTQ, int ROUTE, int SWEEP, int ROUTE2>
__global__ __launch_bounds__(kThreads) void sweep_kernel(const KStep* __restrict__ sp, S* __restrict__ mem,
                                                         double* __restrict__ part, Ctl* __restrict__ ctl, Epi epi) {
    constexpr int MO = ROUTE == kRoute1 ? 1 : 2;
    constexpr int MO2 = ROUTE2 == kRoute1 ? 1 : 2;
    constexpr int LR = VR == 1 ? 0 : VR == 2 ? 1 : 2;
    constexpr int LV = LR + (VG == 4 ? 2 : VG == 2 ? 1 : 0);
    constexpr int V = VR * VG;
    constexpr bool WRITES = SWEEP >= kWrite;
    constexpr bool FUSED = SWEEP == kWriteGram || SWEEP == kWriteDirect;
    constexpr bool GRAM1 = SWEEP == kWriteGram1;
    constexpr int NA = SWEEP == kGram ? 4 : SWEEP == kDirect ? 2 : SWEEP == kWrite ? 2
                     : SWEEP == kWriteGram || SWEEP == kWriteGram1 ? 6 : 4;
    const KStep& s = *sp;
    const int nk = s.nk;
    const int tid = threadIdx.x;
    mem += uint64_t(blockIdx.y) * epi.slot_entries;   // this block's string
    part += size_t(blockIdx.y) * epi.slot_part;
    ctl += blockIdx.y;
    constexpr int lt = LV + 8;                     // log2 cosets per tile

    // parity bits of a coordinate: bit 0 output sign, bit 1 next-step slot index, bit 2 next-step sign, bit 3 the
    // next step's second slot-index bit (four-slot next step)
    auto pb = [&](int j) -> int {
        int p = int((s.pmask[0] >> j) & 1) | (int((s.pmask[1] >> j) & 1) << 1) | (int((s.pmask[2] >> j) & 1) << 2);
        if constexpr (VG == 4) p |= int((s.pmask[3] >> j) & 1) << 3;
        return p;
    };
    uint64_t a_thr = 0;
    int p_thr = 0;
#pragma unroll
    for (int b = 0; b < 8; b++) {
        const int j = LV + b;
        if (j < nk && ((tid >> b) & 1)) {
            a_thr ^= s.cols[j];
            p_thr ^= pb(j);
        }
    }
    const bool active = nk >= lt || (uint64_t(tid) << LV) < (uint64_t(1) << nk);
    uint64_t a_blk = 0;
    int p_blk = 0;
    // s.xcd: blocks are dealt round-robin to the 8 XCDs, so block i's XCD is i mod 8; rotating the 3 low bits of the
    // block index to the top gives each XCD one contiguous eighth of the block coordinates (of each tile window)
    const unsigned bid = s.xcd && s.lg_grid >= 3
                             ? (blockIdx.x >> 3) | ((blockIdx.x & 7u) << (s.lg_grid - 3))
                             : blockIdx.x;
    for (int b = 0; b < s.lg_grid; b++)
        if ((bid >> b) & 1) {
            a_blk ^= s.cols[lt + b];
            p_blk ^= pb(lt + b);
        }
    const int jit = lt + s.lg_grid;
    const int niter = 1 << s.lg_iter;
    int plow[V];                                   // parity bits of the thread's low coordinates
#pragma unroll
    for (int i = 0; i < V; i++) {
        int p = 0;
#pragma unroll
        for (int b = 0; b < LV; b++)
            if ((i >> b) & 1) p ^= pb(b);
        plow[i] = p;
    }
    const uint64_t gam = VG >= 2 ? s.cols[LR] : 0, gam2 = VG == 4 ? s.cols[LR + 1] : 0;
    auto goff = [&](int ig) -> uint64_t { return ((ig & 1) ? gam : 0) ^ ((ig & 2) ? gam2 : 0); };

    double2 w0 = make_double2(0, 0), w1 = w0;
    double2 M[2][2] = {{w0, w0}, {w0, w0}};
    double2 w1t[MO];
    double rho[NTQ];
    if constexpr (SWEEP == kDirect || SWEEP == kWriteDirect) {
        const KStep& ms = SWEEP == kDirect ? epi.plain[epi.k] : epi.plain[epi.k + 1];
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int x = 0; x < 2; x++) M[b][x] = make_double2(ms.mre[b][x], ms.mim[b][x]);
    }
    uint64_t off[NTQ];
#pragma unroll
    for (int j = 0; j < NTQ; j++) off[j] = s.off[j];
    const uint32_t parmask = s.parmask;
    const uint64_t g = s.g;
    const int eps = s.eps, phig = s.phig, nug = s.nug;
    const int sgg = s.sgg, sgk = s.sgk;
    const uint32_t par2mask = VG == 4 ? uint32_t(s.parmask2) : uint32_t(s.par2) << 1;
    const int eps2 = s.eps2;

    double acc[NA];
#pragma unroll
    for (int q = 0; q < NA; q++) acc[q] = 0;
    double gi[kgCount];                            // next-step Gram invariants (kWriteGram)
#pragma unroll
    for (int q = 0; q < kgCount; q++) gi[q] = 0;

    // Each tile is loaded at the top of its iteration, with no software pipeline: on this access pattern (four
    // regions per wave, each read and rewritten in place) issuing the next tile's loads early measured slower
    // (192.6 against 182.6 us per 2^25-coset fused sweep), as did a two-tile-deep pipeline and larger grids -- more
    // requests in flight cost more in the memory system than they hide.
    const uint64_t a_tb = a_thr ^ a_blk;
    S e[NTQ][VG][VR];
    auto load_tile = [&](uint64_t ag, S (&dst)[NTQ][VG][VR]) {
#pragma unroll
        for (int j = 0; j < NTQ; j++)
#pragma unroll
            for (int ig = 0; ig < VG; ig++)
                Run<S, VR>::load(mem, (ag ^ off[j] ^ goff(ig)) & ~uint64_t(VR - 1), dst[j][ig]);
    };
    // Tile index i runs 0 .. niter-1, or niter-1 .. 0 when s.rev (gray(i) ^ gray(i-1) = 1 << ctz(i)): the start of a
    // sweep then meets the end of the previous one, whose last lines may still be in the memory-side cache.
    const bool rev = s.rev != 0;
    uint64_t a_it = 0;
    int p_it = 0;
    if (rev && s.lg_iter > 0) {                     // gray(niter - 1) is the top bit alone
        a_it = s.cols[jit + s.lg_iter - 1];
        p_it = pb(jit + s.lg_iter - 1);
    }
    // Chain state of this launch: the kernel's ctl, or -- when the previous sweep left its block partials unreduced --
    // the chain step of those partials, run by every block on its own copy (the same fixed-order sums, so the same
    // result everywhere) while the first tile's loads are in flight; block 0 stores it at ctl_out.
    bool first_loaded = false;
    Ctl* cur = ctl;
    Ctl cl;
    if (epi.pend_nblk) {
        cur = epi.ctl_out + blockIdx.y;
        if (active) {
            load_tile(a_tb ^ a_it, e);
            first_loaded = true;
        }
        pending_step(cl, ctl, epi);
    } else {
        cl = *ctl;
    }
    if (cl.dead) return;
    if constexpr (WRITES) {
        w0 = make_double2(cl.w[0], cl.w[1]);
        w1 = make_double2(cl.w[2], cl.w[3]);
        write_coefs<ROUTE, NTQ, MO>(w1, s.parmask, w1t, rho);
    }
    for (int it = 0; it < niter; it++) {
        if (it > 0) {                               // Gray code: one coordinate changes
            const int b = __builtin_ctz(unsigned(rev ? niter - it : it));
            a_it ^= s.cols[jit + b];
            p_it ^= pb(jit + b);
        }
        const uint64_t ag = a_tb ^ a_it;
        const int pbase = p_thr ^ p_blk ^ p_it;
        if (!active) continue;
        if (it > 0 || !first_loaded) load_tile(ag, e);
#pragma unroll
        for (int j = 0; j < NTQ; j++)
#pragma unroll
            for (int ig = 0; ig < VG; ig++)
                permute<S, VR>(e[j][ig], unsigned(ag ^ off[j] ^ goff(ig)) & (VR - 1));
        S o[2][VG][VR];
#pragma unroll
        for (int ig = 0; ig < VG; ig++)
#pragma unroll
            for (int ir = 0; ir < VR; ir++) {
                const int i = ir + VR * ig;
                const int pc = (pbase ^ plow[i]) & 1;
                double2 wv[NTQ];
#pragma unroll
                for (int j = 0; j < NTQ; j++) wv[j] = Cx<S>::widen(e[j][ig][ir]);
                if constexpr (SWEEP == kGram || SWEEP == kDirect) {
                    double2 A[MO][2];
                    route_terms<ROUTE, NTQ, MO>(A, wv, pc, parmask);
                    if constexpr (SWEEP == kGram) gram_acc<MO>(A, acc);
                    else direct_acc<MO>(A, M, acc);
                } else {
#pragma unroll
                    for (int t = 0; t < MO; t++) {
                        const double2 v = write_out<ROUTE, NTQ, MO>(t, wv, uint32_t(pc), w0, w1t, rho);
                        const S sv = Cx<S>::narrow(v);
                        o[t][ig][ir] = sv;
                        // the written norm feeds chain1 / run_steps bookkeeping only (sampling renormalises by the
                        // decided branch's norm; accumulating it always is cheaper than selecting); the stored
                        // table's norm is read only by a growth step's analytic norms, and a fused write is never
                        // followed by a growth step
                        add_norm(acc[0], v);
                        if constexpr (GRAM1) {
                            // the next step reads this value as its coset's one slot: |v|^2 into N = G00 = G11 and,
                            // signed by that coset's (-1)^(pc ^ par), into Re G01 (Im G01 = 0)
                            const double nv = norm2(Cx<S>::widen(sv));
                            const uint32_t sg = uint32_t(((pbase ^ plow[i]) >> 2) ^ (t ? sgg : 0) ^ sgk) & 1;
                            acc[2] += nv;
                            acc[4] += flip(nv, sg);
                        } else if constexpr (!FUSED) {
                            add_norm(acc[1], Cx<S>::widen(sv));
                        }
                    }
                }
            }
        if constexpr (WRITES) {
            // stores go through a permuted copy; o stays in coset order for the fused norms
#pragma unroll
            for (int ig = 0; ig < VG; ig++)
#pragma unroll
                for (int t = 0; t < MO; t++) {
                    const uint64_t a = ag ^ goff(ig) ^ (t ? g : 0);
                    S so[VR];
#pragma unroll
                    for (int ir = 0; ir < VR; ir++) so[ir] = o[t][ig][ir];
                    permute<S, VR>(so, unsigned(a) & (VR - 1));
                    Run<S, VR>::store(mem, a & ~uint64_t(VR - 1), so);
                }
        }
        if constexpr (FUSED && VG == 4) {
            // four-slot next step: the next coset holding output (ir, ig=0, tau d) holds output (ir, ig=m, tau d ^
            // eps(m)) of the thread's coset m as its slot j0 ^ m, j0 the slot index of the first (both index bits and
            // the coset's sign are parities of the address)
#pragma unroll
            for (int ir = 0; ir < VR; ir++)
#pragma unroll
                for (int d = 0; d < MO; d++) {
                    const int pl = pbase ^ plow[ir];
                    const int j0 = (((pl >> 1) & 1) | (((pl >> 3) & 1) << 1)) ^ (d ? phig : 0);
                    const int sg = ((pl >> 2) ^ (d & nug)) & 1;
                    S a[4];
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        const int tm = d ^ ((m & 1) ? eps : 0) ^ ((m & 2) ? eps2 : 0);
                        if constexpr (MO == 2) a[m] = tm ? o[1][m][ir] : o[0][m][ir];
                        else a[m] = o[0][m][ir];
                    }
                    // slot q = member q ^ j0, by selects (j0 is per lane)
                    const S b0 = (j0 & 1) ? a[1] : a[0], b1 = (j0 & 1) ? a[0] : a[1];
                    const S b2 = (j0 & 1) ? a[3] : a[2], b3 = (j0 & 1) ? a[2] : a[3];
                    double2 w2[4];
                    w2[0] = Cx<S>::widen((j0 & 2) ? b2 : b0);
                    w2[1] = Cx<S>::widen((j0 & 2) ? b3 : b1);
                    w2[2] = Cx<S>::widen((j0 & 2) ? b0 : b2);
                    w2[3] = Cx<S>::widen((j0 & 2) ? b1 : b3);
                    double2 A2[MO2][2];
                    route_terms<ROUTE2, 4, MO2>(A2, w2, sg, par2mask);
                    if constexpr (SWEEP == kWriteGram) gram_acc<MO2>(A2, acc + 2);
                    else direct_acc<MO2>(A2, M, acc + 2);
                }
        } else if constexpr (FUSED) {
            // next step's cosets: output (ir, ig=0, tau d) pairs with output (ir, ig=1, tau d ^ eps); the element with
            // slot index 0 is the next coset's base slot, the other its second slot.
#pragma unroll
            for (int ir = 0; ir < VR; ir++)
#pragma unroll
                for (int d = 0; d < MO; d++) {
                    const int pl = pbase ^ plow[ir];
                    const int jidx = ((pl >> 1) ^ (d & phig)) & 1;
                    const int sg = ((pl >> 2) ^ (d & nug)) & 1;
                    const S va = o[d][0][ir];
                    S vb;
                    if constexpr (MO == 2) vb = (d ^ eps) ? o[1][1][ir] : o[0][1][ir];
                    else vb = o[0][1][ir];
                    if constexpr (SWEEP == kWriteGram) {
                        gram_invariants<ROUTE2>(Cx<S>::widen(va), Cx<S>::widen(vb), uint32_t(jidx), uint32_t(sg), gi);
                    } else {
                        double2 w2[2];              // select in the stored type, then widen
                        w2[0] = Cx<S>::widen(jidx ? vb : va);
                        w2[1] = Cx<S>::widen(jidx ? va : vb);
                        double2 A2[MO2][2];
                        route_terms<ROUTE2, 2, MO2>(A2, w2, sg, par2mask);
                        direct_acc<MO2>(A2, M, acc + 2);
                    }
                }
        }
    }
    if constexpr (SWEEP == kWriteGram && VG == 2) gram_assemble<ROUTE2>(gi, s.par2, acc + 2);
    if constexpr (GRAM1) acc[3] = acc[2];
    sweep_epilogue<NA>(acc, part, cur, epi, GRAM1 ? int(kWriteGram) : SWEEP);
}

// ---------------------------------------------------------------------------------------------------------------
// dispatch table

template <class S, int VR, int VG, int NTQ, int ROUTE, int SWEEP, int ROUTE2>
void* kptr() {
    return reinterpret_cast<void*>(&sweep_kernel<S, VR, VG, NTQ, ROUTE, SWEEP, ROUTE2>);
}

template <class S, int VR, int VG, int NTQ, int ROUTE, int SWEEP>
void* by_route2(int route2) {
    if constexpr (SWEEP == kWriteGram || SWEEP == kWriteDirect) {
        switch (route2) {
            case kRoute1: return kptr<S, VR, VG, NTQ, ROUTE, SWEEP, kRoute1>();
            case kRouteSplit: return kptr<S, VR, VG, NTQ, ROUTE, SWEEP, kRouteSplit>();
            case kRouteMixA: return kptr<S, VR, VG, NTQ, ROUTE, SWEEP, kRouteMixA>();
            case kRouteMixB: return kptr<S, VR, VG, NTQ, ROUTE, SWEEP, kRouteMixB>();
        }
        return nullptr;
    } else {
        return kptr<S, VR, VG, NTQ, ROUTE, SWEEP, kRoute1>();
    }
}

template <class S, int VR, int VG, int NTQ, int SWEEP>
void* by_route(int route, int route2) {
    switch (route) {
        case kRoute1: return by_route2<S, VR, VG, NTQ, kRoute1, SWEEP>(route2);
        case kRouteSplit: return by_route2<S, VR, VG, NTQ, kRouteSplit, SWEEP>(route2);
        case kRouteMixA: if constexpr (NTQ >= 2) return by_route2<S, VR, VG, NTQ, kRouteMixA, SWEEP>(route2); else return nullptr;
        case kRouteMixB: if constexpr (NTQ >= 2) return by_route2<S, VR, VG, NTQ, kRouteMixB, SWEEP>(route2); else return nullptr;
    }
    return nullptr;
}

template <class S, int VR, int VG, int SWEEP>
void* by_ntq(int ntq, int route, int route2) {
    switch (ntq) {
        case 1: return by_route<S, VR, VG, 1, SWEEP>(route, route2);
        case 2: return by_route<S, VR, VG, 2, SWEEP>(route, route2);
        case 4: return by_route<S, VR, VG, 4, SWEEP>(route, route2);
    }
    return nullptr;
}

// Fused sweeps followed by a four-slot step: mixed routes on both sides (the only ones the planner produces there).
template <class S, int VR, int NTQ, int SWEEP>
void* fused4(int route, int route2) {
    if (route == kRouteMixA)
        return route2 == kRouteMixA ? kptr<S, VR, 4, NTQ, kRouteMixA, SWEEP, kRouteMixA>()
                                    : kptr<S, VR, 4, NTQ, kRouteMixA, SWEEP, kRouteMixB>();
    return route2 == kRouteMixA ? kptr<S, VR, 4, NTQ, kRouteMixB, SWEEP, kRouteMixA>()
                                : kptr<S, VR, 4, NTQ, kRouteMixB, SWEEP, kRouteMixB>();
}

template <class S, int SWEEP>
void* by_layout(int lr, int vg, int ntq, int route, int route2) {
    constexpr bool c64 = sizeof(S) == 8;
    if constexpr (SWEEP == kWriteGram1) {                 // plain layout with runs of 2 only
        return vg == 1 && lr == 1 ? by_ntq<S, 2, 1, SWEEP>(ntq, route, route2) : nullptr;
    } else
    if constexpr (SWEEP == kWriteGram || SWEEP == kWriteDirect) {
        if (vg == 4) {                           // four-slot next step: two- and four-slot steps, mixed routes only
            constexpr int VR4 = c64 ? 2 : 1;
            if (lr != (c64 ? 1 : 0) || (route != kRouteMixA && route != kRouteMixB) ||
                (route2 != kRouteMixA && route2 != kRouteMixB))
                return nullptr;
            if (ntq == 2) return fused4<S, VR4, 2, SWEEP>(route, route2);
            if (ntq == 4) return fused4<S, VR4, 4, SWEEP>(route, route2);
            return nullptr;
        }
        if (vg != 2) return nullptr;
        if constexpr (c64) {
            if (lr == 1) return by_ntq<S, 2, 2, SWEEP>(ntq, route, route2);
            if (lr == 2) return by_ntq<S, 4, 2, SWEEP>(ntq, route, route2);
            return nullptr;
        }
        else return lr == 0 ? by_ntq<S, 1, 2, SWEEP>(ntq, route, route2) : nullptr;
    } else {
        if (vg == 2) {                           // two runs per thread: plain sweeps of one- and two-slot steps
            if (lr != 1) return nullptr;
            if (ntq == 1) return by_route<S, 2, 2, 1, SWEEP>(route, route2);
            if (ntq == 2) return by_route<S, 2, 2, 2, SWEEP>(route, route2);
            return nullptr;
        }
        if (vg != 1) return nullptr;
        if (lr == 0) return by_ntq<S, 1, 1, SWEEP>(ntq, route, route2);
        return lr == 1 ? by_ntq<S, 2, 1, SWEEP>(ntq, route, route2) : nullptr;
    }
}

// Kernel for (log2 run, vg, ntq, route, sweep, next route) of one storage type; nullptr when not built.
template <class S>
void* sweep_for(int lr, int vg, int ntq, int route, int sweep, int route2) {
    switch (sweep) {
        case kGram: return by_layout<S, kGram>(lr, vg, ntq, route, route2);
        case kDirect: return by_layout<S, kDirect>(lr, vg, ntq, route, route2);
        case kWrite: return by_layout<S, kWrite>(lr, vg, ntq, route, route2);
        case kWriteGram: return by_layout<S, kWriteGram>(lr, vg, ntq, route, route2);
        case kWriteDirect: return by_layout<S, kWriteDirect>(lr, vg, ntq, route, route2);
        case kWriteGram1: return by_layout<S, kWriteGram1>(lr, vg, ntq, route, route2);
    }
    return nullptr;
}

}  // namespace gs
