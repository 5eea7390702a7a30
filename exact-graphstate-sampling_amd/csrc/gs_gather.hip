// Gather sweeps of the two-table engine.
#include "gs_sweep.h"

namespace gs {

// Two-table (gather-form) steps (gsamp.cpp:21-29, :39-55; dp.cpp:44-53).  Output cp gathers its 2^nker inputs; S0 sums
// the x = 0 terms, S1 the x = 1 terms with sign (-1)^{parity(c & rho)}; the outputs are M[b][0] S0 + M[b][1] S1.
// Norm pass (SWEEP = kDirect): both branch norms |M[b][0] S0 + M[b][1] S1|^2 summed directly (the reference's chain).
// Write pass (kWrite): w0 S0 + w1 S1 stored at nw[cp] (contiguous), with w from the chain's decision or, for the
// amplitude engine, from wext[4k..4k+3] (the job's per-vertex weights).  NKS = 2^nker inputs per output.  Output
// bits 0..7 are the thread index, then the block index, then the tile index (groups of 4 tiles per thread, see
// below; one tile at a time when a block has fewer than 4).
template <class S, int SWEEP, int NKS>
__global__ __launch_bounds__(kThreads) void gather_kernel(const TStep* __restrict__ tp, const S* __restrict__ old,
                                                          S* __restrict__ nw, double* __restrict__ part,
                                                          Ctl* __restrict__ ctl, Epi epi,
                                                          const double* __restrict__ wext) {
    if (ctl->dead) return;
    const TStep& s = *tp;
    const int tid = threadIdx.x;
    uint64_t a_thr = 0;
#pragma unroll
    for (int b = 0; b < 8; b++)
        if (b < s.rn && ((tid >> b) & 1)) a_thr ^= s.dep[b];
    const bool active = s.rn >= 8 || tid < (1 << s.rn);
    uint64_t a_blk = 0;
    for (int b = 0; b < s.lg_grid; b++)
        if ((blockIdx.x >> b) & 1) a_blk ^= s.dep[8 + b];
    const int jit = 8 + s.lg_grid;
    const int niter = 1 << s.lg_iter;
    double2 M[2][2], w0 = make_double2(0, 0), w1 = w0;
    if constexpr (SWEEP == kDirect) {
        const KStep& ms = epi.plain[epi.k];
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int x = 0; x < 2; x++) M[b][x] = make_double2(ms.mre[b][x], ms.mim[b][x]);
    } else {
        const double* w = wext ? wext + 4 * epi.k : ctl->w;
        w0 = make_double2(w[0], w[1]);
        w1 = make_double2(w[2], w[3]);
    }
    uint64_t ks[NKS];
#pragma unroll
    for (int t = 0; t < NKS; t++) ks[t] = s.kspan[t];
    const uint64_t lowmask = s.lowmask, xbit = s.xbit, rho = s.rho;
    double acc[2] = {0, 0};
    // One output from its NKS gathered inputs (u0: its address before the kernel span): S0, S1, then the branch norms
    // (norm pass) or the write at cp.
    auto output = [&](const S (&v)[NKS], uint64_t u0, uint64_t cp) {
        double2 S0 = make_double2(0, 0), S1 = S0;
#pragma unroll
        for (int t = 0; t < NKS; t++) {
            const uint64_t u = u0 ^ ks[t];
            const double2 x = Cx<S>::widen(v[t]);
            if (u & xbit) S1 = cadd(S1, negate_if(x, __popcll(u & lowmask & rho) & 1));
            else S0 = cadd(S0, x);
        }
        if constexpr (SWEEP == kDirect) {
            add_norm(acc[0], cfma(M[0][0], S0, cmul(M[0][1], S1)));
            add_norm(acc[1], cfma(M[1][0], S0, cmul(M[1][1], S1)));
        } else {
            const double2 o = cfma(w0, S0, cmul(w1, S1));
            const S so = Cx<S>::narrow(o);
            Run<S, 1>::store(nw, cp, {so});
            add_norm(acc[0], o);
            add_norm(acc[1], Cx<S>::widen(so));
        }
    };
    const uint64_t ab = a_thr ^ a_blk;
    const uint64_t cb = (uint64_t(blockIdx.x) << 8) | uint64_t(tid);
    constexpr int U = 4;        // tiles per iteration (every gather of the U tiles in flight at once)
    if (niter >= U) {
        // Tiles of a group: j & 1 selects output bit jit, j >> 1 the second direction -- the partner direction
        // pdelta when the step has one (tiles j = 2, 3 then reuse the loads of tiles 0, 1, permuted by ptd: each
        // table entry is read once instead of twice), else output bit jit + 1.  The other tile bits (jit + 1 ..
        // rn - 1 without h, the second direction's top bit) take a Gray walk over the groups.
        const bool share = s.ph >= 0;
        const int h = share ? s.ph : jit + 1;
        const uint64_t d0 = s.dep[jit];
        const uint64_t D = share ? s.pD : s.dep[jit + 1];
        const uint64_t dc = share ? s.pdelta : uint64_t(1) << (jit + 1);
        const int td = s.ptd;
        uint64_t a_g = 0, c_g = 0;
        for (int g = 0; g < niter / U; g++) {
            if (g) {
                int b = jit + 1 + __builtin_ctz(unsigned(g));
                if (b >= h) b++;
                a_g ^= s.dep[b];
                c_g ^= uint64_t(1) << b;
            }
            if (!active) continue;
            S v[U][NKS];
            if (share) {
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const uint64_t u0 = ab ^ a_g ^ (j ? d0 : 0);
#pragma unroll
                    for (int t = 0; t < NKS; t++) v[j][t] = old[(u0 ^ ks[t]) & lowmask];
#pragma unroll
                    for (int t = 0; t < NKS; t++) {           // v[j][t ^ td] by selects (no indexed registers)
                        S x = v[j][0];
#pragma unroll
                        for (int q = 1; q < NKS; q++)
                            if ((t ^ td) == q) x = v[j][q];
                        v[j + 2][t] = x;
                    }
                }
            } else {
#pragma unroll
                for (int j = 0; j < U; j++) {
                    const uint64_t u0 = ab ^ a_g ^ ((j & 1) ? d0 : 0) ^ ((j & 2) ? D : 0);
#pragma unroll
                    for (int t = 0; t < NKS; t++) v[j][t] = old[(u0 ^ ks[t]) & lowmask];
                }
            }
#pragma unroll
            for (int j = 0; j < U; j++) {
                const uint64_t u0 = ab ^ a_g ^ ((j & 1) ? d0 : 0) ^ ((j & 2) ? D : 0);
                output(v[j], u0, (c_g | (uint64_t(j & 1) << jit) | cb) ^ ((j & 2) ? dc : 0));
            }
        }
    } else {
        uint64_t a_it = 0, c_it = 0;
        for (int it = 0; it < niter; it++) {
            if (it) {
                const int b = __builtin_ctz(unsigned(it));
                a_it ^= s.dep[jit + b];
                c_it ^= uint64_t(1) << (jit + b);
            }
            if (!active) continue;
            const uint64_t u0 = ab ^ a_it;
            S v[NKS];
#pragma unroll
            for (int t = 0; t < NKS; t++) v[t] = old[(u0 ^ ks[t]) & lowmask];
            output(v, u0, c_it | cb);
        }
    }
    if (epi.role != kRoleSilent) sweep_epilogue<2>(acc, part, ctl, epi, SWEEP);
}

// The write pass of step k that also sums step k+1's branch norms, from the values it stores (TFold).  A thread takes
// groups of 2^(ND2 + SHARE) outputs: along ND2 directions whose differences are the low parts of step k+1's kernel, so
// that all the entries one output of step k+1 gathers are in its registers, and with SHARE along the partner direction,
// whose outputs gather the same entries of the old table (see gather_kernel).  Step k+1 gathers every (entry, x) exactly
// once; an output whose kernel holds the bare x bit (PURE) takes both x of its entries, otherwise the two outputs X = 0, 1
// over the same entries take x = X ^ xk[t] of entry t.  One pass over the table per step instead of two: the
// complex128 width-26 sample 19.8 -> 9.5 ms with the writes' pairing, width 20 1.40 -> 0.71 ms.
template <class S, int NKS, int ND2, bool SHARE, bool PURE>
__global__ __launch_bounds__(kThreads) void gather_fold_kernel(const TStep* __restrict__ tp, const TFold* __restrict__ fp,
                                                               const S* __restrict__ old, S* __restrict__ nw,
                                                               double* __restrict__ part, Ctl* __restrict__ ctl,
                                                               Epi epi) {
    if (ctl->dead) return;
    constexpr int NB = 1 << ND2, NA = SHARE ? 2 : 1;
    const TStep& s = *tp;
    const TFold& f = *fp;
    const int tid = threadIdx.x;
    uint64_t cp = 0, u0 = 0;
#pragma unroll
    for (int b = 0; b < 8; b++)
        if ((tid >> b) & 1) {
            cp ^= uint64_t(1) << f.pos[b];
            u0 ^= s.dep[f.pos[b]];
        }
    for (int b = 0; b < f.lg_grid; b++)
        if ((blockIdx.x >> b) & 1) {
            cp ^= uint64_t(1) << f.pos[8 + b];
            u0 ^= s.dep[f.pos[8 + b]];
        }
    const double2 w0 = make_double2(ctl->w[0], ctl->w[1]), w1 = make_double2(ctl->w[2], ctl->w[3]);
    const KStep& ms = epi.plain[epi.k + 1];
    double2 M[2][2];
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
        for (int x = 0; x < 2; x++) M[b][x] = make_double2(ms.mre[b][x], ms.mim[b][x]);
    uint64_t ks[NKS], dv[NB], dD[NB];
    uint32_t sb[NB];                                  // sign parity of each direction sum
#pragma unroll
    for (int t = 0; t < NKS; t++) ks[t] = s.kspan[t];
#pragma unroll
    for (int e = 0; e < NB; e++) {
        dv[e] = ((e & 1) ? f.dvec[0] : 0) ^ ((e & 2) ? f.dvec[1] : 0);
        dD[e] = ((e & 1) ? f.dimg[0] : 0) ^ ((e & 2) ? f.dimg[1] : 0);
        sb[e] = uint32_t(__popcll(dv[e] & f.rho) & 1);
    }
    const uint64_t lowmask = s.lowmask, xbit = s.xbit, rho = s.rho;
    const uint32_t xk = f.xk, sp = uint32_t(__popcll(f.pdelta & f.rho) & 1);
    const int td = f.ptd;
    double acc[4] = {0, 0, 0, 0};
    for (int it = 0; it < (1 << f.lg_iter); it++) {
        if (it) {
            const int j = f.pos[8 + f.lg_grid + __builtin_ctz(unsigned(it))];
            cp ^= uint64_t(1) << j;
            u0 ^= s.dep[j];
        }
        S v[NB][NKS];
#pragma unroll
        for (int e = 0; e < NB; e++)
#pragma unroll
            for (int t = 0; t < NKS; t++) v[e][t] = old[(u0 ^ dD[e] ^ ks[t]) & lowmask];
        const uint32_t sg0 = uint32_t(__popcll(cp & f.rho) & 1);
#pragma unroll
        for (int a = 0; a < NA; a++) {
            double2 ew[NB];
#pragma unroll
            for (int e = 0; e < NB; e++) {
                const uint64_t ue = u0 ^ dD[e] ^ (a ? f.pimg : 0);
                double2 S0 = make_double2(0, 0), S1 = S0;
#pragma unroll
                for (int t = 0; t < NKS; t++) {
                    S y = v[e][t];
                    if (a) {                          // the partner's input t is input t ^ td (selects, no indexing)
                        y = v[e][0];
#pragma unroll
                        for (int q = 1; q < NKS; q++)
                            if ((t ^ td) == q) y = v[e][q];
                    }
                    const uint64_t u = ue ^ ks[t];
                    const double2 x = Cx<S>::widen(y);
                    if (u & xbit) S1 = cadd(S1, negate_if(x, __popcll(u & lowmask & rho) & 1));
                    else S0 = cadd(S0, x);
                }
                const double2 o = cfma(w0, S0, cmul(w1, S1));
                const S so = Cx<S>::narrow(o);
                Run<S, 1>::store(nw, cp ^ dv[e] ^ (a ? f.pdelta : 0), {so});
                ew[e] = Cx<S>::widen(so);
                add_norm(acc[0], o);
                add_norm(acc[1], ew[e]);
            }
            const uint32_t sg = sg0 ^ (a ? sp : 0);   // sign of the group's first entry as an x = 1 input of step k+1
#pragma unroll
            for (int X = 0; X < (PURE ? 1 : 2); X++) {
                double2 S0 = make_double2(0, 0), S1 = S0;
#pragma unroll
                for (int e = 0; e < NB; e++) {
                    const double2 es = negate_if(ew[e], int(sg ^ sb[e]));
                    if (PURE) {
                        S0 = cadd(S0, ew[e]);
                        S1 = cadd(S1, es);
                    } else if (((xk >> e) & 1) ^ X) {  // uniform
                        S1 = cadd(S1, es);
                    } else {
                        S0 = cadd(S0, ew[e]);
                    }
                }
                add_norm(acc[2], cfma(M[0][0], S0, cmul(M[0][1], S1)));
                add_norm(acc[3], cfma(M[1][0], S0, cmul(M[1][1], S1)));
            }
        }
    }
    sweep_epilogue<4>(acc, part, ctl, epi, kWriteDirect);
}

// Entry 0 of a table set to 1 (start of a chain).
template <class S>
__global__ void table_one_kernel(S* t) { t[0] = Cx<S>::narrow(make_double2(1.0, 0.0)); }

// Two-table kernels: sweep kDirect (norm pass) or kWrite; storage 0 = complex64, 1 = complex128.
template <class S, int NKS>
void* gather_for(int sweep) {
    return sweep == kDirect ? reinterpret_cast<void*>(&gather_kernel<S, kDirect, NKS>)
                            : reinterpret_cast<void*>(&gather_kernel<S, kWrite, NKS>);
}
template <class S>
void* gather_by_nks(int sweep, int nks) {
    switch (nks) {
        case 1: return gather_for<S, 1>(sweep);
        case 2: return gather_for<S, 2>(sweep);
        case 4: return gather_for<S, 4>(sweep);
    }
    return nullptr;
}
void* gather_kernel_ptr(int storage, int sweep, int nks) {
    return storage == 0 ? gather_by_nks<float2>(sweep, nks) : gather_by_nks<double2>(sweep, nks);
}
void* table_one_kernel_ptr(int storage) {
    return storage == 0 ? reinterpret_cast<void*>(&table_one_kernel<float2>)
                        : reinterpret_cast<void*>(&table_one_kernel<double2>);
}
// Write pass of a step with nks inputs per output that folds in the next step's norms (TFold); nullptr when not built.
template <class S, int NKS>
void* fold_for(int nd2, int share, int pure) {
#define GS_FK(a, b, c) \
    if (nd2 == a && share == b && pure == c) return reinterpret_cast<void*>(&gather_fold_kernel<S, NKS, a, b != 0, c != 0>);
    GS_FK(0, 0, 1) GS_FK(0, 1, 1) GS_FK(1, 0, 0) GS_FK(1, 1, 0) GS_FK(1, 0, 1) GS_FK(1, 1, 1) GS_FK(2, 0, 0) GS_FK(2, 1, 0)
#undef GS_FK
    return nullptr;
}
template <class S>
void* fold_by_nks(int nks, int nd2, int share, int pure) {
    return nks == 1 ? fold_for<S, 1>(nd2, share, pure) : nks == 2 ? fold_for<S, 2>(nd2, share, pure)
                                                                  : fold_for<S, 4>(nd2, share, pure);
}
void* gather_fold_kernel_ptr(int storage, int nks, int nd2, int share, int pure) {
    return storage == 0 ? fold_by_nks<float2>(nks, nd2, share, pure) : fold_by_nks<double2>(nks, nd2, share, pure);
}

}  // namespace gs
