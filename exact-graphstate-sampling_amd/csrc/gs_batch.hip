// Batched scoring and adjoint: many forced strings of many plans (instances), one launch per step.
//
// The single-string engine runs one chain per stream; scoring thousands of strings that way is launch-bound on small
// steps and repeats every step's launch per string.  Here the arena of an instance holds B strings side by side,
// slot-major and batch-minor (entry (slot, b) at slot * B + b), so every gather of a coset's slot reads B consecutive
// complex numbers: coalesced whatever the plan's layout, with the string index as the wavefront lane.  Semantics are
// those of chain mode (gsamp2.cpp:56-70): one sweep per step, the branch of each lane forced by its string, outputs
// stored unnormalised, per-lane conditionals nb / (2 prev) and log2 Pr = log2(prev) - ns; the last live entry is the
// amplitude Z.
//
// One launch per step index k covers every instance with k < ns_i: the host lists work items (instance, lane group of
// 64 strings, a Gray-ordered range of 2^lg cosets) and each block takes one.  Within a block the 4 waves split the
// coset range; lane b of a wave is string group*64 + b.  Per-lane FP64 sums are reduced over the waves in LDS, then
// over the items of the (instance, lane group) by the last item to finish (agent-scope counter), in a fixed order.
// The sequence init -> steps -> finish can be captured once in a hipGraph and replayed for every batch.
//
// Adjoint.  Z = 1^T L_{ns-1} ... L_0 e_0 with L_k = w_k(0) A_k0 + w_k(1) A_k1 (w_k(x) = M_k[b_k, x]).  The gradient
// G_k(x) = dZ/dw_k(x) = lambda_k^T A_kx P_{k-1}, where P_{k-1} is the table entering step k and
// lambda_{k-1}^T = lambda_k^T L_k.  Per coset, G_k(x) += sum_tau lambda_k[out tau] A[tau][x] (the same routed signed
// slot sums as the forward sweep), and the backward butterfly writes lambda_{k-1}[slot j] =
// sum_x w(x) sign_{j,x} lambda_k[tau(j, x)] into the coset's own input slots: in place in a second arena, race free
// by the same ownership as the forward sweep.  The forward tables are needed in reverse order but the arena is
// overwritten, so the forward pass keeps compact copies ([coset][slot][lane]) of the input tables of every
// checkpoint-segment start, and of every step of the segment being back-propagated (recomputed from its checkpoint).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/gsamp_amd.h"
#include "gs_fly.h"
#include "gs_pair.h"
#include "gs_plan.h"
#include "gs_wave.h"

namespace {

using gs::flip_if;
using gs::fly_each;
using gs::fly_pair;
using gs::fly_pair_back;
using gs::fly_route_of;
using gs::FlyDesc;
using gs::make_fly;
using gs::make_pair;
using gs::uniform_byte;
using gs::pair_route0;
using gs::pair_route1;
using gs::PairDesc;
using gs::PairRegs;
using gs::PairSteps;

constexpr int kLanes = 64;           // strings per wave (one lane group)
constexpr int kWaves = 4;            // waves per block, each on its own part of the coset range
constexpr int kItemGroup = 64;       // items whose partials are reduced together before the groups are
constexpr int kBThreads = kLanes * kWaves;
constexpr int64_t kMinItems = 1024;  // work items (blocks) a step launch should have before tiles get coarser
constexpr int kMaxUnit = 3;          // most steps of one sweep
// Plans whose table fits the LDS (score_lds_kernel): most steps, log2 most slots
constexpr int kLdsSteps = 128, kLdsMaxR = 14;
constexpr int kMaxSums = 4 * kMaxUnit;   // per-lane sums of one item: the norms of its steps, or their G_k(x)

struct BStep {
    uint64_t cols[40];
    uint64_t off[4];
    uint64_t g, rhoc;
    double mre[2][2], mim[2][2];
    int nk, ntq, m;
    int tau0[4], tau1[4], par[4];
    uint32_t t0m, t1m, parm;     // tau0, tau1, par as bit masks over the offsets
};

// A step with its table in LDS at the arena's own slot numbers.  Coordinates: those first whose columns fall on different
// LDS banks.
struct LStep {
    uint32_t cols[kLdsMaxR];
    uint32_t off[4], g;
    uint32_t rho;                // sign mask over the coordinates
    uint32_t t0m, t1m, parm;     // as in BStep
    int nk, ntq, m;
    int pad[2];                  // whole 16-byte words
};
static_assert(sizeof(LStep) % 16 == 0, "the weights behind the descriptors are read as 16-byte words");

struct BItem {
    uint64_t c0;         // first coset of the range (aligned to 2^lg)
    int inst;            // instance
    int group;           // lane group (strings group*64 .. group*64+63)
    int lg;              // log2 cosets in the range
    int index;           // index of this item among the items of (inst, group)
    int count;           // number of items of (inst, group) in this step
    int pad;
};

struct BInst {           // device view of one instance
    void* mem;           // [2^R][B] forward arena
    void* lam;           // [2^R][B] adjoint arena (gradient mode)
    const BStep* steps;  // [ns]
    const PairDesc* pairs;  // [ns]: the sweep of steps k and k+1, where one is taken
    const FlyDesc* flys;    // [ns][kMaxUnit - 2]: ... of 3 steps and more from k on
    const LStep* lsteps;    // [ns]: where the plan's table fits the LDS
    const int8_t* bitsT; // [ns][B] forced bits, step-major
    double* prev;        // [B]
    int* dead;           // [B]
    double* cond;        // [B][ns]
    double* logp;        // [B]
    double* amp;         // [B][2]
    double* grad;        // [B][ns][2][2]: G_k(x) re, im (gradient mode)
    double* part;        // [lane groups][items of the step per lane group][nq][64]: the items' nq sums
    unsigned* arrived;   // [lane groups][1 + narrived]: items (or item groups), and items of each item group, finished
    int B, ns, narrived, pad;
};

// Per launch: what each instance's step sweep does besides the forward butterfly.
struct BLaunch {
    int k;
    int bookkeeping;     // 1: chain-mode conditionals / dead flags (scoring), 0: recomputation
    void* const* copy;   // [ninst] destination of a compact copy of this step's input table, or nullptr entries
    unsigned long long* clock;   // [1 + ns]: device clock at the start and after each step (latest of its reductions)
};

typedef float f2v __attribute__((ext_vector_type(2)));
typedef double d2v __attribute__((ext_vector_type(2)));

// Arena entries: raw (non-temporal) loads and stores of the storage type, widening to FP64 where used.  The arena
// pointers come from the instance table in memory, so the compiler cannot tell their address space; the accesses
// name the global address space explicitly (global instead of flat instructions).
#define GS_GLOBAL __attribute__((address_space(1)))
template <class S>
struct Sto;
template <>
struct Sto<float2> {
    static __device__ __forceinline__ float2 ld(const float2* p) {
        const f2v t = __builtin_nontemporal_load((const GS_GLOBAL f2v*)(p));
        return make_float2(t.x, t.y);
    }
    static __device__ __forceinline__ void st(float2* p, float2 v) {
        const f2v t = {v.x, v.y};
        __builtin_nontemporal_store(t, (GS_GLOBAL f2v*)(p));
    }
    // entry i of a wave-uniform row
    static __device__ __forceinline__ float2 ld(const float2* row, int i) { return ld(row + i); }
    static __device__ __forceinline__ void st(float2* row, int i, float2 v) { st(row + i, v); }
    static __device__ __forceinline__ double2 wide(float2 v) { return make_double2(v.x, v.y); }
    static __device__ __forceinline__ float2 narrow(double2 v) { return make_float2(float(v.x), float(v.y)); }
};
template <>
struct Sto<double2> {
    static __device__ __forceinline__ double2 ld(const double2* p) {
        const d2v t = __builtin_nontemporal_load((const GS_GLOBAL d2v*)(p));
        return make_double2(t.x, t.y);
    }
    static __device__ __forceinline__ void st(double2* p, double2 v) {
        const d2v t = {v.x, v.y};
        __builtin_nontemporal_store(t, (GS_GLOBAL d2v*)(p));
    }
    static __device__ __forceinline__ double2 ld(const double2* row, int i) { return ld(row + i); }
    static __device__ __forceinline__ void st(double2* row, int i, double2 v) { st(row + i, v); }
    static __device__ __forceinline__ double2 wide(double2 v) { return v; }
    static __device__ __forceinline__ double2 narrow(double2 v) { return v; }
};
// Kernels are instantiated per storage S, NQ (the most slots per coset among the instances' step k: 1, 2 or 4) and
// LU (log2 cosets a lane gathers at once: 2^LU * NQ loads in flight per lane).

__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 cneg(double2 a) { return make_double2(-a.x, -a.y); }
__device__ __forceinline__ double2 cfma(double2 a, double2 b, double2 c) {
    return make_double2(fma(a.x, b.x, fma(-a.y, b.y, c.x)), fma(a.x, b.y, fma(a.y, b.x, c.y)));
}
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(fma(a.x, b.x, -a.y * b.y), fma(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ double norm2(double2 a) { return fma(a.x, a.x, a.y * a.y); }

// The step's coordinate columns in LDS, for the whole block (the Gray walk reads one per coset group; read through
// the instance table in memory, each would be a dependent memory round trip).  Every thread of the block calls it.
__device__ __forceinline__ const uint64_t* lds_cols(const uint64_t* __restrict__ cols, int nk, uint64_t* sc) {
    for (int j = threadIdx.x; j < nk; j += blockDim.x) sc[j] = cols[j];
    __syncthreads();
    return sc;
}

// Coset range of this wave: 2^lsub cosets c = cstart | (gray(t) << lu) | u, t < 2^(lsub - lu), u < 2^lu with
// lu = min(LU, lsub): binary inside a group of 2^lu cosets, whose bases are base(t) ^ ubase[u] (all gathered at once),
// Gray-ordered across groups, so the next group's base is one XOR away.
template <int LU>
struct Walk {
    static constexpr int U = 1 << LU;
    uint64_t cstart, base;    // base of cstart | (gray(t) << lu)
    int pc, lsub, lu;
    bool on;
    uint64_t ubase[U];
    int upc[U];
    __device__ Walk(const BItem& it, const uint64_t* __restrict__ cols, uint64_t rhoc, int nk, int wave) {
        const int lw = it.lg >= 2 ? 2 : it.lg;
        on = wave < (1 << lw);
        lsub = it.lg - lw;
        cstart = it.c0 | (uint64_t(wave) << lsub);
        base = 0;
        pc = 0;
        for (int j = lsub; j < nk; j++)
            if ((cstart >> j) & 1) {
                base ^= cols[j];
                pc ^= int((rhoc >> j) & 1);
            }
        lu = lsub < LU ? lsub : LU;
#pragma unroll
        for (int u = 0; u < U; u++) {
            uint64_t a = 0;
            int p = 0;
#pragma unroll
            for (int j = 0; j < LU; j++)
                if (j < lu && ((u >> j) & 1)) {
                    a ^= cols[j];
                    p ^= int((rhoc >> j) & 1);
                }
            ubase[u] = a;
            upc[u] = p;
        }
    }
    __device__ uint64_t groups() const { return on ? uint64_t(1) << (lsub - lu) : 0; }
    __device__ bool valid(int u) const { return u < (1 << lu); }
    __device__ int own(int u) const { return u & ((1 << lu) - 1); }   // the coset whose addresses ubase[u] repeats
    __device__ void next(const uint64_t* __restrict__ cols, uint64_t rhoc, uint64_t t) {   // to group t >= 1
        const int j = lu + __builtin_ctzll(t);
        base ^= cols[j];
        pc ^= int((rhoc >> j) & 1);
    }
    __device__ uint64_t coset(uint64_t t, int u) const { return cstart | ((t ^ (t >> 1)) << lu) | uint64_t(u); }
};

// End of an item: its per-lane sums (over the block's waves, in order) become its partial, and the last item of its
// (instance, lane group) to finish adds up the partials in a fixed order and ends the sweep of STEPS steps from step k
// for those 64 lanes: chain1 bookkeeping (GRAD false: cond, prev, dead; gsamp2.cpp:67) or the gradient entries G_k.
// With more than 2 kItemGroup items the last item of each kItemGroup consecutive ones reduces those first.  Partials are
// published by atomic exchanges, which take effect where the counter does, before the counter is raised: no release
// fence (each would write back the XCD's L2), and no reduction launches, which cost 8-20 us per step against the
// 2-4 us an item's last block needs.
template <int NQ>
__device__ __forceinline__ void add_partials(const double* from, int n, size_t stride, int wave, int lane,
                                             double (&sh)[kWaves][NQ][kLanes]) {
    double tot[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) tot[q] = 0;
    for (int i = wave; i < n; i += kWaves)
#pragma unroll
        for (int q = 0; q < NQ; q++)
            tot[q] += __hip_atomic_load(from + size_t(i) * stride + q * kLanes + lane, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();                                       // sh may still be read
#pragma unroll
    for (int q = 0; q < NQ; q++) sh[wave][q][lane] = tot[q];
    __syncthreads();
}

template <int STEPS, bool GRAD>
__device__ void item_end(const BInst& I, const BItem& it, int k, int wave, int lane,
                         const double (&v)[STEPS * (GRAD ? 4 : 1)], unsigned long long* clock) {
    constexpr int NQ = STEPS * (GRAD ? 4 : 1);
    __shared__ double sh[kWaves][NQ][kLanes];
    __shared__ int s_last;
#pragma unroll
    for (int q = 0; q < NQ; q++) sh[wave][q][lane] = v[q];
    __syncthreads();
    const size_t stride = NQ * kLanes;
    double* part = I.part + size_t(it.group) * size_t(it.count) * stride;
    unsigned* total = I.arrived + size_t(it.group) * (1 + I.narrived);
    // wave w adds up sums w, w + 4, ... of the block and publishes them at `to`; thread 0 then raises the counter: true
    // for the block that makes it n
    auto publish = [&](double* to, unsigned* counter, unsigned n) {
        unsigned long long old = 0;
#pragma unroll
        for (int q0 = 0; q0 < NQ; q0 += kWaves) {
            const int q = q0 + wave;
            if (q >= NQ) break;
            double t = sh[0][q][lane];
#pragma unroll
            for (int w = 1; w < kWaves; w++) t += sh[w][q][lane];
            old |= __hip_atomic_exchange(reinterpret_cast<unsigned long long*>(to + q * kLanes + lane),
                                         (unsigned long long)__double_as_longlong(t), __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
        }
        asm volatile("s_waitcnt vmcnt(0)" : "+v"(old) : : "memory");           // every exchange has returned
        __syncthreads();
        if (threadIdx.x == 0)
            s_last = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n - 1;
        __syncthreads();
        if (!s_last) return false;
        __atomic_thread_fence(__ATOMIC_ACQUIRE);
        if (threadIdx.x == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return true;
    };
    if (it.count > 1) {
        double* mine = part + size_t(it.index) * stride;
        if (it.count <= 2 * kItemGroup) {
            if (!publish(mine, total, unsigned(it.count))) return;
            add_partials<NQ>(part, it.count, stride, wave, lane, sh);
        } else {                                           // a power of two, as kItemGroup
            const int g = it.index / kItemGroup;
            double* first = part + size_t(g) * kItemGroup * stride;
            if (!publish(mine, total + 1 + g, unsigned(kItemGroup))) return;
            add_partials<NQ>(first, kItemGroup, stride, wave, lane, sh);
            if (!publish(first, total, unsigned(it.count / kItemGroup))) return;
            add_partials<NQ>(part, it.count / kItemGroup, kItemGroup * stride, wave, lane, sh);
        }
    }
    if (wave != 0) return;
    double tot[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        tot[q] = sh[0][q][lane];
#pragma unroll
        for (int w = 1; w < kWaves; w++) tot[q] += sh[w][q][lane];
    }
    const int b = it.group * kLanes + lane, ns = I.ns;
    if constexpr (GRAD) {
#pragma unroll
        for (int q = 0; q < NQ; q++) I.grad[(size_t(b) * ns + k) * 4 + q] = tot[q];
    } else {
        double prev = I.prev[b];
        bool dead = I.dead[b] != 0;
#pragma unroll
        for (int j = 0; j < STEPS; j++) {
            if (dead) break;
            I.cond[size_t(b) * ns + k + j] = tot[j] / (2 * prev);
            prev = tot[j];
            if (prev <= 0) {
                for (int q = k + j; q < ns; q++) I.cond[size_t(b) * ns + q] = 0;
                I.dead[b] = 1;
                dead = true;
            }
        }
        I.prev[b] = prev;
    }
    if (clock && lane == 0) atomicMax(clock + 1 + k, (unsigned long long)wall_clock64());
}

// The fields of a step that the inner loops use, copied to registers once per block (read through a reference to
// global memory, they would be reloaded after every arena store the compiler cannot prove disjoint from them).
struct SR {
    uint64_t off[4], g, rhoc;
    int ntq, m;
    int tau0[4], tau1[4], par[4];
    __device__ explicit SR(const BStep& s) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            off[q] = s.off[q];
            tau0[q] = s.tau0[q];
            tau1[q] = s.tau1[q];
            par[q] = s.par[q];
        }
        g = s.g;
        rhoc = s.rhoc;
        ntq = s.ntq;
        m = s.m;
    }
};

// Routed signed slot sums A[tau][x] of one coset from its ntq slot values (ntq = NQ at compile time in the EX
// variants, which have no branch on it).
template <int NQ>
__device__ __forceinline__ void route(const SR& s, const double2 (&v)[NQ], int pc, int ntq, double2 (&A)[2][2]) {
    A[0][0] = A[0][1] = A[1][0] = A[1][1] = make_double2(-0.0, -0.0);   // x + (-0.0) = x: the first add folds away
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        if (q >= ntq) break;
        const double2 w = v[q];
        const double2 ws = (pc ^ s.par[q]) ? cneg(w) : w;
        if (s.tau0[q]) A[1][0] = cadd(A[1][0], w); else A[0][0] = cadd(A[0][0], w);   // uniform branches
        if (s.tau1[q]) A[1][1] = cadd(A[1][1], ws); else A[0][1] = cadd(A[0][1], ws);
    }
}

template <class S, int NQ, int LU, bool EX>
__global__ __launch_bounds__(kBThreads) void batch_step_kernel(const BInst* __restrict__ insts,
                                                               const BItem* __restrict__ items, BLaunch L) {
    const BItem it = items[blockIdx.x];
    const BInst& I = insts[it.inst];
    const int k = L.k;
    const BStep& s = I.steps[k];
    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = threadIdx.x / kLanes;
    const int B = I.B;
    const int b = it.group * kLanes + lane;
    const int bv = I.bitsT[size_t(k) * B + b];
    const double2 w0 = make_double2(s.mre[bv][0], s.mim[bv][0]);
    const double2 w1 = make_double2(s.mre[bv][1], s.mim[bv][1]);
    S* __restrict__ mem = static_cast<S*>(I.mem);
    S* __restrict__ cp = L.copy ? static_cast<S*>(L.copy[it.inst]) : nullptr;
    double nb = 0;
    constexpr int U = 1 << LU;
    const SR r(s);
    __shared__ uint64_t scols[40];
    const uint64_t* cols = lds_cols(s.cols, s.nk, scols);
    Walk<LU> wk(it, cols, r.rhoc, s.nk, wave);
    const uint64_t ng = wk.groups();
    const int ntq = EX ? NQ : r.ntq;                      // EX: every instance has NQ slots at this step
    for (uint64_t t = 0; t < ng; t++) {
        if (t) wk.next(cols, r.rhoc, t);
        S v[U][NQ];
        // Every load of the group first, and unconditionally: slots beyond this instance's ntq re-read slot 0, and the
        // cosets u >= 2^lu of a short range re-read coset u mod 2^lu (ubase keeps only the low lu bits of u); both are
        // discarded.  Loads (or their only uses) under branches leave a load possibly in flight at the loop latch,
        // and the next group's load into the same registers then waits for all but the newest memory operation.
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int q = 0; q < NQ; q++)
                v[u][q] = Sto<S>::ld(mem + (wk.base ^ wk.ubase[u] ^ (q < ntq ? r.off[q] : 0)) * B + b);
        if (cp)
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int q = 0; q < NQ; q++)
                    if (q < ntq && wk.valid(u)) Sto<S>::st(cp + (wk.coset(t, u) * ntq + q) * B + b, v[u][q]);
#pragma unroll
        for (int u = 0; u < U; u++) {
            double2 vw[NQ];
#pragma unroll
            for (int q = 0; q < NQ; q++) vw[q] = q < ntq ? Sto<S>::wide(v[u][q]) : make_double2(0, 0);
            double2 A[2][2];
            route(r, vw, wk.pc ^ wk.upc[u], ntq, A);
            const uint64_t a0 = wk.base ^ wk.ubase[u];
            const double2 o0 = cfma(w0, A[0][0], cmul(w1, A[0][1]));
            const double2 o1 = cfma(w0, A[1][0], cmul(w1, A[1][1]));
            if (!wk.valid(u)) continue;                     // stores and norms of the lane's own cosets only
            Sto<S>::st(mem + a0 * B + b, Sto<S>::narrow(o0));
            nb += norm2(o0);
            if (r.m == 2) {
                Sto<S>::st(mem + (a0 ^ r.g) * B + b, Sto<S>::narrow(o1));
                nb += norm2(o1);
            }
        }
    }
    if (!L.bookkeeping) return;
    const double val[1] = {nb};
    item_end<1, false>(I, it, k, wave, lane, val, L.clock);
}

// Put a compact copy of step k's input table back into the forward arena (restart of a checkpoint segment).
template <class S, int NQ, int LU, bool EX>
__global__ __launch_bounds__(kBThreads) void batch_restore_kernel(const BInst* __restrict__ insts,
                                                                  const BItem* __restrict__ items, BLaunch L) {
    const BItem it = items[blockIdx.x];
    const BInst& I = insts[it.inst];
    const BStep& s = I.steps[L.k];
    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = threadIdx.x / kLanes;
    const int B = I.B;
    const int b = it.group * kLanes + lane;
    S* __restrict__ mem = static_cast<S*>(I.mem);
    const S* __restrict__ cp = static_cast<const S*>(L.copy[it.inst]);
    if (!cp) return;
    constexpr int U = 1 << LU;
    const SR r(s);
    __shared__ uint64_t scols[40];
    const uint64_t* cols = lds_cols(s.cols, s.nk, scols);
    Walk<LU> wk(it, cols, r.rhoc, s.nk, wave);
    const uint64_t ng = wk.groups();
    const int ntq = EX ? NQ : r.ntq;                      // EX: every instance has NQ slots at this step
    for (uint64_t t = 0; t < ng; t++) {
        if (t) wk.next(cols, r.rhoc, t);
        S v[U][NQ];
        // No branches around the loads or their uses (see batch_step_kernel): a coset u >= 2^lu of a short range is
        // coset u mod 2^lu, whose value it copies to the same address again.
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int q = 0; q < NQ; q++)
                if (q < ntq) v[u][q] = Sto<S>::ld(cp + (wk.coset(t, wk.own(u)) * ntq + q) * B + b);
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int q = 0; q < NQ; q++)
                if (q < ntq) Sto<S>::st(mem + (wk.base ^ wk.ubase[u] ^ r.off[q]) * B + b, v[u][q]);
    }
}

// Backward step k: lambda_k (adjoint arena, at the coset's outputs) and the compact copy of P_{k-1} give
// G_k(x) += sum_tau lambda[tau] A[tau][x]; lambda_{k-1} goes to the coset's input slots.
template <class S, int NQ, int LU, bool EX>
__global__ __launch_bounds__(kBThreads) void batch_back_kernel(const BInst* __restrict__ insts,
                                                               const BItem* __restrict__ items, BLaunch L) {
    const BItem it = items[blockIdx.x];
    const BInst& I = insts[it.inst];
    const int k = L.k;
    const BStep& s = I.steps[k];
    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = threadIdx.x / kLanes;
    const int B = I.B;
    const int b = it.group * kLanes + lane;
    const int bv = I.bitsT[size_t(k) * B + b];
    const double2 w0 = make_double2(s.mre[bv][0], s.mim[bv][0]);
    const double2 w1 = make_double2(s.mre[bv][1], s.mim[bv][1]);
    S* __restrict__ lam = static_cast<S*>(I.lam);
    const S* __restrict__ cp = static_cast<const S*>(L.copy[it.inst]);
    double2 g0 = make_double2(0, 0), g1 = g0;
    constexpr int U = 1 << LU;
    const SR r(s);
    __shared__ uint64_t scols[40];
    const uint64_t* cols = lds_cols(s.cols, s.nk, scols);
    Walk<LU> wk(it, cols, r.rhoc, s.nk, wave);
    const uint64_t ng = wk.groups();
    const int ntq = EX ? NQ : r.ntq;                      // EX: every instance has NQ slots at this step
    for (uint64_t t = 0; t < ng; t++) {
        if (t) wk.next(cols, r.rhoc, t);
        S v[U][NQ], l0[U], l1[U];
        // Every load of the group first, with no branches around the loads or their uses (see batch_step_kernel): a
        // coset u >= 2^lu of a short range reads coset u mod 2^lu and only its stores and gradient terms are dropped;
        // a one-output step (g = 0) reads its output slot twice.
        const uint64_t gq = r.m == 2 ? r.g : 0;
#pragma unroll
        for (int u = 0; u < U; u++) {
            const uint64_t a0 = wk.base ^ wk.ubase[u];
#pragma unroll
            for (int q = 0; q < NQ; q++)
                if (q < ntq) v[u][q] = Sto<S>::ld(cp + (wk.coset(t, wk.own(u)) * ntq + q) * B + b);
            l0[u] = Sto<S>::ld(lam + a0 * B + b);
            l1[u] = Sto<S>::ld(lam + (a0 ^ gq) * B + b);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const uint64_t a0 = wk.base ^ wk.ubase[u];
            const int pc = wk.pc ^ wk.upc[u];
            double2 vw[NQ];
#pragma unroll
            for (int q = 0; q < NQ; q++) vw[q] = q < ntq ? Sto<S>::wide(v[u][q]) : make_double2(0, 0);
            double2 A[2][2];
            route(r, vw, pc, ntq, A);
            const double2 m0 = Sto<S>::wide(l0[u]);
            const double2 m1 = r.m == 2 ? Sto<S>::wide(l1[u]) : make_double2(0, 0);
            double2 h0 = cfma(m0, A[0][0], g0);
            double2 h1 = cfma(m0, A[0][1], g1);
            if (r.m == 2) {
                h0 = cfma(m1, A[1][0], h0);
                h1 = cfma(m1, A[1][1], h1);
            }
            if (!wk.valid(u)) continue;                     // gradient terms and stores of the lane's own cosets only
            g0 = h0;
            g1 = h1;
#pragma unroll
            for (int q = 0; q < NQ; q++) {
                if (q >= ntq) break;
                const double2 lt0 = r.tau0[q] ? m1 : m0;
                const double2 lt1 = r.tau1[q] ? m1 : m0;
                const double2 x1 = cmul(w1, lt1);
                const double2 out = cfma(w0, lt0, (pc ^ r.par[q]) ? cneg(x1) : x1);
                Sto<S>::st(lam + (a0 ^ r.off[q]) * B + b, Sto<S>::narrow(out));
            }
        }
    }
    const double val[4] = {g0.x, g0.y, g1.x, g1.y};
    item_end<1, true>(I, it, k, wave, lane, val, nullptr);
}

// ---- two steps per sweep (PairDesc)
//
// A single step's sweep is bound by HBM: it reads and writes one table (n = 70 band 26, 64 lanes, 2^22 cosets: 4.3 GB
// in 0.85 ms, 5.0 TB/s) and its FP64 work takes a quarter of that time.  Two steps in one sweep move the same bytes
// once instead of twice.  Everything that depends on the super-coset alone (addresses, signs, slot indices) is
// wave-uniform and kept in scalar registers; a lane holds the NI * NQ inputs of its string.  The table between the
// steps is rounded to the storage type in registers, so the results are the single steps' bit for bit up to the order
// of the FP64 sums over the cosets.
__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
    return (uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(v >> 32)))) << 32) |
           uint32_t(__builtin_amdgcn_readfirstlane(int(v)));
}
// Super-cosets a wave gathers at once: about 8 loads in flight per lane for 8-byte entries, 4 for 16-byte ones.
template <class S>
constexpr int pair_lu(int loads) {
    const int most = sizeof(S) == 8 ? 8 : 4;
    return loads * 4 <= most ? 2 : loads * 2 <= most ? 1 : 0;
}

// The super-cosets of one wave (as Walk, with uniform state): U at a time, Gray-ordered groups.
template <int LU>
struct PairWalk {
    static constexpr int U = 1 << LU;
    const uint64_t* cols;                     // in LDS
    const int* pn;
    uint64_t cstart, base, ubase[U];
    uint32_t p, up[U];
    int lsub, lu;
    bool on;
    __device__ __forceinline__ uint64_t col(int j) const { return uniform64(cols[j]); }
    __device__ __forceinline__ uint32_t nib(int j) const { return uint32_t(__builtin_amdgcn_readfirstlane(pn[j])); }
    template <class Desc>
    __device__ PairWalk(const BItem& it, const Desc& P, uint64_t* scols, int* spn, int wave) : cols(scols), pn(spn) {
        for (int j = threadIdx.x; j < P.nk; j += blockDim.x) {
            scols[j] = P.cols[j];
            spn[j] = P.pn[j];
        }
        __syncthreads();
        const int lw = it.lg >= 2 ? 2 : it.lg;
        on = wave < (1 << lw);
        lsub = it.lg - lw;
        cstart = it.c0 | (uint64_t(wave) << lsub);
        base = 0;
        p = 0;
        for (int j = lsub; j < P.nk; j++)
            if ((cstart >> j) & 1) {
                base ^= col(j);
                p ^= nib(j);
            }
        lu = lsub < LU ? lsub : LU;
#pragma unroll
        for (int u = 0; u < U; u++) {
            ubase[u] = 0;
            up[u] = 0;
#pragma unroll
            for (int j = 0; j < LU; j++)
                if (j < lu && ((u >> j) & 1)) {
                    ubase[u] ^= col(j);
                    up[u] ^= nib(j);
                }
        }
    }
    __device__ uint64_t groups() const { return on ? uint64_t(1) << (lsub - lu) : 0; }
    __device__ bool valid(int u) const { return u < (1 << lu); }
    __device__ int own(int u) const { return u & ((1 << lu) - 1); }
    __device__ void next(uint64_t t) {
        const int j = lu + __builtin_ctzll(t);
        base ^= col(j);
        p ^= nib(j);
    }
    __device__ uint64_t index(uint64_t t, int u) const { return cstart | ((t ^ (t >> 1)) << lu) | uint64_t(u); }
};

__device__ __forceinline__ PairSteps pair_steps(const BStep& s0, const BStep& s1) {
    return PairSteps{s0.off, s1.g, s1.m, s0.t0m, s0.t1m, s0.parm, s1.t0m, s1.t1m, s1.parm};
}

template <class S, int NQ, int NI, int MO, bool DEG>
__global__ __launch_bounds__(kBThreads) void pair_step_kernel(const BInst* __restrict__ insts,
                                                              const BItem* __restrict__ items, BLaunch L) {
    constexpr int NU = DEG ? 1 : MO, LU = pair_lu<S>(NI * NQ), U = 1 << LU;
    const BItem it = items[blockIdx.x];
    const BInst& I = insts[it.inst];
    const int k = L.k;
    const BStep& s0 = I.steps[k];
    const BStep& s1 = I.steps[k + 1];
    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes);
    const int B = I.B;
    const int b = it.group * kLanes + lane;
    const int b0 = I.bitsT[size_t(k) * B + b], b1 = I.bitsT[size_t(k + 1) * B + b];
    const double2 w0 = make_double2(s0.mre[b0][0], s0.mim[b0][0]), w1 = make_double2(s0.mre[b0][1], s0.mim[b0][1]);
    const double2 x0 = make_double2(s1.mre[b1][0], s1.mim[b1][0]), x1 = make_double2(s1.mre[b1][1], s1.mim[b1][1]);
    S* __restrict__ mem = static_cast<S*>(I.mem);
    S* __restrict__ cp = L.copy ? static_cast<S*>(L.copy[it.inst]) : nullptr;
    const PairRegs r(I.pairs[k], pair_steps(s0, s1));
    __shared__ uint64_t scols[40];
    __shared__ int spn[40];
    PairWalk<LU> wk(it, I.pairs[k], scols, spn, wave);
    const uint64_t ng = wk.groups();
    double nb[2] = {0, 0};
    for (uint64_t t = 0; t < ng; t++) {
        if (t) wk.next(t);
        S v[U][NI][NQ];
        // every load first and unconditionally (see batch_step_kernel): super-cosets u >= 2^lu of a short range repeat
        // the ones before them and are discarded
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int i = 0; i < NI; i++)
#pragma unroll
                for (int q = 0; q < NQ; q++)
                    v[u][i][q] = Sto<S>::ld(mem + (wk.base ^ wk.ubase[u] ^ r.lab[i] ^ r.off[q]) * B + b);
        if (cp)
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int i = 0; i < NI; i++)
#pragma unroll
                    for (int q = 0; q < NQ; q++)
                        if (wk.valid(u)) Sto<S>::st(cp + ((wk.index(t, u) * NI + i) * NQ + q) * B + b, v[u][i][q]);
#pragma unroll
        for (int u = 0; u < U; u++) {
            const uint32_t pa = wk.p ^ wk.up[u];
            const uint64_t a = wk.base ^ wk.ubase[u];
            const bool mine = wk.valid(u);
            double2 e[NI][MO];
#pragma unroll
            for (int i = 0; i < NI; i++) {
                double2 A[2][2];
                pair_route0<S, NQ>(r, v[u][i], pa, i, A);
#pragma unroll
                for (int m = 0; m < MO; m++) {
                    const double2 o = cfma(w0, A[m][0], cmul(w1, A[m][1]));
                    if (mine) nb[0] += norm2(o);
                    e[i][m] = Sto<S>::wide(Sto<S>::narrow(o));
                }
            }
#pragma unroll
            for (int c = 0; c < NU; c++) {
                double2 A[2][2];
                pair_route1<NI, MO, DEG>(r, e, pa, pa, c, A);
                const double2 f0 = cfma(x0, A[0][0], cmul(x1, A[0][1]));
                const double2 f1 = cfma(x0, A[1][0], cmul(x1, A[1][1]));
                if (!mine) continue;
                const uint64_t at = r.out(a, pa, c);
                Sto<S>::st(mem + at * B + b, Sto<S>::narrow(f0));
                nb[1] += norm2(f0);
                if (r.m1 == 2) {
                    Sto<S>::st(mem + (at ^ r.g1) * B + b, Sto<S>::narrow(f1));
                    nb[1] += norm2(f1);
                }
            }
        }
    }
    if (!L.bookkeeping) return;
    item_end<2, false>(I, it, k, wave, lane, nb, L.clock);
}

// Put a compact copy of a pair's input table back into the forward arena.
template <class S, int NQ, int NI, int MO, bool DEG>
__global__ __launch_bounds__(kBThreads) void pair_restore_kernel(const BInst* __restrict__ insts,
                                                                 const BItem* __restrict__ items, BLaunch L) {
    constexpr int LU = pair_lu<S>(NI * NQ), U = 1 << LU;
    const BItem it = items[blockIdx.x];
    const BInst& I = insts[it.inst];
    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes);
    const int B = I.B;
    const int b = it.group * kLanes + lane;
    S* __restrict__ mem = static_cast<S*>(I.mem);
    const S* __restrict__ cp = static_cast<const S*>(L.copy[it.inst]);
    if (!cp) return;
    const PairRegs r(I.pairs[L.k], pair_steps(I.steps[L.k], I.steps[L.k + 1]));
    __shared__ uint64_t scols[40];
    __shared__ int spn[40];
    PairWalk<LU> wk(it, I.pairs[L.k], scols, spn, wave);
    const uint64_t ng = wk.groups();
    for (uint64_t t = 0; t < ng; t++) {
        if (t) wk.next(t);
        S v[U][NI][NQ];
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int i = 0; i < NI; i++)
#pragma unroll
                for (int q = 0; q < NQ; q++)
                    v[u][i][q] = Sto<S>::ld(cp + ((wk.index(t, wk.own(u)) * NI + i) * NQ + q) * B + b);
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int i = 0; i < NI; i++)
#pragma unroll
                for (int q = 0; q < NQ; q++)
                    Sto<S>::st(mem + (wk.base ^ wk.ubase[u] ^ r.lab[i] ^ r.off[q]) * B + b, v[u][i][q]);
    }
}

// Backward through both steps: the copy of step k's input gives the table between them again (in registers), lambda
// goes from step k+1's outputs to step k's inputs, and both gradients are summed.
template <class S, int NQ, int NI, int MO, bool DEG>
__global__ __launch_bounds__(kBThreads) void pair_back_kernel(const BInst* __restrict__ insts,
                                                              const BItem* __restrict__ items, BLaunch L) {
    constexpr int NU = DEG ? 1 : MO, LU = pair_lu<S>(NI * NQ + 2 * NU), U = 1 << LU;
    const BItem it = items[blockIdx.x];
    const BInst& I = insts[it.inst];
    const int k = L.k;
    const BStep& s0 = I.steps[k];
    const BStep& s1 = I.steps[k + 1];
    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes);
    const int B = I.B;
    const int b = it.group * kLanes + lane;
    const int b0 = I.bitsT[size_t(k) * B + b], b1 = I.bitsT[size_t(k + 1) * B + b];
    const double2 w0 = make_double2(s0.mre[b0][0], s0.mim[b0][0]), w1 = make_double2(s0.mre[b0][1], s0.mim[b0][1]);
    const double2 x0 = make_double2(s1.mre[b1][0], s1.mim[b1][0]), x1 = make_double2(s1.mre[b1][1], s1.mim[b1][1]);
    S* __restrict__ lam = static_cast<S*>(I.lam);
    const S* __restrict__ cp = static_cast<const S*>(L.copy[it.inst]);
    const PairRegs r(I.pairs[k], pair_steps(s0, s1));
    const uint64_t gq = r.m1 == 2 ? r.g1 : 0;
    __shared__ uint64_t scols[40];
    __shared__ int spn[40];
    PairWalk<LU> wk(it, I.pairs[k], scols, spn, wave);
    const uint64_t ng = wk.groups();
    double2 ga[2] = {make_double2(0, 0), make_double2(0, 0)}, gb[2] = {ga[0], ga[0]};   // G_k(x), G_{k+1}(x)
    for (uint64_t t = 0; t < ng; t++) {
        if (t) wk.next(t);
        S v[U][NI][NQ], l2[U][NU][2];
#pragma unroll
        for (int u = 0; u < U; u++) {
#pragma unroll
            for (int i = 0; i < NI; i++)
#pragma unroll
                for (int q = 0; q < NQ; q++)
                    v[u][i][q] = Sto<S>::ld(cp + ((wk.index(t, wk.own(u)) * NI + i) * NQ + q) * B + b);
#pragma unroll
            for (int c = 0; c < NU; c++) {
                const uint64_t at = r.out(wk.base ^ wk.ubase[u], wk.p ^ wk.up[u], c);
                l2[u][c][0] = Sto<S>::ld(lam + at * B + b);
                l2[u][c][1] = Sto<S>::ld(lam + (at ^ gq) * B + b);     // a one-output step reads its output twice
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const uint32_t pa = wk.p ^ wk.up[u];
            const uint64_t a = wk.base ^ wk.ubase[u];
            double2 e[NI][MO], l1[NI][MO];
            double2 ha[2] = {ga[0], ga[1]}, hb[2] = {gb[0], gb[1]};
#pragma unroll
            for (int i = 0; i < NI; i++) {
                double2 A[2][2];
                pair_route0<S, NQ>(r, v[u][i], pa, i, A);
#pragma unroll
                for (int m = 0; m < MO; m++)
                    e[i][m] = Sto<S>::wide(Sto<S>::narrow(cfma(w0, A[m][0], cmul(w1, A[m][1]))));
            }
#pragma unroll
            for (int c = 0; c < NU; c++) {
                double2 A[2][2];
                pair_route1<NI, MO, DEG>(r, e, pa, pa, c, A);
                const double2 m0 = Sto<S>::wide(l2[u][c][0]);
                const double2 m1 = r.m1 == 2 ? Sto<S>::wide(l2[u][c][1]) : make_double2(0, 0);
#pragma unroll
                for (int x = 0; x < 2; x++) {
                    hb[x] = cfma(m0, A[0][x], hb[x]);
                    if (r.m1 == 2) hb[x] = cfma(m1, A[1][x], hb[x]);
                }
                const double2 y0 = cmul(x1, m0), y1 = cmul(x1, m1);
                const uint32_t sg = r.sign(pa, c);
#pragma unroll
                for (int i = 0; i < NI; i++)
#pragma unroll
                    for (int m = 0; m < MO; m++) {
                        if (!DEG && m != c) continue;
                        const uint32_t j = r.slot(pa, i, m);
                        const double2 lt = ((r.u0m >> j) & 1) ? m1 : m0;
                        const double2 y = ((r.u1m >> j) & 1) ? y1 : y0;
                        l1[i][m] = Sto<S>::wide(Sto<S>::narrow(cfma(x0, lt, flip_if(y, sg ^ ((r.uparm >> j) & 1)))));
                    }
            }
#pragma unroll
            for (int i = 0; i < NI; i++) {
                double2 A[2][2];
                pair_route0<S, NQ>(r, v[u][i], pa, i, A);
#pragma unroll
                for (int x = 0; x < 2; x++)
#pragma unroll
                    for (int m = 0; m < MO; m++) ha[x] = cfma(l1[i][m], A[m][x], ha[x]);
            }
            if (!wk.valid(u)) continue;             // gradient terms and stores of the wave's own super-cosets only
#pragma unroll
            for (int x = 0; x < 2; x++) {
                ga[x] = ha[x];
                gb[x] = hb[x];
            }
#pragma unroll
            for (int i = 0; i < NI; i++) {
                const uint32_t pc = (pa ^ r.pd[i]) & 1, sw = (r.pd[i] >> 4) & 1;
#pragma unroll
                for (int q = 0; q < NQ; q++) {
                    const uint32_t t0 = ((r.t0m >> q) & 1) ^ sw, t1 = ((r.t1m >> q) & 1) ^ sw;
                    const double2 m0 = MO == 2 && t0 ? l1[i][MO - 1] : l1[i][0];
                    const double2 m1 = MO == 2 && t1 ? l1[i][MO - 1] : l1[i][0];
                    const double2 out = cfma(w0, m0, flip_if(cmul(w1, m1), pc ^ ((r.parm >> q) & 1)));
                    Sto<S>::st(lam + (a ^ r.lab[i] ^ r.off[q]) * B + b, Sto<S>::narrow(out));
                }
            }
        }
    }
    const double val[8] = {ga[0].x, ga[0].y, ga[1].x, ga[1].y, gb[0].x, gb[0].y, gb[1].x, gb[1].y};
    item_end<2, true>(I, it, k, wave, lane, val, nullptr);
}

// ---- three steps and more per sweep (FlyDesc): a run of butterfly steps, whose outputs take the places of their slots
//
// A lane holds the 2^NS entries of a group of its string; addresses, signs and slot indices are wave-uniform (the fields
// are made so by hand: bytes and loads through the instance table land in vector registers, and with them the routes
// became divergent branches and a step took 168 VGPRs instead of 128).  The pairs' saving goes on: 64 strings of the
// n = 70 band 26 instance, which has 17 such steps in a row, take 18.2 ms instead of 24.6, 128 gradients of n = 60
// band 24 11.8 ms instead of 16.0.  Sixteen entries (four steps) and their weights take 290 VGPRs.
template <int NS>
struct FlyGroup {
    static constexpr int NE = 1 << NS;
    uint64_t de[NE];                          // entries relative to the group's base, and their parities
    uint32_t pe[NE];
    int route[NS];
    uint32_t par[NS];
    __device__ explicit FlyGroup(const FlyDesc& f) {
#pragma unroll
        for (int i = 0; i < NS; i++) {
            route[i] = int(uniform_byte(f.route[i]));
            par[i] = uniform_byte(f.par[i]);
        }
#pragma unroll
        for (int e = 0; e < NE; e++) {
            de[e] = 0;
            pe[e] = uniform_byte(f.cn);
#pragma unroll
            for (int i = 0; i < NS; i++)
                if ((e >> i) & 1) {
                    de[e] ^= uniform64(f.dir[i]);
                    pe[e] ^= uniform_byte(f.dn[i]);
                }
        }
    }
    __device__ uint32_t slot(uint32_t p, int e, int i) const { return ((p ^ pe[e]) >> (4 + i)) & 1; }
    __device__ uint32_t sign(uint32_t p, int e, int i) const { return ((p ^ pe[e]) >> i) & 1; }
};

template <class S, int NS, int I>
__device__ __forceinline__ void fly_step(const FlyGroup<NS>& g, uint32_t p, const double2 (&w)[2], const S (&x)[1 << NS],
                                         S (&y)[1 << NS], double& nb) {
    fly_route_of(g.route[I], [&](auto r) {
#pragma unroll
        for (int e = 0; e < (1 << NS); e++) {
            if ((e >> I) & 1) continue;
            double2 ylo, yhi;
            fly_pair<decltype(r)::value>(g.par[I], g.slot(p, e, I), g.sign(p, e, I), Sto<S>::wide(x[e]),
                                         Sto<S>::wide(x[e | (1 << I)]), w[0], w[1], ylo, yhi);
            nb += norm2(ylo);
            nb += norm2(yhi);
            y[e] = Sto<S>::narrow(ylo);
            y[e | (1 << I)] = Sto<S>::narrow(yhi);
        }
    });
}

// Forgets that v was widened before: its FP64 copy need not stay in registers.
__device__ __forceinline__ void forget(float2& v) { asm("" : "+v"(v.x), "+v"(v.y)); }
__device__ __forceinline__ void forget(double2&) {}

template <int NS>
__device__ __forceinline__ void fly_weights(const BInst& I, int k, int b, double2 (&w)[NS][2]) {
#pragma unroll
    for (int i = 0; i < NS; i++) {
        const BStep& s = I.steps[k + i];
        const int bv = I.bitsT[size_t(k + i) * I.B + b];
#pragma unroll
        for (int x = 0; x < 2; x++) w[i][x] = make_double2(s.mre[bv][x], s.mim[bv][x]);
    }
}

template <class S, int NS>
__global__ __launch_bounds__(kBThreads) void fly_step_kernel(const BInst* __restrict__ insts,
                                                             const BItem* __restrict__ items, BLaunch L) {
    constexpr int NE = 1 << NS;
    const BItem it = items[blockIdx.x];
    const BInst& I = insts[it.inst];
    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes);
    const int B = I.B;
    const int b = it.group * kLanes + lane;
    double2 w[NS][2];
    fly_weights<NS>(I, L.k, b, w);
    S* __restrict__ mem = static_cast<S*>(I.mem);
    S* __restrict__ cp = L.copy ? static_cast<S*>(L.copy[it.inst]) : nullptr;
    const FlyDesc& f = I.flys[size_t(L.k) * (kMaxUnit - 2) + NS - 3];
    const FlyGroup<NS> g(f);
    __shared__ uint64_t scols[40];
    __shared__ int spn[40];
    PairWalk<0> wk(it, f, scols, spn, wave);
    const uint64_t ng = wk.groups();
    double nb[NS];
#pragma unroll
    for (int i = 0; i < NS; i++) nb[i] = 0;
    for (uint64_t t = 0; t < ng; t++) {
        if (t) wk.next(t);
        const uint64_t base = uniform64(wk.base);
        const uint32_t p = uint32_t(__builtin_amdgcn_readfirstlane(int(wk.p)));
        S v[NE];
#pragma unroll
        for (int e = 0; e < NE; e++) v[e] = Sto<S>::ld(mem + (base ^ g.de[e]) * uint64_t(B), b);
        if (cp)
#pragma unroll
            for (int e = 0; e < NE; e++) Sto<S>::st(cp + (wk.index(t, 0) * NE + e) * uint64_t(B), b, v[e]);
        fly_each([&](auto i) { fly_step<S, NS, decltype(i)::value>(g, p, w[decltype(i)::value], v, v, nb[decltype(i)::value]); },
                 std::make_integer_sequence<int, NS>{});
#pragma unroll
        for (int e = 0; e < NE; e++) Sto<S>::st(mem + (base ^ g.de[e]) * uint64_t(B), b, v[e]);
    }
    if (!L.bookkeeping) return;
    item_end<NS, false>(I, it, L.k, wave, lane, nb, L.clock);
}

// Put a compact copy of the run's input table back into the forward arena.
template <class S, int NS>
__global__ __launch_bounds__(kBThreads) void fly_restore_kernel(const BInst* __restrict__ insts,
                                                                const BItem* __restrict__ items, BLaunch L) {
    constexpr int NE = 1 << NS;
    const BItem it = items[blockIdx.x];
    const BInst& I = insts[it.inst];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes);
    const int B = I.B;
    const int b = it.group * kLanes + (threadIdx.x & (kLanes - 1));
    S* __restrict__ mem = static_cast<S*>(I.mem);
    const S* __restrict__ cp = static_cast<const S*>(L.copy[it.inst]);
    if (!cp) return;
    const FlyDesc& f = I.flys[size_t(L.k) * (kMaxUnit - 2) + NS - 3];
    const FlyGroup<NS> g(f);
    __shared__ uint64_t scols[40];
    __shared__ int spn[40];
    PairWalk<0> wk(it, f, scols, spn, wave);
    const uint64_t ng = wk.groups();
    for (uint64_t t = 0; t < ng; t++) {
        if (t) wk.next(t);
        const uint64_t base = uniform64(wk.base);
        S v[NE];
#pragma unroll
        for (int e = 0; e < NE; e++) v[e] = Sto<S>::ld(cp + (wk.index(t, 0) * NE + e) * uint64_t(B), b);
#pragma unroll
        for (int e = 0; e < NE; e++) Sto<S>::st(mem + (base ^ g.de[e]) * uint64_t(B), b, v[e]);
    }
}

// Backward through the run: the copy of its first input gives the tables between the steps again (in registers), lambda
// goes from the last step's outputs to the first one's inputs, and every step's gradient is summed.
template <class S, int NS>
__global__ __launch_bounds__(kBThreads, 2) void fly_back_kernel(const BInst* __restrict__ insts,
                                                             const BItem* __restrict__ items, BLaunch L) {
    constexpr int NE = 1 << NS;
    const BItem it = items[blockIdx.x];
    const BInst& I = insts[it.inst];
    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes);
    const int B = I.B;
    const int b = it.group * kLanes + lane;
    double2 w[NS][2];
    fly_weights<NS>(I, L.k, b, w);
    S* __restrict__ lam = static_cast<S*>(I.lam);
    const S* __restrict__ cp = static_cast<const S*>(L.copy[it.inst]);
    const FlyDesc& f = I.flys[size_t(L.k) * (kMaxUnit - 2) + NS - 3];
    const FlyGroup<NS> g(f);
    __shared__ uint64_t scols[40];
    __shared__ int spn[40];
    PairWalk<0> wk(it, f, scols, spn, wave);
    const uint64_t ng = wk.groups();
    double2 G[NS][2];
#pragma unroll
    for (int i = 0; i < NS; i++) G[i][0] = G[i][1] = make_double2(0, 0);
    for (uint64_t t = 0; t < ng; t++) {
        if (t) wk.next(t);
        const uint64_t base = uniform64(wk.base);
        const uint32_t p = uint32_t(__builtin_amdgcn_readfirstlane(int(wk.p)));
        S x[NS][NE], l[NE];
#pragma unroll
        for (int e = 0; e < NE; e++) x[0][e] = Sto<S>::ld(cp + (wk.index(t, 0) * NE + e) * uint64_t(B), b);
#pragma unroll
        for (int e = 0; e < NE; e++) l[e] = Sto<S>::ld(lam + (base ^ g.de[e]) * uint64_t(B), b);
        fly_each([&](auto i) {
            constexpr int J = decltype(i)::value;
            double unused = 0;
            fly_step<S, NS, J>(g, p, w[J], x[J], x[J + 1], unused);
        }, std::make_integer_sequence<int, NS - 1>{});
#pragma unroll
        for (int i = 0; i < NS; i++)
#pragma unroll
            for (int e = 0; e < NE; e++) forget(x[i][e]);
        fly_each([&](auto i) {
            constexpr int J = NS - 1 - decltype(i)::value;
            fly_route_of(g.route[J], [&](auto r) {
#pragma unroll
                for (int e = 0; e < NE; e++) {
                    if ((e >> J) & 1) continue;
                    double2 llo = Sto<S>::wide(l[e]), lhi = Sto<S>::wide(l[e | (1 << J)]);
                    fly_pair_back<decltype(r)::value>(g.par[J], g.slot(p, e, J), g.sign(p, e, J),
                                                      Sto<S>::wide(x[J][e]), Sto<S>::wide(x[J][e | (1 << J)]), w[J][0],
                                                      w[J][1], llo, lhi, G[J]);
                    l[e] = Sto<S>::narrow(llo);
                    l[e | (1 << J)] = Sto<S>::narrow(lhi);
                }
            });
        }, std::make_integer_sequence<int, NS>{});
#pragma unroll
        for (int e = 0; e < NE; e++) Sto<S>::st(lam + (base ^ g.de[e]) * uint64_t(B), b, l[e]);
    }
    double val[4 * NS];
#pragma unroll
    for (int i = 0; i < NS; i++)
#pragma unroll
        for (int x = 0; x < 2; x++) {
            val[4 * i + 2 * x] = G[i][x].x;
            val[4 * i + 2 * x + 1] = G[i][x].y;
        }
    item_end<NS, true>(I, it, L.k, wave, lane, val, nullptr);
}

template <class S>
__global__ void batch_init_kernel(const BInst* __restrict__ insts, int ninst, unsigned long long* clock, int ns) {
    const int i = blockIdx.x;
    if (i >= ninst) return;
    if (i == 0)
        for (int k = threadIdx.x; k <= ns; k += blockDim.x) clock[k] = k ? 0 : (unsigned long long)wall_clock64();
    const BInst& I = insts[i];
    S* mem = static_cast<S*>(I.mem);
    for (int b = threadIdx.x; b < I.B; b += blockDim.x) {
        Sto<S>::st(mem + b, Sto<S>::narrow(make_double2(1.0, 0.0)));
        I.prev[b] = 1.0;
        I.dead[b] = 0;
    }
}

template <class S>
__global__ void batch_finish_kernel(const BInst* __restrict__ insts, int ninst) {
    const int i = blockIdx.x;
    if (i >= ninst) return;
    const BInst& I = insts[i];
    const S* mem = static_cast<const S*>(I.mem);
    for (int b = threadIdx.x; b < I.B; b += blockDim.x) {
        I.logp[b] = I.dead[b] ? -INFINITY : log2(I.prev[b]) - I.ns;
        const double2 z = Sto<S>::wide(Sto<S>::ld(mem + b));
        I.amp[2 * b] = z.x;
        I.amp[2 * b + 1] = z.y;
    }
}

// ---- whole strings in LDS
//
// Small plans are bound by launches: five width-11 plans of 128 lanes took 40 launches of 10 us for tables of 17 KB a
// string, and plans of unlike steps share no sweep of several steps.  Where every plan's table fits the LDS, one block
// takes a string from its first step to its last: one barrier per step (none while 64 cosets or fewer keep one wave busy),
// the steps' norms left as a sum per wave and put together at the end.  Those five plans take 146 us a call instead of
// 514; what is left is the chain of 45 steps (0.9 us each) and 60 us of launch, copies and transposition of the bits.
// Device time of 64 / 1024 / 4096 strings, sweeps against this: 140 / 173 / 306 us and 43 / 70 / 200 at 2^11 complex64
// slots, 178 / 239 / 533 and 58 / 116 / 381 at 2^12, 178 / 288 / 777 and 56 / 142 / 506 at 2^12 complex128 ones, and at
// 2^4 and 4096 strings, the one place where they are level, 56 and 64.
template <class S, int NTQ>
__device__ __forceinline__ double lds_step(const LStep& s, S* tab, double2 w0, double2 w1, int t, int lt) {
    auto uni = [](uint32_t v) { return uint32_t(__builtin_amdgcn_readfirstlane(int(v))); };
    const int nk = int(uni(uint32_t(s.nk))), m = int(uni(uint32_t(s.m)));
    const uint32_t rho = uni(s.rho), t0m = uni(s.t0m), t1m = uni(s.t1m), parm = uni(s.parm), g = uni(s.g);
    uint32_t off[NTQ], a = 0;
#pragma unroll
    for (int q = 0; q < NTQ; q++) off[q] = uni(s.off[q]);
#pragma unroll
    for (int j = 0; j < 9; j++)
        if (j < lt) a ^= ((t >> j) & 1) ? s.cols[j] : 0;      // columns beyond nk are 0
    double nb = 0;
    if (nk < lt && (t >> nk)) return nb;
    uint32_t sg = uint32_t(__popc(uint32_t(t) & rho)) & 1;
    const int groups = nk > lt ? 1 << (nk - lt) : 1;
    for (int it = 0; it < groups; it++) {
        if (it) {
            const int j = lt + __builtin_ctz(unsigned(it));
            a ^= uni(s.cols[j]);
            sg ^= (rho >> j) & 1;
        }
        S v[NTQ];
#pragma unroll
        for (int q = 0; q < NTQ; q++) v[q] = tab[a ^ off[q]];
        double2 A[2][2];
        A[0][0] = A[0][1] = A[1][0] = A[1][1] = make_double2(-0.0, -0.0);
#pragma unroll
        for (int q = 0; q < NTQ; q++)
            gs::route_one(A, Sto<S>::wide(v[q]), (t0m >> q) & 1, (t1m >> q) & 1, sg ^ ((parm >> q) & 1));
        const double2 o0 = cfma(w0, A[0][0], cmul(w1, A[0][1]));
        tab[a] = Sto<S>::narrow(o0);
        nb += norm2(o0);
        if (m == 2) {
            const double2 o1 = cfma(w0, A[1][0], cmul(w1, A[1][1]));
            tab[a ^ g] = Sto<S>::narrow(o1);
            nb += norm2(o1);
        }
    }
    return nb;
}

// Blocks blk0[j] .. blk0[j + 1] - 1 take the strings of instance order[j].
template <class S, int NT>
__global__ __launch_bounds__(NT) void score_lds_kernel(const BInst* __restrict__ insts, int ninst,
                                                                const int* __restrict__ order,
                                                                const int* __restrict__ blk0, int tab_bytes,
                                                                unsigned long long* __restrict__ clock) {
    constexpr int NW = NT / 64, LT = NT == 64 ? 6 : NT == 256 ? 8 : 9;
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ double nbs[kLdsSteps];
    __shared__ int s_dead;
    int j = 0;
    while (j + 1 < ninst && int(blockIdx.x) >= blk0[j + 1]) j++;
    const BInst& I = insts[order[j]];
    const int b = int(blockIdx.x) - blk0[j], B = I.B, ns = I.ns;
    S* tab = reinterpret_cast<S*>(lds);
    LStep* st = reinterpret_cast<LStep*>(lds + tab_bytes);
    double2* wt = reinterpret_cast<double2*>(st + ns);          // [ns][2]
    double* part = reinterpret_cast<double*>(wt + 2 * ns);      // [ns][NW]
    unsigned long long* at = reinterpret_cast<unsigned long long*>(nbs);
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const bool times = b == B - 1;                              // the instance's last string tells the steps' times
    for (int i = t; i < ns * int(sizeof(LStep) / 4); i += NT)
        reinterpret_cast<uint32_t*>(st)[i] = reinterpret_cast<const uint32_t*>(I.lsteps)[i];
    for (int i = t; i < ns * NW; i += NT) part[i] = 0;
    for (int k = t; k < ns; k += NT) {
        const BStep& s = I.steps[k];
        const int bv = I.bitsT[size_t(k) * B + b];
        wt[2 * k] = make_double2(s.mre[bv][0], s.mim[bv][0]);
        wt[2 * k + 1] = make_double2(s.mre[bv][1], s.mim[bv][1]);
    }
    if (t == 0) {
        tab[0] = Sto<S>::narrow(make_double2(1.0, 0.0));
        s_dead = ns;
    }
    __syncthreads();
    for (int k = 0; k < ns; k++) {
        const LStep& s = st[k];
        const bool wide = NW > 1 && __builtin_amdgcn_readfirstlane(s.nk) > 6;
        if (wide || wave == 0) {
            const int ntq = __builtin_amdgcn_readfirstlane(s.ntq), lt = wide ? LT : 6;
            const double2 w0 = wt[2 * k], w1 = wt[2 * k + 1];
            double nb = ntq == 1   ? lds_step<S, 1>(s, tab, w0, w1, t, lt)
                        : ntq == 2 ? lds_step<S, 2>(s, tab, w0, w1, t, lt)
                                   : lds_step<S, 4>(s, tab, w0, w1, t, lt);
            nb = gs::wave_sum(nb);
            if (lane == 0) part[k * NW + wave] = nb;
            if (times && t == 0) at[k] = wall_clock64();
            gs::wave_fence();
        }
        const bool next = NW > 1 && k + 1 < ns && __builtin_amdgcn_readfirstlane(st[k + 1].nk) > 6;
        if (wide || next) __syncthreads();
    }
    if (times) {
        __syncthreads();
        for (int k = t; k < ns && clock; k += NT) atomicMax(clock + 1 + k, at[k]);
    }
    __syncthreads();
    for (int k = t; k < ns; k += NT) {
        double nb = part[k * NW];
#pragma unroll
        for (int w = 1; w < NW; w++) nb += part[k * NW + w];
        nbs[k] = nb;
        if (nb <= 0) atomicMin(&s_dead, k);
    }
    __syncthreads();
    const int dead = s_dead;
    for (int k = t; k < ns; k += NT)
        I.cond[size_t(b) * ns + k] = k >= dead ? 0 : nbs[k] / (2 * (k ? nbs[k - 1] : 1.0));
    if (t != 0) return;
    I.logp[b] = dead < ns ? -INFINITY : log2(ns ? nbs[ns - 1] : 1.0) - ns;
    const double2 z = Sto<S>::wide(tab[0]);
    I.amp[2 * b] = z.x;
    I.amp[2 * b + 1] = z.y;
    if (clock && ns) atomicMax(clock + ns, (unsigned long long)wall_clock64());
}

// A step for score_lds_kernel; esz: bytes of an entry.
LStep make_lstep(const gs::StepInfo& s, int R, size_t esz) {
    LStep d{};
    gs::GfBasis span, taken, banks;
    for (uint64_t c : s.cols) (void)span.add(c);
    const uint64_t form = span.form(s.rhoc & ((uint64_t(1) << s.nk) - 1)), bank = 256 / esz - 1;
    std::vector<uint64_t> cand;
    for (int i = 0; i < R; i++)
        if (span.has(uint64_t(1) << i)) cand.push_back(uint64_t(1) << i);
    cand.insert(cand.end(), s.cols.begin(), s.cols.end());
    for (int pass = 0; pass < 2; pass++)
        for (uint64_t c : cand) {
            if (pass == 0 && banks.has(c & bank)) continue;
            if (!taken.add(c)) continue;
            (void)banks.add(c & bank);
            d.rho |= uint32_t(gs::parity(c & form)) << d.nk;
            d.cols[d.nk++] = uint32_t(c);
        }
    for (int q = 0; q < s.ntq; q++) {
        d.off[q] = uint32_t(s.off[q]);
        d.t0m |= uint32_t(s.tau0[q] & 1) << q;
        d.t1m |= uint32_t(s.tau1[q] & 1) << q;
        d.parm |= uint32_t(s.par[q] & 1) << q;
    }
    d.g = uint32_t(s.g);
    d.ntq = s.ntq;
    d.m = s.m;
    return d;
}

// lambda at the end of the chain: dZ/d(final single entry) = 1
template <class S>
__global__ void batch_lambda_init_kernel(const BInst* __restrict__ insts, int ninst) {
    const int i = blockIdx.x;
    if (i >= ninst) return;
    const BInst& I = insts[i];
    S* lam = static_cast<S*>(I.lam);
    for (int b = threadIdx.x; b < I.B; b += blockDim.x) Sto<S>::st(lam + b, Sto<S>::narrow(make_double2(1.0, 0.0)));
}

thread_local std::string g_berr;

int bfail(int code, const std::string& m) {
    g_berr = m;
    return code;
}

}  // namespace

struct gs_plan {
    gs::Plan p;
};

// A launch of the batch: steps k .. k + n - 1 of the instances of its work items.
struct Sweep {
    int k, n;
    const PairDesc* pair;                 // n == 2: the kind of pair
    int nq;                               // most slots per coset among the instances at step k (kernel variant)
    bool exact;                           // ... every one has nq
    BItem* items;
    int nitems;
};

struct gs_batch {
    int device = 0;
    int storage = GS_C64;
    size_t esz = 8;
    hipStream_t stream = nullptr;
    std::vector<gs::Plan> plans;
    std::vector<int> B;
    std::vector<BInst> hinst;
    std::vector<std::vector<BStep>> hsteps;
    BInst* dinst = nullptr;
    std::vector<void*> allocs;
    int maxns = 0;
    void* item_mem = nullptr;             // the launches' work items (device)
    std::vector<std::vector<int>> lg;     // [inst][step]: log2 cosets per item
    int lg_default = 8;                   // smallest tile (sizes the partial buffers); steps start at 2^9
    // sweeps of several steps (build_several; empty until a batch that scores in LDS takes a gradient)
    std::vector<std::vector<PairDesc>> hpairs;   // [inst][step]: steps k and k+1 as one sweep (ni 0: not possible)
    std::vector<std::vector<FlyDesc>> hflys;     // [inst][step][kMaxUnit - 2]: 3 steps and more (d 0: not possible)
    // scoring with whole strings in LDS (score_lds_kernel): bytes of its table and of all its LDS (0: not all plans fit)
    int lds_table = 0, lds_bytes = 0, lds_blocks = 0, lds_threads = 512;
    int *dorder = nullptr, *dblk0 = nullptr;
    std::vector<char> unit;               // per step: steps of the sweep that starts there (0: inside another's)
    std::vector<Sweep> common;            // the launches of these sweeps, every instance in each (gradients)
    std::vector<Sweep> sweeps;            // scoring: the launches, by first step; instances may take sweeps of their own
    bool pairs_on = true;
    int lu = 2;                           // log2 cosets a lane gathers at once
    bool items_dirty = false;             // tiles changed since the work lists were built
    int xcd_items = 1;                    // work lists ordered so each XCD takes consecutive items (2: coset-major)
    double auto_budget = -1;              // mem_budget argument of the last automatic segment choice
    // graph replay
    bool use_graph = false;
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    unsigned long long *dclock = nullptr, *hclock = nullptr;   // [1 + maxns]: device clock at the start, after each step
    int clock_khz = 0;
    // every instance's strings, and its results: log2 Pr, Z, the clock, then the conditionals of all; pinned copies
    int8_t *dbits = nullptr, *hbits = nullptr;
    double *dout = nullptr, *hout = nullptr;
    size_t nbits = 0, nhead = 0, nout = 0;   // bytes of strings; doubles before the conditionals; in all
    std::vector<size_t> at_bits, at_logp, at_amp, at_cond;
    double last_ms = 0;
    std::vector<double> step_ms;          // end of step k, ms after the start (last call)
    // gradient mode
    int seg = 0;                          // steps per checkpoint segment in use
    std::vector<void*> galloc;            // adjoint arena, copies
    std::vector<void**> dcopy;            // per step: device array [ninst] of copy destinations (forward, last segment)
    std::vector<std::vector<void*>> ckpt; // [segment][inst]
    std::vector<std::vector<void*>> stack;// [slot in segment][inst]
    void** dptrs = nullptr;               // device scratch for per-launch pointer arrays
    double grad_fwd_ms = 0, grad_ms = 0;
};

namespace {

template <class T>
T* dalloc(gs_batch* b, size_t n) {
    void* p = nullptr;
    if (hipMalloc(&p, std::max<size_t>(n * sizeof(T), 16)) != hipSuccess) return nullptr;
    b->allocs.push_back(p);
    return static_cast<T*>(p);
}

// Descriptors of every instance's sweeps of several steps, host and device, and the instances' device table with their
// addresses.  Batches whose strings are scored in LDS have that table without them, until a gradient first asks: five plans
// of width 11 are made in 1.6 ms with them, 1.2 without.
int build_several(gs_batch* bt) {
    const size_t ni = bt->plans.size();
    std::vector<std::vector<PairDesc>> pairs(ni);
    std::vector<std::vector<FlyDesc>> flys(ni);
    size_t np = 0, nf = 0;
    for (size_t i = 0; i < ni; i++) {
        const gs::Plan& P = bt->plans[i];
        std::vector<PairDesc>& hp = pairs[i];
        hp.resize(size_t(P.ns));
        for (int k = 0; k < P.ns; k++)
            if (k + 1 >= P.ns || !make_pair(P.steps[size_t(k)], P.steps[size_t(k) + 1], false, hp[size_t(k)])) hp[size_t(k)].ni = 0;
        std::vector<FlyDesc>& hf = flys[i];
        hf.resize(size_t(P.ns) * (kMaxUnit - 2));
        for (int k = 0; k < P.ns; k++)
            for (int n = 3; n <= kMaxUnit; n++) {
                const gs::StepInfo* st[kMaxUnit] = {};
                for (int j = 0; j < n && k + j < P.ns; j++) st[j] = &P.steps[size_t(k + j)];
                FlyDesc& f = hf[size_t(k) * (kMaxUnit - 2) + size_t(n - 3)];
                if (!st[n - 1] || !make_fly(st, n, 0, 0, f)) f.d = 0;
            }
        np += hp.size();
        nf += hf.size();
    }
    auto up256 = [](size_t n) { return (n + 255) & ~size_t(255); };
    const size_t table = ni * sizeof(BInst), at_pair = bt->dinst ? 0 : up256(table),
                 at_fly = at_pair + up256(np * sizeof(PairDesc));
    std::vector<char> up(at_fly + nf * sizeof(FlyDesc));
    char* mem = dalloc<char>(bt, up.size());
    if (!mem) return bfail(11, "allocation of the sweep descriptors failed");
    size_t p = at_pair, f = at_fly;
    for (size_t i = 0; i < ni; i++) {
        if (!pairs[i].empty()) memcpy(up.data() + p, pairs[i].data(), pairs[i].size() * sizeof(PairDesc));
        if (!flys[i].empty()) memcpy(up.data() + f, flys[i].data(), flys[i].size() * sizeof(FlyDesc));
        bt->hinst[i].pairs = reinterpret_cast<PairDesc*>(mem + p);
        bt->hinst[i].flys = reinterpret_cast<FlyDesc*>(mem + f);
        p += pairs[i].size() * sizeof(PairDesc);
        f += flys[i].size() * sizeof(FlyDesc);
    }
    if (at_pair) memcpy(up.data(), bt->hinst.data(), table);
    if (!up.empty() && hipMemcpy(mem, up.data(), up.size(), hipMemcpyHostToDevice) != hipSuccess)
        return bfail(17, "plan upload failed");
    if (at_pair) bt->dinst = reinterpret_cast<BInst*>(mem);
    else if (hipMemcpy(bt->dinst, bt->hinst.data(), table, hipMemcpyHostToDevice) != hipSuccess)
        return bfail(17, "instance upload failed");
    bt->hpairs = std::move(pairs);
    bt->hflys = std::move(flys);
    return 0;
}

constexpr double kLaunch = 40e6;                          // bytes moved in the time a launch and its reduction take

// Bytes that one sweep of instance i over the n steps from k saves against a sweep more of the table.
double unit_bytes(const gs_batch* bt, size_t i, int k, int n) {
    return 2.0 * double(bt->B[i]) * double(bt->esz) *
           double(uint64_t(n > 2 ? 2 : bt->hpairs[i][size_t(k)].mo) << bt->plans[i].steps[size_t(k)].nk);
}

// Which sweeps the members' step sequence takes (per step: the steps of the sweep that starts there): single steps, or
// several at once where every member that is still running has the same kind of pair, or a run of butterfly steps.  A
// sweep of n steps saves n - 1 writes and reads of the table (and launches); the sweeps are the disjoint ones that save
// the most.
std::vector<char> choose_units(const gs_batch* bt, const std::vector<size_t>& members) {
    int ns = 0;
    for (size_t i : members) ns = std::max(ns, bt->plans[i].ns);
    std::vector<char> unit(size_t(bt->maxns), 1);
    if (!bt->pairs_on || bt->hpairs.empty()) return unit;
    std::vector<double> best(size_t(ns + kMaxUnit), 0.0);
    std::vector<char> take(size_t(ns), 1);
    for (int k = ns - 1; k >= 0; k--) {
        best[size_t(k)] = best[size_t(k) + 1];
        for (int n = 2; n <= kMaxUnit && k + n <= ns; n++) {
            double g = kLaunch;
            const PairDesc* first = nullptr;
            int ntq = 0;
            bool ok = true;
            for (size_t i : members) {
                const gs::Plan& P = bt->plans[i];
                if (k >= P.ns) continue;
                const PairDesc& p = bt->hpairs[i][size_t(k)];
                if (k + n > P.ns) {
                    ok = false;
                } else if (n > 2) {
                    ok = bt->hflys[i][size_t(k) * (kMaxUnit - 2) + size_t(n - 3)].d == n;
                } else if (!first) {
                    first = &p;
                    ntq = P.steps[size_t(k)].ntq;
                    ok = p.ni != 0;
                } else {
                    ok = p.ni == first->ni && p.mo == first->mo && p.deg == first->deg && P.steps[size_t(k)].ntq == ntq;
                }
                if (!ok) break;
                g += unit_bytes(bt, i, k, n);
            }
            g *= n - 1;
            if (ok && g + best[size_t(k + n)] > best[size_t(k)]) {
                best[size_t(k)] = g + best[size_t(k + n)];
                take[size_t(k)] = char(n);
            }
        }
    }
    for (int k = 0; k < ns; k += take[size_t(k)]) {
        unit[size_t(k)] = take[size_t(k)];
        for (int j = 1; j < take[size_t(k)]; j++) unit[size_t(k + j)] = 0;
    }
    return unit;
}

// The instances whose sweeps at step k can share a launch, as groups (first member first).
std::vector<std::vector<size_t>> sweep_groups(const gs_batch* bt, const std::vector<const std::vector<char>*>& unit, int k) {
    std::vector<std::vector<size_t>> groups;
    for (size_t i = 0; i < bt->plans.size(); i++) {
        if (k >= bt->plans[i].ns || !(*unit[i])[size_t(k)]) continue;
        const int n = (*unit[i])[size_t(k)];
        bool found = false;
        for (auto& g : groups) {
            const size_t f = g[0];
            if ((*unit[f])[size_t(k)] != n) continue;
            if (n == 2) {
                const PairDesc &a = bt->hpairs[i][size_t(k)], &b = bt->hpairs[f][size_t(k)];
                if (a.ni != b.ni || a.mo != b.mo || a.deg != b.deg ||
                    bt->plans[i].steps[size_t(k)].ntq != bt->plans[f].steps[size_t(k)].ntq)
                    continue;
            }
            g.push_back(i);
            found = true;
            break;
        }
        if (!found) groups.push_back({i});
    }
    return groups;
}

// What a choice of sweeps costs, in bytes, up to a constant: its launches, less the bytes its sweeps save.
double units_cost(const gs_batch* bt, const std::vector<const std::vector<char>*>& unit) {
    double c = 0;
    for (int k = 0; k < bt->maxns; k++)
        for (const auto& g : sweep_groups(bt, unit, k)) {
            c += kLaunch;
            for (size_t i : g) {
                const int n = (*unit[i])[size_t(k)];
                if (n > 1) c -= (n - 1) * unit_bytes(bt, i, k, n);
            }
        }
    return c;
}

// Scoring: instances do not wait for each other, so an instance may take the sweeps that suit its own plan, in launches
// of its own where no other takes the same kind at that step.  The widest instances leave the common sequence first,
// while what the sweeps save is more than the launches cost; at most kLeave of them, so that the choice takes a time
// proportional to the number of plans (400 plans: the batch is made in 50 ms instead of 60, its scores take 7.2 ms either
// way).  64 lanes each of four plans of bands 19 to 21: 4.00 -> 2.83 ms complex64, 6.77 -> 3.84 complex128; 96 plans of
// widths 13 to 24: 11,800 strings/s one batch each, 13,200 in two.
constexpr size_t kLeave = 64;
std::vector<std::vector<char>> score_units(const gs_batch* bt) {
    const size_t ni = bt->plans.size(), most = std::min(ni, kLeave);
    std::vector<size_t> order(ni);
    for (size_t i = 0; i < ni; i++) order[i] = i;
    auto bytes = [&](size_t i) {
        int nk = 0;
        for (const gs::StepInfo& st : bt->plans[i].steps) nk = std::max(nk, st.nk);
        return double(bt->B[i]) * double(uint64_t(1) << nk);
    };
    std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) { return bytes(a) > bytes(b); });
    std::vector<std::vector<char>> best(ni, bt->unit), own(ni);
    if (ni == 1 || !bt->pairs_on || bt->lds_bytes) return best;
    for (size_t j = 0; j < most; j++) own[order[j]] = choose_units(bt, {order[j]});
    auto view = [&](const std::vector<char>& common, size_t leave) {
        std::vector<const std::vector<char>*> v(ni, &common);
        for (size_t j = 0; j < leave; j++) v[order[j]] = &own[order[j]];
        return v;
    };
    double cost = units_cost(bt, view(bt->unit, 0));
    for (size_t leave = 1; leave <= most; leave++) {
        const std::vector<char> common = choose_units(bt, std::vector<size_t>(order.begin() + ptrdiff_t(leave), order.end()));
        const auto v = view(common, leave);
        const double c = units_cost(bt, v);
        if (c >= cost) continue;
        cost = c;
        for (size_t i = 0; i < ni; i++) best[i] = *v[i];
    }
    return best;
}

// Cosets (or super-cosets of several steps) of instance i's sweep of the n steps from k, log2, and log2 of the step-k cosets in each.
void sweep_size(const gs_batch* bt, size_t i, int k, int n, int& nk, int& inner) {
    nk = bt->plans[i].steps[size_t(k)].nk;
    inner = 0;
    if (n < 2) return;
    if (n > 2) {
        inner = n - 1;
        nk -= inner;
        return;
    }
    const PairDesc& p = bt->hpairs[i][size_t(k)];
    inner = p.ni == 4 ? 2 : p.ni == 2 ? 1 : 0;
    nk = p.nk;
}

// log2 (super-)cosets per work item.  Tiles set per step index (by hand or by the autotuner, often on a larger batch)
// are made finer, down to 2^kFinestTile cosets, while the launch has fewer than kMinItems items: one item per block,
// and a launch of a few dozen blocks leaves the chip idle while each wave walks a long range (five width-11 plans of
// 128 lanes: 40 blocks of 2^8 cosets took 30 us a step).  The backward sums of several steps take more room per item, so their
// tiles start coarser.
constexpr int kFinestTile = 4;
int item_lg(const gs_batch* bt, size_t i, int k, int n, int shrink, bool& finer) {
    int nk, inner;
    sweep_size(bt, i, k, n, nk, inner);
    const int floor = std::min(nk, std::max(0, kFinestTile - inner));
    int lg = bt->lg[i][size_t(k)];
    if (n > 1) lg = std::max(lg, bt->lg_default + (n > 2 ? 2 : 1));
    lg = std::min(nk, std::max(lg - inner - shrink, floor));
    finer = finer || lg > floor;
    return lg;
}

// The work items of one launch: the n steps from k of the instances in `group`.
std::vector<BItem> sweep_items(const gs_batch* bt, const std::vector<size_t>& group, int k, int n) {
    int shrink = 0;
    for (;; shrink++) {
        int64_t tot = 0;
        bool finer = false;
        for (size_t i : group) {
            int nk, inner;
            sweep_size(bt, i, k, n, nk, inner);
            tot += int64_t(bt->B[i] / kLanes) << (nk - item_lg(bt, i, k, n, shrink, finer));
        }
        if (tot >= kMinItems || !finer) break;
    }
    std::vector<BItem> items;
    for (size_t i : group) {
        int nk, inner;
        bool finer = false;
        sweep_size(bt, i, k, n, nk, inner);
        const int lg = item_lg(bt, i, k, n, shrink, finer);
        const int count = 1 << (nk - lg);
        const int ng = bt->B[i] / kLanes;
        for (int o = 0; o < ng * count; o++) {
            // group-major (every coset range of lane group 0, then group 1, ...) or, with xcd_items == 2,
            // coset-major (all lane groups of a coset range next to each other: whole slot rows)
            const int g = bt->xcd_items == 2 ? o % ng : o / count;
            const int q = bt->xcd_items == 2 ? o / ng : o % count;
            BItem it{};
            it.c0 = uint64_t(q) << lg;
            it.inst = int(i);
            it.group = g;
            it.lg = lg;
            it.index = q;
            it.count = count;
            items.push_back(it);
        }
    }
    if (bt->xcd_items && items.size() >= 8 && items.size() % 8 == 0) {
        // blocks are dealt round-robin to the 8 XCDs (block i on XCD i mod 8): list position b = (j mod n/8) * 8
        // + j / (n/8) gives XCD x the consecutive items x n/8 .. (x+1) n/8 - 1 (adjacent coset ranges)
        const size_t m = items.size(), chunk = m / 8;
        std::vector<BItem> order(m);
        for (size_t j = 0; j < m; j++) order[(j % chunk) * 8 + j / chunk] = items[j];
        items.swap(order);
    }
    return items;
}

int build_items(gs_batch* bt) {
    (void)hipFree(bt->item_mem);
    bt->item_mem = nullptr;
    std::vector<BItem> all;                               // the lists of every launch, in one allocation
    std::vector<size_t> at;                               // ... where each begins
    const size_t ni = bt->plans.size();
    std::vector<size_t> everyone(ni);
    for (size_t i = 0; i < ni; i++) everyone[i] = i;
    bt->unit = choose_units(bt, everyone);
    auto add = [&](std::vector<Sweep>& to, const std::vector<size_t>& group, int k, int n) {
        Sweep w{k, n, n == 2 ? &bt->hpairs[group[0]][size_t(k)] : nullptr, 1, true, nullptr, 0};
        for (size_t i : group) w.nq = std::max(w.nq, bt->plans[i].steps[size_t(k)].ntq);
        for (size_t i : group) w.exact = w.exact && bt->plans[i].steps[size_t(k)].ntq == w.nq;
        const std::vector<BItem> items = sweep_items(bt, group, k, n);
        w.nitems = int(items.size());
        at.push_back(all.size());
        all.insert(all.end(), items.begin(), items.end());
        to.push_back(w);
    };
    bt->common.clear();
    bt->sweeps.clear();
    for (int k = 0; k < bt->maxns; k++) {
        std::vector<size_t> group;
        for (size_t i = 0; i < ni; i++)
            if (k < bt->plans[i].ns) group.push_back(i);
        if (bt->unit[size_t(k)]) add(bt->common, group, k, bt->unit[size_t(k)]);
    }
    const std::vector<std::vector<char>> own = score_units(bt);
    std::vector<const std::vector<char>*> view(ni);
    bool same = true;
    for (size_t i = 0; i < ni; i++) {
        view[i] = &own[i];
        same = same && own[i] == bt->unit;
    }
    for (int k = 0; k < bt->maxns && !same; k++)
        for (const auto& g : sweep_groups(bt, view, k)) add(bt->sweeps, g, k, own[g[0]][size_t(k)]);
    if (hipMalloc(&bt->item_mem, std::max<size_t>(all.size() * sizeof(BItem), 16)) != hipSuccess) {
        bt->item_mem = nullptr;
        return bfail(11, "work-item allocation failed");
    }
    if (hipMemcpy(bt->item_mem, all.data(), all.size() * sizeof(BItem), hipMemcpyHostToDevice) != hipSuccess)
        return bfail(17, "work-item upload failed");
    size_t a = 0;
    for (Sweep& w : bt->common) w.items = static_cast<BItem*>(bt->item_mem) + at[a++];
    for (Sweep& w : bt->sweeps) w.items = static_cast<BItem*>(bt->item_mem) + at[a++];
    if (same) bt->sweeps = bt->common;
    return 0;
}

// Most items of one lane group of instance i in a launch: a step at the smallest tile gs_batch_set_tile accepts
// (2^lg_default cosets), or a launch that was made finer (fewer than 2 kMinItems over all groups).
size_t part_items(const gs_batch* bt, size_t i) {
    size_t m = 1;
    for (const gs::StepInfo& s : bt->plans[i].steps)
        m = std::max(m, size_t(1) << (s.nk - std::min(s.nk, bt->lg_default)));
    return std::max(m, 2 * size_t(kMinItems) * kLanes / size_t(bt->B[i]));
}

// Doubles of one lane group's partials: four sums per lane of every item (a pair's eight at twice the smallest tile, ...).
size_t part_doubles(const gs_batch* bt, size_t i) {
    const size_t fine = 2 * size_t(kMinItems) * kLanes / size_t(bt->B[i]);
    return kLanes * std::max(4 * part_items(bt, i), size_t(kMaxSums) * std::max<size_t>(fine, 1));
}

// Instantiation of kernel K<S, NQ, LU, EX> for NQ in {1, 2, 4}, LU in 0..3, EX (every instance has NQ slots at the
// step) false or true.
#define GS_BV(K, S, nq, lu)                                                                                        \
    case (nq) * 8 + (lu) * 2: return reinterpret_cast<const void*>(&K<S, nq, lu, false>);                          \
    case (nq) * 8 + (lu) * 2 + 1: return reinterpret_cast<const void*>(&K<S, nq, lu, true>);
#define GS_BATCH_VARIANT(K, S, nq, lu, ex)                                                                        \
    [&]() -> const void* {                                                                                         \
        switch ((nq) * 8 + (lu) * 2 + ((ex) ? 1 : 0)) {                                                           \
            GS_BV(K, S, 1, 0) GS_BV(K, S, 1, 1) GS_BV(K, S, 1, 2) GS_BV(K, S, 1, 3)                                 \
            GS_BV(K, S, 2, 0) GS_BV(K, S, 2, 1) GS_BV(K, S, 2, 2) GS_BV(K, S, 2, 3)                                 \
            GS_BV(K, S, 4, 0) GS_BV(K, S, 4, 1) GS_BV(K, S, 4, 2) GS_BV(K, S, 4, 3)                                 \
        }                                                                                                          \
        return nullptr;                                                                                            \
    }()

// Instantiation of pair kernel K<S, NQ, NI, MO, DEG> for the step's slots and the kind of pair.
#define GS_PV(K, S, nq, ni, mo, deg)                                                                               \
    case (nq) * 32 + (ni) * 4 + (mo) * 2 + (deg) - 2: return reinterpret_cast<const void*>(&K<S, nq, ni, mo, deg>);
#define GS_PVN(K, S, nq)                                                                                           \
    GS_PV(K, S, nq, 1, 1, 0) GS_PV(K, S, nq, 1, 2, 0) GS_PV(K, S, nq, 1, 2, 1)                                      \
    GS_PV(K, S, nq, 2, 1, 0) GS_PV(K, S, nq, 2, 2, 0) GS_PV(K, S, nq, 2, 2, 1)                                      \
    GS_PV(K, S, nq, 4, 1, 0) GS_PV(K, S, nq, 4, 2, 0)
#define GS_PAIR_VARIANT(K, S, nq, p)                                                                               \
    [&]() -> const void* {                                                                                         \
        switch ((nq) * 32 + (p).ni * 4 + (p).mo * 2 + (p).deg - 2) {                                                \
            GS_PVN(K, S, 1) GS_PVN(K, S, 2) GS_PVN(K, S, 4)                                                        \
        }                                                                                                          \
        return nullptr;                                                                                            \
    }()

enum BKernel { kBStep, kBRestore, kBBack };

template <class S>
const void* fly_variant(BKernel kind, int n) {
#define GS_FV(n) (kind == kBStep ? reinterpret_cast<const void*>(&fly_step_kernel<S, n>)                            \
                  : kind == kBRestore ? reinterpret_cast<const void*>(&fly_restore_kernel<S, n>)                     \
                                      : reinterpret_cast<const void*>(&fly_back_kernel<S, n>))
    return n == 3 ? GS_FV(3) : nullptr;
#undef GS_FV
}

template <class S>
int launch_batch(gs_batch* bt, BKernel kind, const Sweep& w, BLaunch L) {
    if (w.nitems == 0) return 0;
    const int nq = w.nq, lu = bt->lu;
    const bool ex = w.exact;
    const void* fn = w.n > 2 ? fly_variant<S>(kind, w.n)
                   : w.pair ? (kind == kBStep ? GS_PAIR_VARIANT(pair_step_kernel, S, nq, *w.pair)
                               : kind == kBRestore ? GS_PAIR_VARIANT(pair_restore_kernel, S, nq, *w.pair)
                                                   : GS_PAIR_VARIANT(pair_back_kernel, S, nq, *w.pair))
                   : kind == kBStep ? GS_BATCH_VARIANT(batch_step_kernel, S, nq, lu, ex)
                   : kind == kBRestore ? GS_BATCH_VARIANT(batch_restore_kernel, S, nq, lu, ex)
                                       : GS_BATCH_VARIANT(batch_back_kernel, S, nq, lu, ex);
    if (!fn) return bfail(16, "no kernel variant");
    const BInst* insts = bt->dinst;
    const BItem* items = w.items;
    void* args[] = {&insts, &items, &L};
    return hipLaunchKernel(fn, dim3(w.nitems), dim3(kBThreads), args, 0, bt->stream) == hipSuccess
               ? 0 : bfail(17, "step launch failed");
}

template <class S>
int launch_step(gs_batch* bt, const Sweep& w, int bookkeeping, void* const* copy) {
    return launch_batch<S>(bt, kBStep, w, BLaunch{w.k, bookkeeping, copy, bt->dclock});
}

template <class S>
int enqueue_t(gs_batch* bt) {
    const int ninst = int(bt->plans.size());
    hipLaunchKernelGGL(batch_init_kernel<S>, dim3(ninst), dim3(256), 0, bt->stream, bt->dinst, ninst,
                       bt->dclock, bt->maxns);
    if (bt->lds_bytes && bt->pairs_on) {
        const int nt = bt->lds_threads;
        hipLaunchKernelGGL((nt == 64 ? score_lds_kernel<S, 64> : nt == 256 ? score_lds_kernel<S, 256> : score_lds_kernel<S, 512>),
                           dim3(bt->lds_blocks), dim3(nt), bt->lds_bytes, bt->stream, bt->dinst, ninst, bt->dorder, bt->dblk0,
                           bt->lds_table, bt->dclock);
        return hipGetLastError() == hipSuccess ? 0 : bfail(17, "batch launch failed");
    }
    for (const Sweep& w : bt->sweeps)
        if (int rc = launch_step<S>(bt, w, 1, nullptr)) return rc;
    hipLaunchKernelGGL(batch_finish_kernel<S>, dim3(ninst), dim3(256), 0, bt->stream, bt->dinst, ninst);
    if (hipGetLastError() != hipSuccess) return bfail(17, "batch launch failed");
    return 0;
}

int enqueue(gs_batch* bt) {
    return bt->storage == GS_C64 ? enqueue_t<float2>(bt) : enqueue_t<double2>(bt);
}

void drop_graph(gs_batch* bt) {
    if (bt->gexec) (void)hipGraphExecDestroy(bt->gexec);
    if (bt->graph) (void)hipGraphDestroy(bt->graph);
    bt->gexec = nullptr;
    bt->graph = nullptr;
}

int build_graph(gs_batch* bt) {
    drop_graph(bt);
    if (hipStreamBeginCapture(bt->stream, hipStreamCaptureModeThreadLocal) != hipSuccess)
        return bfail(17, "stream capture failed");
    const int rc = enqueue(bt);
    hipGraph_t g = nullptr;
    if (hipStreamEndCapture(bt->stream, &g) != hipSuccess || rc) return rc ? rc : bfail(17, "stream capture failed");
    bt->graph = g;
    if (hipGraphInstantiate(&bt->gexec, g, nullptr, nullptr, 0) != hipSuccess) return bfail(17, "graph instantiate failed");
    return 0;
}

// The strings of every instance, transposed to step-major, in one copy.
int upload_bits(gs_batch* bt, const int8_t* const* bits) {
    int8_t bad = 0;
    for (size_t i = 0; i < bt->plans.size(); i++) {
        const int B = bt->B[i], ns = bt->plans[i].ns;
        int8_t* to = bt->hbits + bt->at_bits[i];
        for (int b0 = 0; b0 < B; b0 += kLanes)            // 64 strings at a time: whole cache lines of the result
            for (int k = 0; k < ns; k++)
                for (int b = b0; b < b0 + kLanes; b++) {
                    const int8_t v = bits[i][size_t(b) * ns + k];
                    bad |= v & ~int8_t(1);
                    to[size_t(k) * B + b] = v;
                }
    }
    if (bad) return bfail(16, "bits must be 0 or 1");
    if (bt->nbits && hipMemcpyAsync(bt->dbits, bt->hbits, bt->nbits, hipMemcpyHostToDevice, bt->stream) != hipSuccess)
        return bfail(17, "bits upload failed");
    return 0;
}

// Entries of the compact copy of step k's input table of instance i.
size_t copy_entries(const gs_batch* bt, size_t i, int k) {
    const gs::StepInfo& s = bt->plans[i].steps[size_t(k)];
    return (size_t(1) << s.nk) * size_t(s.ntq) * size_t(bt->B[i]);
}

void free_grad(gs_batch* bt) {
    for (void* p : bt->galloc) (void)hipFree(p);
    bt->galloc.clear();
    bt->ckpt.clear();
    bt->stack.clear();
    bt->seg = 0;
}

// First step of segment s's sweeps: its sweeps are those that start in steps s seg .. (s + 1) seg - 1, so a pair that
// straddles the boundary belongs to the earlier segment (the pairs, and with them the order of every sum, do not
// depend on seg).
int seg_first(const gs_batch* bt, int seg, int s) {
    int k = std::min(s * seg, bt->maxns);
    while (k < bt->maxns && !bt->unit[size_t(k)]) k++;
    return k;
}

// Allocate the adjoint arenas and the copies for segments of `seg` steps.
int alloc_grad(gs_batch* bt, int seg) {
    free_grad(bt);
    const size_t ni = bt->plans.size();
    auto galloc = [&](size_t bytes) -> void* {
        void* p = nullptr;
        if (hipMalloc(&p, std::max<size_t>(bytes, 16)) != hipSuccess) return nullptr;
        bt->galloc.push_back(p);
        return p;
    };
    for (size_t i = 0; i < ni; i++) {
        BInst& I = bt->hinst[i];
        if (!I.lam) {
            I.lam = dalloc<char>(bt, (size_t(1) << bt->plans[i].R) * size_t(bt->B[i]) * bt->esz);
            I.grad = dalloc<double>(bt, size_t(bt->B[i]) * bt->plans[i].ns * 4);
            if (!I.lam || !I.grad) return bfail(11, "adjoint arena allocation failed");
        }
    }
    const int nseg = (bt->maxns + seg - 1) / seg;
    bt->ckpt.assign(size_t(nseg), std::vector<void*>(ni, nullptr));
    bt->stack.assign(size_t(seg), std::vector<void*>(ni, nullptr));
    for (int sgi = 0; sgi < nseg; sgi++)
        for (size_t i = 0; i < ni; i++) {
            const int k = seg_first(bt, seg, sgi);
            if (k >= bt->plans[i].ns || k >= (sgi + 1) * seg) continue;
            if (!(bt->ckpt[size_t(sgi)][i] = galloc(copy_entries(bt, i, k) * bt->esz))) return bfail(11, "checkpoint allocation failed");
        }
    for (int j = 0; j < seg; j++)
        for (size_t i = 0; i < ni; i++) {
            size_t mx = 0;
            for (int sgi = 0; sgi < nseg; sgi++) {
                const int k = sgi * seg + j;
                if (k < bt->plans[i].ns && bt->unit[size_t(k)]) mx = std::max(mx, copy_entries(bt, i, k));
            }
            if (mx && !(bt->stack[size_t(j)][i] = galloc(mx * bt->esz))) return bfail(11, "segment stack allocation failed");
        }
    if (hipMemcpy(bt->dinst, bt->hinst.data(), bt->hinst.size() * sizeof(BInst), hipMemcpyHostToDevice) != hipSuccess)
        return bfail(17, "instance upload failed");
    bt->seg = seg;
    return 0;
}

// Bytes of adjoint memory for segments of `seg` steps.
size_t grad_bytes(const gs_batch* bt, int seg) {
    size_t tot = 0;
    const int nseg = (bt->maxns + seg - 1) / seg;
    for (size_t i = 0; i < bt->plans.size(); i++) {
        for (int sgi = 0; sgi < nseg; sgi++) {
            const int k = seg_first(bt, seg, sgi);
            if (k < bt->plans[i].ns && k < (sgi + 1) * seg) tot += copy_entries(bt, i, k);
        }
        for (int j = 0; j < seg; j++) {
            size_t mx = 0;
            for (int sgi = 0; sgi < nseg; sgi++)
                if (sgi * seg + j < bt->plans[i].ns && bt->unit[size_t(sgi * seg + j)])
                    mx = std::max(mx, copy_entries(bt, i, sgi * seg + j));
            tot += mx;
        }
    }
    return tot * bt->esz;
}

// Steps per checkpoint segment: among the segment lengths whose copies fit the budget (mem_budget <= 0: 70 % of the
// device memory free now, plus what the current copies hold), the one that re-sweeps the fewest entries (every
// segment but the last is recomputed once); the smallest footprint when none fits.
int choose_segment(const gs_batch* bt, double mem_budget) {
    if (mem_budget <= 0) {
        size_t fr = 0, tot = 0;
        if (hipMemGetInfo(&fr, &tot) != hipSuccess) fr = 0;
        mem_budget = 0.7 * double(fr) + (bt->seg ? double(grad_bytes(bt, bt->seg)) : 0.0);
    }
    int best = -1, smallest = 1;
    double best_cost = 0, small_bytes = -1;
    for (int sg = 1; sg <= bt->maxns; sg++) {
        const double bytes = double(grad_bytes(bt, sg));
        if (small_bytes < 0 || bytes < small_bytes) {
            small_bytes = bytes;
            smallest = sg;
        }
        if (bytes > mem_budget) continue;
        const int last_start = ((bt->maxns - 1) / sg) * sg;
        double cost = 0;
        for (size_t i = 0; i < bt->plans.size(); i++)
            for (int k = 0; k < std::min(bt->plans[i].ns, last_start); k++) cost += double(copy_entries(bt, i, k));
        if (best < 0 || cost <= best_cost) {
            best = sg;
            best_cost = cost;
        }
    }
    return best < 0 ? smallest : best;
}

template <class S>
int grad_t(gs_batch* bt) {
    const int ninst = int(bt->plans.size());
    const int seg = bt->seg, ns = bt->maxns;
    const int nseg = (ns + seg - 1) / seg;
    const int last = nseg - 1;
    // per-launch pointer arrays live in a device scratch of [maxns][ninst] (forward) and [seg][ninst] (recompute/back)
    const size_t rows = size_t(ns + seg + nseg);
    std::vector<void*> host(rows * size_t(ninst), nullptr);
    auto fwd_ptr = [&](int k) { return bt->dptrs + size_t(k) * ninst; };
    auto rec_ptr = [&](int j) { return bt->dptrs + size_t(ns + j) * ninst; };
    auto ck_ptr = [&](int s) { return bt->dptrs + size_t(ns + seg + s) * ninst; };
    // forward: checkpoint the input of every segment start; keep every input of the last segment
    for (int k = 0; k < ns; k++)
        for (int i = 0; i < ninst; i++)
            host[size_t(k) * ninst + i] = k / seg == last ? bt->stack[size_t(k - last * seg)][size_t(i)]
                                        : (k == seg_first(bt, seg, k / seg) ? bt->ckpt[size_t(k / seg)][size_t(i)]
                                                                            : nullptr);
    for (int j = 0; j < seg; j++)
        for (int i = 0; i < ninst; i++) host[size_t(ns + j) * ninst + i] = bt->stack[size_t(j)][size_t(i)];
    for (int s = 0; s < nseg; s++)
        for (int i = 0; i < ninst; i++) host[size_t(ns + seg + s) * ninst + i] = bt->ckpt[size_t(s)][size_t(i)];
    if (hipMemcpy(bt->dptrs, host.data(), sizeof(void*) * host.size(), hipMemcpyHostToDevice) != hipSuccess)
        return bfail(17, "pointer upload failed");
    hipEvent_t e0 = bt->ev0, e1 = bt->ev1, em;
    if (hipEventCreate(&em) != hipSuccess) return bfail(17, "event creation failed");
    (void)hipEventRecord(e0, bt->stream);
    hipLaunchKernelGGL(batch_init_kernel<S>, dim3(ninst), dim3(256), 0, bt->stream, bt->dinst, ninst, bt->dclock, ns);
    for (const Sweep& w : bt->common)
        if (int rc = launch_step<S>(bt, w, 1, fwd_ptr(w.k))) return rc;
    hipLaunchKernelGGL(batch_finish_kernel<S>, dim3(ninst), dim3(256), 0, bt->stream, bt->dinst, ninst);
    (void)hipEventRecord(em, bt->stream);
    hipLaunchKernelGGL(batch_lambda_init_kernel<S>, dim3(ninst), dim3(256), 0, bt->stream, bt->dinst, ninst);
    for (int s = last; s >= 0; s--) {
        const int k0 = s * seg, k1 = std::min(ns, k0 + seg);
        size_t a = 0, b = 0;                                // the segment's sweeps: a .. b - 1
        while (a < bt->common.size() && bt->common[a].k < k0) a++;
        for (b = a; b < bt->common.size() && bt->common[b].k < k1;) b++;
        if (s != last && a < b) {                           // recompute the segment from its checkpoint
            const Sweep& f = bt->common[a];
            if (int rc = launch_batch<S>(bt, kBRestore, f, BLaunch{f.k, 0, ck_ptr(s), nullptr})) return rc;
            for (size_t j = a; j < b; j++)
                if (int rc = launch_step<S>(bt, bt->common[j], 0, rec_ptr(bt->common[j].k - k0))) return rc;
        }
        for (size_t j = b; j-- > a;) {
            const Sweep& w = bt->common[j];
            if (int rc = launch_batch<S>(bt, kBBack, w, BLaunch{w.k, 0, rec_ptr(w.k - k0), nullptr})) return rc;
        }
    }
    (void)hipEventRecord(e1, bt->stream);
    if (hipEventSynchronize(e1) != hipSuccess || hipGetLastError() != hipSuccess) {
        (void)hipEventDestroy(em);
        return bfail(17, "gradient run failed");
    }
    float a = 0, c = 0;
    (void)hipEventElapsedTime(&a, e0, em);
    (void)hipEventElapsedTime(&c, e0, e1);
    bt->grad_fwd_ms = a;
    bt->grad_ms = c;
    (void)hipEventDestroy(em);
    return 0;
}

}  // namespace

extern "C" {

const char* gs_batch_last_error(void) { return g_berr.c_str(); }

int gs_batch_create(const gs_plan* const* plans, const int* lanes, int nplans, int storage, int device, gs_batch** out) {
    if (!plans || !lanes || nplans <= 0 || !out) return bfail(16, "bad argument");
    if (storage != GS_C64 && storage != GS_C128) return bfail(16, "storage must be GS_C64 or GS_C128");
    auto* bt = new gs_batch;
    bt->device = device;
    bt->storage = storage;
    bt->esz = storage == GS_C64 ? 8 : 16;
    bt->lu = storage == GS_C64 ? 2 : 1;
    auto bail = [&](int rc) {
        for (void* p : bt->allocs) (void)hipFree(p);
        (void)hipFree(bt->item_mem);
        (void)hipHostFree(bt->hout);
        delete bt;
        return rc;
    };
    if (hipSetDevice(device) != hipSuccess) return bail(bfail(17, "hipSetDevice failed"));
    for (int i = 0; i < nplans; i++) {
        if (!plans[i] || lanes[i] <= 0 || lanes[i] % kLanes) return bail(bfail(16, "lanes must be a positive multiple of 64"));
        bt->plans.push_back(plans[i]->p);
        bt->B.push_back(lanes[i]);
        bt->maxns = std::max(bt->maxns, plans[i]->p.ns);
    }
    bt->lg.resize(size_t(nplans));
    for (int i = 0; i < nplans; i++) bt->lg[size_t(i)].assign(size_t(bt->plans[size_t(i)].ns), bt->lg_default + 1);
    if (hipStreamCreate(&bt->stream) != hipSuccess || hipEventCreate(&bt->ev0) != hipSuccess ||
        hipEventCreate(&bt->ev1) != hipSuccess)
        return bail(bfail(17, "stream creation failed"));
    if (hipDeviceGetAttribute(&bt->clock_khz, hipDeviceAttributeWallClockRate, device) != hipSuccess || bt->clock_khz <= 0)
        return bail(bfail(17, "device clock rate unknown"));
    for (int i = 0; i < nplans; i++) {                    // strings and results of all instances, one buffer each
        bt->at_bits.push_back(bt->nbits);
        bt->nbits += size_t(lanes[i]) * size_t(bt->plans[size_t(i)].ns);
        bt->at_logp.push_back(bt->nout);
        bt->at_amp.push_back(bt->nout + size_t(lanes[i]));
        bt->nout += 3 * size_t(lanes[i]);
    }
    const size_t at_clock = bt->nout;
    bt->nhead = bt->nout += size_t(1 + bt->maxns);
    for (int i = 0; i < nplans; i++) {
        bt->at_cond.push_back(bt->nout);
        bt->nout += size_t(lanes[i]) * size_t(bt->plans[size_t(i)].ns);
    }
    bt->dbits = dalloc<int8_t>(bt, bt->nbits);
    bt->dout = dalloc<double>(bt, bt->nout);
    bt->dclock = reinterpret_cast<unsigned long long*>(bt->dout + at_clock);
    if (!bt->dbits || !bt->dout ||
        hipHostMalloc(reinterpret_cast<void**>(&bt->hout), bt->nout * sizeof(double) + std::max<size_t>(bt->nbits, 16), 0) !=
            hipSuccess)
        return bail(bfail(11, "batch buffer allocation failed"));
    bt->hbits = reinterpret_cast<int8_t*>(bt->hout + bt->nout);
    bt->hclock = reinterpret_cast<unsigned long long*>(bt->hout + at_clock);
    // whether every plan's strings fit the LDS: the table, then per step its descriptor, weights and sums.  One wave per
    // string up to 2^9 slots, else eight while the chip has a CU per string, four where several tables share a CU: with
    // 1 / 4 / 8 waves 4096 strings take 83 / 112 / 173 us at 2^9 complex64 slots, 261 / 200 / 280 at 2^11, 659 / 381 /
    // 438 at 2^12, 1096 / 526 / 506 at 2^12 complex128 ones; 64 strings 34 / 32 / 33, 72 / 45 / 43 and 136 / 65 / 58.
    int maxR = 0, lds_most = 0;
    for (const gs::Plan& P : bt->plans) maxR = std::max(maxR, P.R);
    bool lds_fits = maxR <= kLdsMaxR && bt->maxns <= kLdsSteps;
    if (lds_fits) {
        bt->lds_table = int(std::max<size_t>(bt->esz << maxR, 16));
        for (int b : bt->B) bt->lds_blocks += b;
        bt->lds_threads = maxR <= 9 ? 64 : bt->lds_blocks > 256 && bt->lds_table <= (32 << 10) ? 256 : 512;
        bt->lds_bytes = bt->lds_table + bt->maxns * int(sizeof(LStep) + 2 * sizeof(double2) + sizeof(double) * size_t(bt->lds_threads / 64));
        if (hipDeviceGetAttribute(&lds_most, hipDeviceAttributeMaxSharedMemoryPerBlock, device) != hipSuccess)
            return bail(bfail(17, "device LDS size unknown"));
        lds_fits = bt->lds_bytes + int(sizeof(double)) * kLdsSteps + 64 <= lds_most;
        if (!lds_fits) bt->lds_bytes = 0;
    }
    for (int i = 0; i < nplans; i++) {
        const gs::Plan& P = bt->plans[size_t(i)];
        const int B = lanes[i];
        BInst I{};
        I.B = B;
        I.ns = P.ns;
        I.mem = dalloc<char>(bt, (size_t(1) << P.R) * size_t(B) * bt->esz);
        if (!I.mem) return bail(bfail(11, "arena allocation failed"));
        std::vector<BStep> hs(size_t(P.ns));
        for (int k = 0; k < P.ns; k++) {
            const gs::StepInfo& si = P.steps[size_t(k)];
            BStep& s = hs[size_t(k)];
            memset(&s, 0, sizeof s);
            for (int j = 0; j < si.nk; j++) s.cols[j] = si.cols[size_t(j)];
            for (int j = 0; j < si.ntq; j++) {
                s.off[j] = si.off[j];
                s.tau0[j] = si.tau0[j];
                s.tau1[j] = si.tau1[j];
                s.par[j] = si.par[j];
                s.t0m |= uint32_t(si.tau0[j] & 1) << j;
                s.t1m |= uint32_t(si.tau1[j] & 1) << j;
                s.parm |= uint32_t(si.par[j] & 1) << j;
            }
            s.g = si.g;
            s.rhoc = si.rhoc;
            for (int bb = 0; bb < 2; bb++)
                for (int x = 0; x < 2; x++) {
                    s.mre[bb][x] = si.M[bb][x].real();
                    s.mim[bb][x] = si.M[bb][x].imag();
                }
            s.nk = si.nk;
            s.ntq = si.ntq;
            s.m = si.m;
        }
        std::vector<LStep> hl;
        if (lds_fits)
            for (const gs::StepInfo& si : P.steps) hl.push_back(make_lstep(si, P.R, bt->esz));
        // the instance's small buffers in one allocation: descriptors first, uploaded in one copy
        size_t used = 0;
        auto take = [&](size_t bytes) {
            const size_t at = used;
            used += (bytes + 255) & ~size_t(255);
            return at;
        };
        I.narrived = int(part_items(bt, size_t(i)) / kItemGroup);
        const size_t n_arrived = size_t(B / kLanes) * size_t(1 + I.narrived);
        const size_t o_steps = take(hs.size() * sizeof(BStep)), o_lsteps = take(hl.size() * sizeof(LStep)),
                     o_arrived = take(sizeof(unsigned) * n_arrived), head = used;   // counters start at 0
        const size_t o_prev = take(sizeof(double) * B), o_dead = take(sizeof(int) * B),
                     o_part = take(sizeof(double) * size_t(B / kLanes) * part_doubles(bt, size_t(i)));
        char* mem = dalloc<char>(bt, used);
        if (!mem) return bail(bfail(11, "batch buffer allocation failed"));
        std::vector<char> up(head);
        if (!hs.empty()) memcpy(up.data() + o_steps, hs.data(), hs.size() * sizeof(BStep));
        if (!hl.empty()) memcpy(up.data() + o_lsteps, hl.data(), hl.size() * sizeof(LStep));
        if (head && hipMemcpy(mem, up.data(), head, hipMemcpyHostToDevice) != hipSuccess)
            return bail(bfail(17, "plan upload failed"));
        bt->hsteps.push_back(std::move(hs));
        I.steps = reinterpret_cast<BStep*>(mem + o_steps);
        I.lsteps = reinterpret_cast<LStep*>(mem + o_lsteps);
        I.bitsT = bt->dbits + bt->at_bits[size_t(i)];
        I.prev = reinterpret_cast<double*>(mem + o_prev);
        I.dead = reinterpret_cast<int*>(mem + o_dead);
        I.cond = bt->dout + bt->at_cond[size_t(i)];
        I.logp = bt->dout + bt->at_logp[size_t(i)];
        I.amp = bt->dout + bt->at_amp[size_t(i)];
        I.arrived = reinterpret_cast<unsigned*>(mem + o_arrived);
        I.part = reinterpret_cast<double*>(mem + o_part);
        bt->hinst.push_back(I);
    }
    if (!bt->lds_bytes) {
        if (int rc = build_several(bt)) return bail(rc);
    } else {                                              // the largest plans' strings first
        bt->dinst = dalloc<BInst>(bt, bt->hinst.size());
        if (!bt->dinst || hipMemcpy(bt->dinst, bt->hinst.data(), bt->hinst.size() * sizeof(BInst), hipMemcpyHostToDevice) != hipSuccess)
            return bail(bfail(17, "instance upload failed"));
        std::vector<int> list(size_t(2 * nplans + 1), 0);
        for (int i = 0; i < nplans; i++) list[size_t(i)] = i;
        std::stable_sort(list.begin(), list.begin() + nplans,
                         [&](int a, int b) { return bt->plans[size_t(a)].R > bt->plans[size_t(b)].R; });
        for (int i = 0; i < nplans; i++)
            list[size_t(nplans + i + 1)] = list[size_t(nplans + i)] + lanes[list[size_t(i)]];
        bt->dorder = dalloc<int>(bt, list.size());
        bt->dblk0 = bt->dorder + nplans;
        if (!bt->dorder || hipMemcpy(bt->dorder, list.data(), list.size() * sizeof(int), hipMemcpyHostToDevice) != hipSuccess)
            return bail(bfail(17, "work list upload failed"));
    }
    bt->dptrs = dalloc<void*>(bt, size_t(4 * bt->maxns + 4) * size_t(nplans));
    if (!bt->dptrs) return bail(bfail(11, "allocation failed"));
    if (int rc = build_items(bt)) return bail(rc);
    if (hipDeviceSynchronize() != hipSuccess) return bail(bfail(17, "device synchronisation failed"));
    *out = bt;
    return 0;
}

void gs_batch_destroy(gs_batch* bt) {
    if (!bt) return;
    (void)hipSetDevice(bt->device);
    (void)hipStreamSynchronize(bt->stream);
    drop_graph(bt);
    free_grad(bt);
    for (void* p : bt->allocs) (void)hipFree(p);
    (void)hipFree(bt->item_mem);
    (void)hipHostFree(bt->hout);
    (void)hipEventDestroy(bt->ev0);
    (void)hipEventDestroy(bt->ev1);
    (void)hipStreamDestroy(bt->stream);
    delete bt;
}

// Set the log2 coset range per work item of instance i, step k (k < 0: all steps); rebuilds the work lists.
int gs_batch_set_tile(gs_batch* bt, int i, int k, int lg) {
    if (!bt || i < 0 || i >= int(bt->plans.size()) || lg < 0 || lg > 40) return bfail(16, "bad argument");
    const int ns = bt->plans[size_t(i)].ns;
    if (k >= ns) return bfail(16, "bad step");
    for (int kk = (k < 0 ? 0 : k); kk < (k < 0 ? ns : k + 1); kk++) {
        // the partial buffer was sized for the tiles chosen at creation; only coarser tiles are allowed later
        const int nk = bt->plans[size_t(i)].steps[size_t(kk)].nk;
        if (lg < std::min(nk, bt->lg_default)) return bfail(16, "tile below the default size");
        bt->lg[size_t(i)][size_t(kk)] = lg;
    }
    drop_graph(bt);
    bt->items_dirty = true;                               // rebuilt once, before the next run
    return 0;
}

// Work-list order: 0 round-robin over the XCDs (items group-major), 1 (default) each XCD takes consecutive
// group-major items, 2 each XCD takes consecutive coset-major items (all lane groups of a coset range together).
// Results do not depend on it.  Measured on one MI355X (uniform 2^10-coset tiles): n=60 x 1024 lanes forward
// 85.3 / 74.6 / 78.5 ms, gradient 218.5 / 204.2 / 211.8 ms; n=70 band 26 x 512 lanes 363.6 / 366.3 / 368.8 ms.
// The lists are rebuilt before the next run.
int gs_batch_set_xcd_items(gs_batch* bt, int on) {
    if (!bt) return bfail(16, "bad argument");
    if (on < 0 || on > 2) return bfail(16, "xcd item order must be 0, 1 or 2");
    bt->xcd_items = on;
    drop_graph(bt);
    bt->items_dirty = true;
    return 0;
}

// log2 cosets each lane gathers at once (0..3; default 2 for complex64, 1 for complex128).
int gs_batch_set_unroll(gs_batch* bt, int lu) {
    if (!bt || lu < 0 || lu > 3) return bfail(16, "unroll must be 0..3");
    bt->lu = lu;
    drop_graph(bt);
    return 0;
}

// Two or three consecutive steps per sweep where the plans allow it, and whole strings in LDS where all plans fit (on,
// default), or one step per sweep (off); the results differ at most by the order of FP64 sums.  A gradient's copies are
// laid out anew by its next call.
int gs_batch_set_pairs(gs_batch* bt, int on) {
    if (!bt) return bfail(16, "null batch");
    bt->pairs_on = on != 0;
    drop_graph(bt);
    (void)hipSetDevice(bt->device);
    (void)hipStreamSynchronize(bt->stream);
    free_grad(bt);
    bt->items_dirty = true;
    return 0;
}

int gs_batch_use_graph(gs_batch* bt, int on) {
    if (!bt) return bfail(16, "null batch");
    bt->use_graph = on != 0;
    if (!bt->use_graph) drop_graph(bt);
    return 0;
}

// Replace instance i's measurement matrices: M [ns][2][2] complex as re, im (M[k][b][x]); plan structure unchanged.
int gs_batch_set_matrices(gs_batch* bt, int i, const double* M) {
    if (!bt || !M || i < 0 || i >= int(bt->plans.size())) return bfail(16, "bad argument");
    auto& hs = bt->hsteps[size_t(i)];
    for (size_t k = 0; k < hs.size(); k++)
        for (int b = 0; b < 2; b++)
            for (int x = 0; x < 2; x++) {
                hs[k].mre[b][x] = M[((k * 2 + size_t(b)) * 2 + size_t(x)) * 2];
                hs[k].mim[b][x] = M[((k * 2 + size_t(b)) * 2 + size_t(x)) * 2 + 1];
            }
    (void)hipSetDevice(bt->device);
    if (hipMemcpy(const_cast<BStep*>(bt->hinst[size_t(i)].steps), hs.data(), hs.size() * sizeof(BStep),
                  hipMemcpyHostToDevice) != hipSuccess)
        return bfail(17, "matrix upload failed");
    return 0;
}

// Score one batch: bits[i] is instance i's [B_i][ns_i] forced strings (step order, 0/1); log2p[i] [B_i],
// cond[i] [B_i][ns_i] and amp[i] [B_i][2] (may be NULL) receive chain-mode outputs.  Returns after the device is done.
int gs_batch_score(gs_batch* bt, const int8_t* const* bits, double* const* log2p, double* const* cond,
                   double* const* amp) {
    if (!bt || !bits || !log2p) return bfail(16, "bad argument");
    if (hipSetDevice(bt->device) != hipSuccess) return bfail(17, "hipSetDevice failed");
    if (bt->items_dirty) {
        if (int rc = build_items(bt)) return rc;
        bt->items_dirty = false;
    }
    if (int rc = upload_bits(bt, bits)) return rc;
    if (hipEventRecord(bt->ev0, bt->stream) != hipSuccess) return bfail(17, "event record failed");
    if (bt->use_graph) {
        if (!bt->gexec)
            if (int rc = build_graph(bt)) return rc;
        if (hipGraphLaunch(bt->gexec, bt->stream) != hipSuccess) return bfail(17, "graph launch failed");
    } else {
        if (int rc = enqueue(bt)) return rc;
    }
    bool any_cond = false;
    for (size_t i = 0; i < bt->plans.size(); i++) any_cond = any_cond || (cond && cond[i]);
    if (hipEventRecord(bt->ev1, bt->stream) != hipSuccess ||
        hipMemcpyAsync(bt->hout, bt->dout, sizeof(double) * (any_cond ? bt->nout : bt->nhead), hipMemcpyDeviceToHost,
                       bt->stream) != hipSuccess ||
        hipStreamSynchronize(bt->stream) != hipSuccess)
        return bfail(17, "batch failed");
    float ms = 0;
    (void)hipEventElapsedTime(&ms, bt->ev0, bt->ev1);
    bt->last_ms = ms;
    bt->step_ms.assign(size_t(bt->maxns), -1.0);
    if (!bt->use_graph) {
        const bool lds = bt->lds_bytes && bt->pairs_on;
        size_t a = 0;
        for (int k = 0, u = 0; k < bt->maxns; k++) {      // the steps of one sweep end together
            while (a < bt->sweeps.size() && bt->sweeps[a].k <= k) u = bt->sweeps[a++].k;
            if (lds) u = k;
            bt->step_ms[size_t(k)] = double(bt->hclock[size_t(1 + u)] - bt->hclock[0]) / bt->clock_khz;
        }
    }
    for (size_t i = 0; i < bt->plans.size(); i++) {
        const size_t B = size_t(bt->B[i]), ns = size_t(bt->plans[i].ns);
        memcpy(log2p[i], bt->hout + bt->at_logp[i], sizeof(double) * B);
        if (cond && cond[i]) memcpy(cond[i], bt->hout + bt->at_cond[i], sizeof(double) * B * ns);
        if (amp && amp[i]) memcpy(amp[i], bt->hout + bt->at_amp[i], sizeof(double) * B * 2);
    }
    return 0;
}

// Gradient of every string's amplitude with respect to its per-step weights: G[i] [B_i][ns_i][2] complex (re, im)
// with G_k(x) = dZ / dM_k[b_k, x]; also log2p[i] and amp[i] (Z).  seg = steps per checkpoint segment (0: the largest
// whose copies fit in mem_budget bytes, all steps when they fit).  Returns the segment length used in *seg_used.
int gs_batch_grad(gs_batch* bt, const int8_t* const* bits, double* const* log2p, double* const* amp, double* const* G,
                  int seg, double mem_budget, int* seg_used) {
    if (!bt || !bits || !log2p || !G) return bfail(16, "bad argument");
    if (hipSetDevice(bt->device) != hipSuccess) return bfail(17, "hipSetDevice failed");
    if (bt->pairs_on && bt->hpairs.empty()) {
        if (int rc = build_several(bt)) return rc;
        bt->items_dirty = true;
    }
    if (bt->items_dirty) {
        if (int rc = build_items(bt)) return rc;
        bt->items_dirty = false;
    }
    if (seg <= 0) {                                       // automatic: chosen once per budget argument
        if (bt->seg && bt->auto_budget == mem_budget) seg = bt->seg;
        else seg = choose_segment(bt, mem_budget);
        bt->auto_budget = mem_budget;
    } else {
        bt->auto_budget = -1;
    }
    seg = std::min(std::max(seg, 1), bt->maxns);
    if (seg != bt->seg)
        if (int rc = alloc_grad(bt, seg)) return rc;
    if (seg_used) *seg_used = seg;
    if (int rc = upload_bits(bt, bits)) return rc;
    if (int rc = bt->storage == GS_C64 ? grad_t<float2>(bt) : grad_t<double2>(bt)) return rc;
    if (hipMemcpy(bt->hout, bt->dout, sizeof(double) * bt->nhead, hipMemcpyDeviceToHost) != hipSuccess)
        return bfail(17, "readback failed");
    for (size_t i = 0; i < bt->plans.size(); i++) {
        const size_t B = size_t(bt->B[i]), ns = size_t(bt->plans[i].ns);
        memcpy(log2p[i], bt->hout + bt->at_logp[i], sizeof(double) * B);
        if (amp && amp[i]) memcpy(amp[i], bt->hout + bt->at_amp[i], sizeof(double) * B * 2);
        if (hipMemcpy(G[i], bt->hinst[i].grad, sizeof(double) * B * ns * 4, hipMemcpyDeviceToHost) != hipSuccess)
            return bfail(17, "readback failed");
    }
    return 0;
}

// Device time of the last gs_batch_score (ms); step_end_ms[k] (may be NULL) the time from its start to the end of
// step k (without a graph; -1 where no instance has step k or when the batch ran as a graph).
double gs_batch_last_ms(const gs_batch* bt, double* step_end_ms) {
    if (!bt) return 0;
    if (step_end_ms)
        for (int k = 0; k < bt->maxns; k++) step_end_ms[k] = bt->step_ms.empty() ? -1 : bt->step_ms[size_t(k)];
    return bt->last_ms;
}

// Forward part and total device time (ms) of the last gs_batch_grad.
double gs_batch_grad_ms(const gs_batch* bt, double* forward_ms) {
    if (!bt) return 0;
    if (forward_ms) *forward_ms = bt->grad_fwd_ms;
    return bt->grad_ms;
}

}  // extern "C"
