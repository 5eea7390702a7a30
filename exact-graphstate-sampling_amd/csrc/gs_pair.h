// Two consecutive steps as one sweep: the geometry (host) and the butterflies of both steps (device), shared by the
// batched kernels (a string per lane) and the in-place engine's chain sweeps (a super-coset per lane).
#pragma once
#include <cstring>
#include <vector>

#include "gs_gf2.h"
#include "gs_math.h"
#include "gs_plan.h"

namespace gs {

// L1, the live table between the steps, splits into W, the span of step k+1's slot offsets (relative to its first) and
// step k's g, and a complement C inside the span of step k's columns.  A super-coset a + W (a in C) is closed under both
// steps: its ni step-k cosets i (at a ^ D[i]) give the elements (i, t) at a ^ D[i] ^ t g, which are all the slots of
// its step-(k+1) cosets (two of them when step k has two outputs and g is no slot offset, else one), so it goes from
// step k's inputs to step k+1's outputs without the table between them ever being stored.
struct PairDesc {
    uint64_t cols[40];   // columns of the super-coset coordinates
    uint64_t D[4];
    uint64_t lab[4];     // D[i], or D[i] ^ g where it is labelled output 1: the base address of step k's coset
    uint64_t g, d1, d2;  // step k's g; step k+1's second and third offsets relative to the first
    uint64_t o0;         // step k+1's first offset
    uint8_t pn[40];      // per coordinate: bit 0 step k's sign, bit 1 step k+1's sign, bits 2-3 step k+1's slot index
    uint8_t pd[4], pg;   // the same of D[i] (bit 4: the output index it is labelled with) and of g
    uint8_t pc;          // the same of step k+1's first offset
    int nk;              // super-coset coordinates
    int ni, mo, deg;     // step-k cosets (0: no pair), outputs of step k, 1 when g is among step k+1's slot offsets
};

// Steps k and k+1 of a plan as one sweep; false (ni = 0) when a super-coset cannot be closed or would write a slot that
// another super-coset still reads.  units: coordinates whose columns are the unit bits 1, 2, 4, ... first, and those that
// change step k+1's slot index last (the in-place engine's lanes take the first coordinates).
inline bool make_pair(const StepInfo& s0, const StepInfo& s1, bool units, PairDesc& p) {
    memset(&p, 0, sizeof p);
    GfBasis live;                                     // L1: the columns of step k (its output 0), then g
    for (uint64_t c : s0.cols)
        if (!live.add(c)) return false;
    if (s0.m == 2 && !live.add(s0.g)) return false;
    const int lg1 = s1.ntq == 4 ? 2 : s1.ntq == 2 ? 1 : 0;
    uint64_t d[4] = {0, 0, 0, 0};
    for (int j = 1; j < s1.ntq; j++) d[j] = s1.off[j] ^ s1.off[0];
    if (s1.ntq == 4 && (d[3] != (d[1] ^ d[2]))) return false;
    GfBasis next;                                     // the same space as step k+1 reads it: its columns, then d1, d2
    for (uint64_t c : s1.cols)
        if (!live.has(c) || !next.add(c)) return false;
    for (int j = 1; j <= lg1; j++)
        if (!live.has(d[j]) || !next.add(d[j])) return false;
    if (next.n != live.n || !live.has(s1.off[0])) return false;
    // parities of an address of L1: bit 0 step k's sign, bit 1 step k+1's, bits 2-3 its slot, bit 4 step k's output
    const uint64_t forms[5] = {live.form(s0.rhoc & ((uint64_t(1) << s0.nk) - 1)),
                               next.form(s1.rhoc & ((uint64_t(1) << s1.nk) - 1)), next.form(uint64_t(1) << s1.nk),
                               next.form(uint64_t(2) << s1.nk), live.form(uint64_t(1) << s0.nk)};
    auto nib = [&](uint64_t x) {
        int n = 0;
        for (int i = 0; i < 5; i++) n |= parity(x & forms[i]) << i;
        return uint8_t(n);
    };
    GfBasis slots;
    for (int j = 1; j <= lg1; j++) (void)slots.add(d[j]);
    p.deg = s0.m == 2 && slots.has(s0.g);
    p.mo = s0.m;
    const int ni = p.deg ? s1.ntq / 2 : s1.ntq;
    if (p.deg) p.D[1] = ni == 2 ? (d[1] != s0.g ? d[1] : d[2]) : 0;
    else
        for (int i = 1; i < ni; i++) p.D[i] = d[i];
    GfBasis W;
    if (s0.m == 2) (void)W.add(s0.g);
    for (int i = 1; i < ni; i++) (void)W.add(p.D[i]);
    std::vector<uint64_t> cand;                       // candidates for C, all in the span of step k's columns
    if (units) {
        for (int i = 0; i < 40; i++)
            if (live.has(uint64_t(1) << i) && !(nib(uint64_t(1) << i) & 0x1c)) cand.push_back(uint64_t(1) << i);
        uint64_t piv[4] = {0, 0, 0, 0};               // columns by slot index (1, 2, 3) once one is found
        for (uint64_t c : s0.cols) {
            for (int q = 1; q < 4 && (nib(c) >> 2 & 3); q++)
                if (piv[q] && (nib(c) >> 2 & 3) == q) c ^= piv[q];
            const int q = nib(c) >> 2 & 3;
            if (!q) {
                cand.push_back(c);
                continue;
            }
            for (int o = 1; o < 4; o++)
                if (o != q && piv[o] && !piv[o ^ q]) piv[o ^ q] = piv[o] ^ c;
            piv[q] = c;
        }
        for (int q = 1; q < 4; q++)
            if (piv[q]) cand.push_back(piv[q]);
    } else {
        cand = s0.cols;
    }
    GfBasis C;
    for (uint64_t c : cand)
        if (W.add(c)) {
            (void)C.add(c);
            p.cols[p.nk] = c;
            p.pn[p.nk++] = uint8_t(nib(c) & 15);
        }
    if (W.n != live.n) return false;
    p.g = s0.m == 2 ? s0.g : 0;
    p.d1 = d[1];
    p.d2 = lg1 == 2 ? d[2] : 0;
    p.o0 = s1.off[0];
    p.pg = s0.m == 2 ? nib(s0.g) : 0;
    p.pc = nib(s1.off[0]);
    for (int i = 0; i < ni; i++) {
        p.pd[i] = nib(p.D[i]);
        p.lab[i] = p.D[i] ^ ((p.pd[i] & 16) ? s0.g : 0);
    }
    // slots read and written relative to the super-coset's base: no two super-cosets may meet on a written slot
    std::vector<uint64_t> rd, wr;
    for (int i = 0; i < ni; i++)
        for (int q = 0; q < s0.ntq; q++) rd.push_back(p.lab[i] ^ s0.off[q]);
    for (int c = 0; c < (p.deg ? 1 : p.mo); c++)
        for (int j = 0; j < s1.ntq; j++) {
            const uint64_t at = (c ? s0.g : 0) ^ s1.off[0] ^ d[j];
            wr.push_back(at);
            if (s1.m == 2) wr.push_back(at ^ s1.g);
        }
    const std::vector<uint64_t> rd0 = rd, wr0 = wr;
    for (auto* v : {&rd, &wr})
        for (uint64_t& u : *v) u = C.residue(u);
    // one and the same slot of a super-coset meets itself only
    auto clash = [&](const std::vector<uint64_t>& x, const std::vector<uint64_t>& y, const std::vector<uint64_t>& x0,
                     const std::vector<uint64_t>& y0) {
        for (size_t i = 0; i < x.size(); i++)
            for (size_t j = 0; j < y.size(); j++)
                if (x[i] == y[j] && x0[i] != y0[j]) return true;
        return false;
    };
    if (clash(wr, rd, wr0, rd0) || clash(wr, wr, wr0, wr0) || clash(rd, rd, rd0, rd0)) return false;
    p.ni = ni;
    return true;
}

// ---- device

__device__ __forceinline__ double2 flip_if(double2 a, uint32_t s) {          // (-1)^s a
    const int m = int(s << 31);
    return make_double2(__hiloint2double(__double2hiint(a.x) ^ m, __double2loint(a.x)),
                        __hiloint2double(__double2hiint(a.y) ^ m, __double2loint(a.y)));
}
// One slot's terms: t0, t1 (outputs of its x = 0 and x = 1 terms) are wave-uniform, the sign may be per lane.
__device__ __forceinline__ void route_one(double2 (&A)[2][2], double2 w, uint32_t t0, uint32_t t1, uint32_t neg) {
    const double2 ws = flip_if(w, neg);
    if (t0) A[1][0] = cadd(A[1][0], w); else A[0][0] = cadd(A[0][0], w);     // uniform branches
    if (t1) A[1][1] = cadd(A[1][1], ws); else A[0][1] = cadd(A[0][1], ws);
}

// What the sweep needs of the two steps: step k's offsets and routing (a bit per offset), step k+1's g, outputs, routing.
struct PairSteps {
    const uint64_t* off;
    uint64_t g1;
    int m1;
    uint32_t t0m, t1m, parm, u0m, u1m, uparm;
};

// Uniform per-launch constants of a pair.  pa: the parities of a super-coset's base as in PairDesc::pn (signs; may be
// per lane), ph: the same for the slot index (wave-uniform).
struct PairRegs {
    uint64_t lab[4], off[4], g, d1, d2, o0, g1;
    uint32_t pd[4], pg, pc, t0m, t1m, parm, u0m, u1m, uparm;
    int m1;
    __device__ PairRegs(const PairDesc& P, const PairSteps& s) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            lab[i] = P.lab[i];
            off[i] = s.off[i];
            pd[i] = P.pd[i];
        }
        g = P.g; d1 = P.d1; d2 = P.d2; o0 = P.o0; pg = P.pg; pc = P.pc;
        g1 = s.g1;
        m1 = s.m1;
        t0m = s.t0m; t1m = s.t1m; parm = s.parm;
        u0m = s.u0m; u1m = s.u1m; uparm = s.uparm;
    }
    // slot of step k+1 at element (i, t), and its coset's sign
    __device__ uint32_t slot(uint32_t ph, int i, int t) const { return ((ph ^ pd[i] ^ (t ? pg : 0) ^ pc) >> 2) & 3; }
    __device__ uint32_t sign(uint32_t pa, int c) const { return ((pa ^ (c ? pg : 0) ^ pc) >> 1) & 1; }
    // output 0 of step-(k+1) coset c of the super-coset at a
    __device__ uint64_t out(uint64_t a, uint32_t ph, int c) const {
        const uint32_t j = slot(ph, 0, c);
        return a ^ (c ? g : 0) ^ o0 ^ ((j & 1) ? d1 : 0) ^ ((j & 2) ? d2 : 0);
    }
};

// Slot sums of step-k coset i: A[t][x], t the element label (output index t ^ label bit).
template <class S, int NQ>
__device__ __forceinline__ void pair_route0(const PairRegs& r, const S (&v)[NQ], uint32_t pa, int i,
                                            double2 (&A)[2][2]) {
    A[0][0] = A[0][1] = A[1][0] = A[1][1] = make_double2(-0.0, -0.0);
    const uint32_t pc = (pa ^ r.pd[i]) & 1, sw = (r.pd[i] >> 4) & 1;
#pragma unroll
    for (int q = 0; q < NQ; q++)
        route_one(A, Cx<S>::widen(v[q]), ((r.t0m >> q) & 1) ^ sw, ((r.t1m >> q) & 1) ^ sw, pc ^ ((r.parm >> q) & 1));
}

// Slot sums of step-(k+1) coset c from the elements e[i][t] (already rounded to the storage type).
template <int NI, int MO, bool DEG>
__device__ __forceinline__ void pair_route1(const PairRegs& r, const double2 (&e)[NI][MO], uint32_t pa, uint32_t ph,
                                            int c, double2 (&A)[2][2]) {
    A[0][0] = A[0][1] = A[1][0] = A[1][1] = make_double2(-0.0, -0.0);
    const uint32_t sg = r.sign(pa, c);
#pragma unroll
    for (int i = 0; i < NI; i++)
#pragma unroll
        for (int t = 0; t < MO; t++) {
            if (!DEG && t != c) continue;
            const uint32_t j = r.slot(ph, i, t);
            route_one(A, e[i][t], (r.u0m >> j) & 1, (r.u1m >> j) & 1, sg ^ ((r.uparm >> j) & 1));
        }
}

}  // namespace gs
