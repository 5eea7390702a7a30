// Runs of butterfly steps: consecutive steps of two slots and two outputs whose outputs take the place of their slots
// (g is the slot offset), over one live table.  Step i pairs the entries x and x ^ dir[i]; with slot index and sign
// affine parities of the address, D such steps act on the 2^D entries of a + span(dir) alone.  Geometry (host) and the
// butterflies (device), shared by the in-place engine's sweeps (a group per lane) and the batched ones (a string per lane).
#pragma once
#include <cstring>
#include <type_traits>
#include <utility>
#include <vector>

#include "gs_device.h"
#include "gs_gf2.h"
#include "gs_pair.h"
#include "gs_plan.h"

namespace gs {

constexpr int kMaxFly = 4;
// Coordinates of the complement of span(dir); see make_fly for their order.
struct FlyDesc {
    uint64_t cols[40];
    uint64_t dir[kMaxFly];
    uint8_t pn[40];                    // per coordinate: bit i the change of step i's sign, bit 4 + i of its slot index
    uint8_t dn[kMaxFly], cn;           // the same of the directions and of the coordinate origin
    uint8_t route[kMaxFly], par[kMaxFly];   // Route of step i; sign of its slot 1's x = 1 term relative to slot 0's
    int nk, d;                         // coordinates, directions (0: none)
    int lg_grid, lg_iter, xcd;
};

// A step that acts in place on pairs of slots.
inline bool is_fly(const StepInfo& s) { return s.ntq == 2 && s.m == 2 && s.g == (s.off[0] ^ s.off[1]); }

// Canonical route of a butterfly step with its slots in the order `slot` (slot[j]: index into off), or -1.
inline int fly_route(const StepInfo& s, int (&slot)[2]) {
    slot[0] = 0;
    slot[1] = 1;
    if (s.tau0[0] == 0 && s.tau0[1] == 0 && s.tau1[0] == 1 && s.tau1[1] == 1) return kRouteSplit;
    if (s.tau0[0] == s.tau0[1] || s.tau1[0] == s.tau1[1]) return -1;
    if (s.tau0[0] == 1) std::swap(slot[0], slot[1]);
    return s.tau1[slot[0]] == 1 ? kRouteMixA : kRouteMixB;
}

// Steps p[0..d-1] of a plan as one butterfly of d directions.  With lr = 1 coordinate 0 is the unit bit 0 (one aligned
// run of 2 per thread); none of the first lr + lanes coordinates changes a slot index.
inline bool make_fly(const StepInfo* const* p, int d, int lr, int lanes, FlyDesc& f) {
    memset(&f, 0, sizeof f);
    GfBasis live[kMaxFly], W;
    uint64_t o0[kMaxFly];
    for (int i = 0; i < d; i++) {
        const StepInfo& s = *p[i];
        int slot[2];
        const int r = is_fly(s) ? fly_route(s, slot) : -1;
        if (r < 0 || s.nk != p[0]->nk) return false;
        f.route[i] = uint8_t(r);
        f.par[i] = uint8_t((s.par[slot[0]] ^ s.par[slot[1]]) & 1);
        o0[i] = s.off[slot[0]];
        f.dir[i] = s.off[0] ^ s.off[1];
        for (uint64_t c : s.cols)
            if (!live[i].add(c) || (i && !live[0].has(c))) return false;
        if (!live[i].add(f.dir[i]) || (i && !live[0].has(f.dir[i])) || !W.add(f.dir[i])) return false;
        // output 0 is written at the coset's base, which has to be the place of slot 0 (output 1 at slot 1's then)
        if (o0[i] != 0) return false;
        f.cn |= uint8_t((s.par[slot[0]] & 1) << i);
    }
    uint64_t sign[kMaxFly], index[kMaxFly];
    for (int i = 0; i < d; i++) {
        sign[i] = live[i].form(p[i]->rhoc & ((uint64_t(1) << p[i]->nk) - 1));
        index[i] = live[i].form(uint64_t(1) << p[i]->nk);
    }
    auto bits = [&](uint64_t x) {
        int n = 0;
        for (int i = 0; i < d; i++) n |= (parity(x & sign[i]) << i) | (parity(x & index[i]) << (4 + i));
        return uint8_t(n);
    };
    for (int i = 0; i < d; i++) f.dn[i] = bits(f.dir[i]);
    // complement of the directions: unit bits that leave every slot index alone, then other such vectors, then the rest
    std::vector<uint64_t> cand, piv;
    for (int i = 0; i < 40; i++)
        if (live[0].has(uint64_t(1) << i) && !(bits(uint64_t(1) << i) >> 4)) cand.push_back(uint64_t(1) << i);
    std::vector<uint64_t> all(p[0]->cols);
    all.push_back(f.dir[0]);
    GfBasis idx;                                          // slot-index patterns of piv
    for (uint64_t c : all) {
        int j = bits(c) >> 4;
        uint64_t comb = 0;
        if (j && idx.solve(j, comb)) {
            for (size_t q = 0; q < piv.size(); q++)
                if ((comb >> q) & 1) c ^= piv[q];
            j = 0;
        }
        if (!j) cand.push_back(c);
        else {
            (void)idx.add(uint64_t(j));
            piv.push_back(c);
        }
    }
    cand.insert(cand.end(), piv.begin(), piv.end());
    for (uint64_t c : cand)
        if (c && W.add(c)) {
            f.cols[f.nk] = c;
            f.pn[f.nk++] = bits(c);
        }
    if (W.n != live[0].n || f.nk < lr + lanes || (lr && f.cols[0] != 1)) return false;
    for (int q = 0; q < lr + lanes; q++)
        if (f.pn[q] >> 4) return false;
    if (lr)
        for (int q = 1; q < f.nk; q++)                    // the run's bit in coordinate 0 only
            if (f.cols[q] & 1) {
                f.cols[q] ^= 1;
                f.pn[q] ^= f.pn[0];
            }
    f.d = d;
    return true;
}

// ---- device

__device__ __forceinline__ uint32_t uniform_byte(uint8_t v) { return uint32_t(__builtin_amdgcn_readfirstlane(int(v))); }

// A pair of step i: lo is slot J, hi slot 1 - J, s the coset's sign; J, route and par are uniform.  Outputs take their
// places.
template <int ROUTE>
__device__ __forceinline__ void fly_pair(uint32_t par, uint32_t J, uint32_t s, double2 lo, double2 hi, double2 w0,
                                         double2 w1, double2& ylo, double2& yhi) {
    const uint32_t slo = s ^ (J ? par : 0), shi = s ^ (J ? 0 : par);   // signs of the x = 1 terms
    if constexpr (ROUTE == kRouteMixA) {
        ylo = cfma(w0, lo, flip_if(cmul(w1, hi), shi));
        yhi = cfma(w0, hi, flip_if(cmul(w1, lo), slo));
    } else if constexpr (ROUTE == kRouteMixB) {
        ylo = cfma(w0, lo, flip_if(cmul(w1, lo), slo));
        yhi = cfma(w0, hi, flip_if(cmul(w1, hi), shi));
    } else {
        const double2 u = cmul(w0, cadd(lo, hi));
        const double2 v = flip_if(cmul(w1, cadd(lo, flip_if(hi, par))), slo);
        ylo = J ? v : u;
        yhi = J ? u : v;
    }
}

// Backward through a pair: llo, lhi are lambda at the outputs' places; G(x) += sum over outputs of lambda times the
// routed inputs, and lambda goes to the slots.
template <int ROUTE>
__device__ __forceinline__ void fly_pair_back(uint32_t par, uint32_t J, uint32_t s, double2 lo, double2 hi, double2 w0,
                                              double2 w1, double2& llo, double2& lhi, double2 (&G)[2]) {
    const uint32_t slo = s ^ (J ? par : 0), shi = s ^ (J ? 0 : par);
    const double2 xl = flip_if(lo, slo), xh = flip_if(hi, shi);
    const double2 a = llo, b = lhi;
    if constexpr (ROUTE == kRouteSplit) {
        const double2 m0 = J ? b : a, m1 = J ? a : b, y = cmul(w1, m1);
        G[0] = cfma(m0, cadd(lo, hi), G[0]);
        G[1] = cfma(m1, cadd(xl, xh), G[1]);
        llo = cfma(w0, m0, flip_if(y, slo));
        lhi = cfma(w0, m0, flip_if(y, shi));
    } else {
        constexpr bool MIXA = ROUTE == kRouteMixA;
        G[0] = cfma(a, lo, cfma(b, hi, G[0]));
        G[1] = cfma(a, MIXA ? xh : xl, cfma(b, MIXA ? xl : xh, G[1]));
        llo = cfma(w0, a, flip_if(cmul(w1, MIXA ? b : a), slo));
        lhi = cfma(w0, b, flip_if(cmul(w1, MIXA ? a : b), shi));
    }
}

// f(std::integral_constant<int, route>) for the three routes of a butterfly (uniform branch).
template <class F>
__device__ __forceinline__ void fly_route_of(int route, F&& f) {
    if (route == kRouteMixA) f(std::integral_constant<int, kRouteMixA>{});
    else if (route == kRouteMixB) f(std::integral_constant<int, kRouteMixB>{});
    else f(std::integral_constant<int, kRouteSplit>{});
}

// f(std::integral_constant<int, i>) for i = 0 .. N-1.
template <class F, int... I>
__device__ __forceinline__ void fly_each(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}

}  // namespace gs
