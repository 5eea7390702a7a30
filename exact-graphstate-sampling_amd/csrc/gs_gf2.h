// GF(2) linear algebra over 64-bit vectors (host): a basis kept in echelon form together with the combination of the
// added vectors that gives each row, so membership and coordinates cost one pass over the rows.
#pragma once
#include <cstdint>

namespace gs {

inline int parity(uint64_t x) { return __builtin_parityll(x); }

struct GfBasis {
    uint64_t row[64] = {};      // row[b]: the row whose top bit is b (0: none)
    uint64_t comb[64] = {};     // the added vectors (bit i: the i-th) whose XOR is that row
    int n = 0;                  // vectors added

    // Adds v when it raises the rank.
    bool add(uint64_t v) {
        uint64_t c = uint64_t(1) << n;
        reduce(v, c);
        if (!v) return false;
        const int b = 63 - __builtin_clzll(v);
        row[b] = v;
        comb[b] = c;
        n++;
        return true;
    }
    // The combination of the added vectors that gives x; false when x is outside their span.
    bool solve(uint64_t x, uint64_t& coef) const {
        coef = 0;
        reduce(x, coef);
        return x == 0;
    }
    // Mask m with parity(x & m) == parity(combination of x & f) for every x of the span.
    uint64_t form(uint64_t f) const {
        uint64_t m = 0;
        for (int b = 0; b < 64; b++)
            if (row[b] && (parity(comb[b] & f) ^ parity(row[b] & m))) m |= uint64_t(1) << b;
        return m;
    }
    // What is left of x modulo the span: equal for x and y when their difference is in it.
    uint64_t residue(uint64_t x) const {
        for (uint64_t left = x; left;) {
            const int b = 63 - __builtin_clzll(left);
            x ^= row[b];
            left = x & ((uint64_t(1) << b) - 1);
        }
        return x;
    }
    bool has(uint64_t x) const { return residue(x) == 0; }

private:
    void reduce(uint64_t& v, uint64_t& c) const {
        for (uint64_t left = v; left;) {
            const int b = 63 - __builtin_clzll(left);
            if (row[b]) {
                v ^= row[b];
                c ^= comb[b];
            }
            left = v & ((uint64_t(1) << b) - 1);
        }
    }
};

}  // namespace gs
