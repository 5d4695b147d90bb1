// Column ranges of the strip sweeps (pf_kernels.hip): which levels of a column a
// momentum sweep reads and updates, and which of them one strip hands to the next.
// Plain integer arithmetic: a host compiler takes it with the function
// attributes defined away.
#pragma once

// Metadata of a sweep position as the strips' rows keep it (uniform); a column
// outside the sub-domains or the sweep has VI = -1.
struct StripCol { int KK, VI, ks, kend, veg; };   // ks: KSTART, kend: first level the sweep updates
struct StripLevels { int lo, hi; };               // lo > hi: none

// from the four words of Dom::meta
template <int COMP>
__host__ __device__ __forceinline__ StripCol strip_col(int x, int y, int z, int w) {
    StripCol c;
    c.KK = x;
    c.VI = (z & 0x10000) ? y : -1;
    c.ks = z & 0xffff;
    // U and V skip the levels inside the building or its upstream neighbour; W
    // updates every level from KSTART
    c.kend = (COMP == 2) ? c.ks : (COMP == 0) ? (w & 0xffff) + 1 : ((w >> 16) & 0xffff) + 1;
    c.veg = z & 0x20000;
    return c;
}

// first level with a source: the sweep reads the column's four neighbours from here to VI
template <int COMP>
__host__ __device__ __forceinline__ int strip_first(const StripCol &c) { return COMP == 2 ? c.ks : c.KK + 1; }

// Column a of a strip's last row (p) and column a of the next strip's row 0 (c) read
// each other: c the new values of p where p has them (p.kend..VI), p the old values
// of c at all its source levels.  p hands on one word for each of its source
// levels, below kend too, and c waits for the words of all levels both columns have.
// So c stores nothing before p has read it: the levels c stores lie in its own
// source range, those of them that p reads in both ranges, and a word leaves p only
// after p's reads.  Waiting for the updated levels alone would not do: U and V
// update a low roof beside a wall higher than the sub-domain only above all levels
// of open ground next to it (kend > c.VI), but read that ground from the roof up.
template <int COMP>
__host__ __device__ __forceinline__ StripLevels hand_sent(const StripCol &p) {
    return StripLevels{strip_first<COMP>(p), p.VI};
}
template <int COMP>
__host__ __device__ __forceinline__ StripLevels hand_needed(const StripCol &c, const StripCol &p) {
    const int a = strip_first<COMP>(c), b = strip_first<COMP>(p);
    return StripLevels{a > b ? a : b, c.VI < p.VI ? c.VI : p.VI};
}
