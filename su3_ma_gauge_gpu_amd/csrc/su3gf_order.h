// su3gf_order.h -- the order in which a launch's blocks walk a lattice.
//
// The eight XCDs take blocks round-robin (block b runs on XCD b % 8), each
// with its own L2.  A launch over a lattice therefore deals the blocks out so
// that each XCD works through one contiguous eighth of a sequence in which a
// block's neighbours are near: the timeslices are walked in groups of `span`,
// t innermost, so that the t neighbours, a whole timeslice away in plain
// order, come just before or after, and the x neighbours (blocks per x row) *
// span places away.  A shorter span brings the x neighbours closer at the cost
// of the t neighbours across a group's boundary.
//
// Any lattice has such an order: where a timeslice's sites of a parity are no
// whole number of blocks, the blocks are counted off in timeslices of the next
// whole number (a neighbour is then at most one block from where it would
// be), and where the sequence is no multiple of 8 the last XCD's range is
// padded.  Plain order (block b is logical block b) spreads every
// neighbourhood over the eight L2s: the 24-bit gauge-transformation sweep takes
// 35.3 us per launch in plain order and 23.1 in this one at 28^4, 90.8 and 64.3
// at 36^4, 12.1 and 8.7 at 20^4; in FP64 71.9 and 53.3 at 28^4.
//
// Plain C++ as well, so that the order is checked on the CPU.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define SU3GF_HD __host__ __device__ __forceinline__
#else
#define SU3GF_HD inline
#endif

namespace su3gf {

// Division by a runtime constant d < 2^31 for dividends n < 2^31:
// q = (umulhi(n, m) + n) >> s with s = ceil(log2 d), m = 2^32 (2^s - d)/d + 1.
struct FastDiv {
    uint32_t d, m, s;
};

SU3GF_HD uint32_t fdiv(uint32_t n, const FastDiv &f)
{
    return ((uint32_t)(((uint64_t)n * f.m) >> 32) + n) >> f.s;
}

// the multiplier and shift of fdiv for divisor d (1 <= d < 2^31)
inline FastDiv make_fastdiv(uint32_t d)
{
    FastDiv f;
    f.d = d;
    f.s = 0;
    while ((1ull << f.s) < d) f.s++;
    f.m = (uint32_t)(((1ull << 32) * ((1ull << f.s) - d)) / d + 1);
    return f;
}

struct BlockOrder {
    uint32_t n;        // logical blocks
    uint32_t slice;    // blocks per timeslice, rounded up
    uint32_t span;     // timeslices walked together
    uint32_t per_xcd;  // places of the sequence per XCD
    FastDiv by_group, by_span;  // division by span * slice and by span
};

// the span of a lattice of Nt timeslices for the setting `request` (0 or one
// that does not fit: the default, Nt / 8 where that is whole, so that each
// XCD walks its own timeslices in one pass, else the largest divisor of Nt up
// to 8)
inline int order_span(int Nt, int request)
{
    const int own = Nt % 8 == 0 ? Nt / 8 : Nt;  // a span divides this
    if (request > 0 && own % request == 0) return request;
    if (Nt % 8 == 0) return own;
    int s = 1;
    for (int d = 2; d <= 8; d++)
        if (Nt % d == 0) s = d;
    return s;
}

inline BlockOrder make_block_order(int64_t n, int Nt, int request)
{
    BlockOrder o;
    o.n = (uint32_t)n;
    o.slice = (uint32_t)((n + Nt - 1) / Nt);
    o.span = (uint32_t)order_span(Nt, request);
    o.per_xcd = (uint32_t)(((int64_t)o.slice * Nt + 7) / 8);
    o.by_group = make_fastdiv(o.span * o.slice);
    o.by_span = make_fastdiv(o.span);
    return o;
}

inline int64_t order_grid(const BlockOrder &o) { return 8 * (int64_t)o.per_xcd; }

// the logical block of block b of the launch, or -1 for a padding block
SU3GF_HD int64_t ordered_block(const BlockOrder &o, uint32_t b)
{
    const uint32_t place = (b & 7) * o.per_xcd + (b >> 3);
    const uint32_t group = fdiv(place, o.by_group);
    const uint32_t rem = place - group * o.span * o.slice;
    const uint32_t q = fdiv(rem, o.by_span);
    const uint32_t L = (group * o.span + (rem - q * o.span)) * o.slice + q;
    return L < o.n ? (int64_t)L : -1;
}

}  // namespace su3gf
