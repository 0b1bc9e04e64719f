// Which block of a launch a workgroup takes: quotients by numbers that the host knows, and the dense product's walk.  No
// GPU header in here: the host compiler takes the file as well.
#pragma once
#include <cstdint>

#ifdef __HIPCC__
#define ET_BOTH __host__ __device__ __forceinline__
#else
#define ET_BOTH inline
#endif

namespace et {

// A division in front of a kernel's first request costs tens of vector instructions, fetched cold at every launch; this is
// a scalar multiplication, and another one for the rest.  magic_of(d) is 2^32 / d rounded up (0: d = 1), too large by less
// than one part in 2^32 / d: while n * d < 2^32 the product's high half is the quotient, for every other n < 2^31 it is the
// quotient or one more, and the rest tells.
inline unsigned magic_of(int d) { return d == 1 ? 0u : 0xFFFFFFFFu / (unsigned)d + 1u; }
struct QuotRem {
    int q, r;
};
ET_BOTH QuotRem quot_rem_small(int n, int d, unsigned magic) { // n * d < 2^32
    const unsigned q = magic ? (unsigned)((uint64_t)(unsigned)n * magic >> 32) : (unsigned)n;
    return QuotRem{(int)q, (int)((unsigned)n - q * (unsigned)d)};
}
ET_BOTH QuotRem quot_rem(int n, int d, unsigned magic) {
    const QuotRem v = quot_rem_small(n, d, magic);
    return v.r < 0 ? QuotRem{v.q - 1, v.r + d} : v;
}

// Outer x inner tiles, walked in groups of `group` outer ones: block `vid` goes through a group's outer tiles first, then to
// the next inner one.  The last group has `last` outer tiles.
struct GroupWalk {
    int total, div; // blocks; of a group
    int group, last;
    unsigned div_magic, group_magic, last_magic;
};
inline GroupWalk group_walk(int outer, int inner, int group) {
    const int last = outer - (outer - 1) / group * group;
    return GroupWalk{outer * inner, group * inner, group, last, magic_of(group * inner), magic_of(group), magic_of(last)};
}
ET_BOTH void group_walk_at(const GroupWalk &w, int vid, int &outer, int &inner) {
    const QuotRem of = quot_rem(vid, w.div, w.div_magic);
    outer = of.q;
    inner = of.r;
    if (w.group > 1) {
        const bool last = vid - of.r > w.total - w.div;
        const QuotRem in = last ? quot_rem_small(of.r, w.last, w.last_magic) : quot_rem_small(of.r, w.group, w.group_magic);
        outer = of.q * w.group + in.r;
        inner = in.q;
    }
}

} // namespace et
