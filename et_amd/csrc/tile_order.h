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
// than one part in 2^32 / d: the product's high half is the quotient while n * d < 2^32.  A launch with more blocks than
// that takes its rows in halves (ROWS_TOO_MANY).  (Correcting the quotient in the kernel instead took 0.05 us of every
// launch: 1000 rows 3072 -> 768 on the caller's arrays 8.80 / 8.85.)
inline unsigned magic_of(int d) { return d == 1 ? 0u : 0xFFFFFFFFu / (unsigned)d + 1u; }
struct QuotRem {
    int q, r;
};
ET_BOTH QuotRem quot_rem(int n, int d, unsigned magic) {
    const int q = magic ? (int)((uint64_t)(unsigned)n * magic >> 32) : n;
    return QuotRem{q, n - q * d};
}
inline bool quotients_fit(int64_t blocks, int64_t div) { return blocks <= INT32_MAX && div <= INT32_MAX && blocks * div < (int64_t)1 << 32; }
constexpr int ROWS_TOO_MANY = INT32_MIN; // a launcher's answer: not in one launch

// Outer x inner tiles, walked in groups of `group` outer ones: block `vid` goes through a group's outer tiles first, then to
// the next inner one.  The last group has `last` outer tiles.
struct GroupWalk {
    int total, div; // blocks; of a group
    int group, last;
    unsigned div_magic, group_magic, last_magic;
};
// (smaller groups where the quotient asks for it; false: not even single tiles)
inline bool group_walk(GroupWalk &w, int outer, int inner, int group) {
    while (group > 1 && !quotients_fit((int64_t)outer * inner, (int64_t)group * inner))
        group >>= 1;
    if (!quotients_fit((int64_t)outer * inner, (int64_t)group * inner))
        return false;
    const int last = outer - (outer - 1) / group * group;
    w = GroupWalk{outer * inner, group * inner, group, last, magic_of(group * inner), magic_of(group), magic_of(last)};
    return true;
}
ET_BOTH void group_walk_at(const GroupWalk &w, int vid, int &outer, int &inner) {
    const QuotRem of = quot_rem(vid, w.div, w.div_magic);
    outer = of.q;
    inner = of.r;
    if (w.group > 1) {
        const bool last = vid - of.r > w.total - w.div;
        const QuotRem in = last ? quot_rem(of.r, w.last, w.last_magic) : quot_rem(of.r, w.group, w.group_magic);
        outer = of.q * w.group + in.r;
        inner = in.q;
    }
}

} // namespace et
