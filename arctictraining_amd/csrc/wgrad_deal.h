// How the tiles of weight gradients of uneven loads are dealt to 256 workgroups by depth (gemm_pp.hip): whole numbers only, constexpr, so that it
// is replayed on the host as well.
//
// A tile is as deep as its expert has rows.  Experts are taken in the order of their depth, their tiles in turns to all workgroups; where
// the next ones are lower by a fifth or more, the workgroups that the last turn did not reach are first filled up with those.
#pragma once

namespace amoe_deal {

constexpr int ALL = 256;

// An expert: tiles [0, fill) go in turns to the `behind` workgroups from `from` on, the first to the one `skip` further, the others to all
// from `from2` on.
struct Record {
    int from, skip, behind, fill, from2;
    constexpr unsigned word() const { return (unsigned)(from | skip << 8 | from2 << 16); }
    static constexpr Record of(unsigned word, int behind, int fill)
    {
        return {(int)(word & 255u), (int)(word >> 8 & 255u), behind, fill, (int)(word >> 16 & 255u)};
    }
};

// the records of experts with `per` tiles of depth d each, d falling from one to the next
struct Walk {
    int from = 0, behind = ALL, skip = 0;
    int left = 0;     // depth that the workgroups behind lack
    int last = 0;     // depth of the tiles dealt to all
    constexpr Record next(int d, int per)
    {
        if (behind == ALL && 5 * d < 4 * last && skip) {
            from = (from + skip) & 255;
            behind = ALL - skip;
            left = behind * last;
            skip = 0;
        }
        Record r = {from, skip, behind, 0, 0};
        if (behind < ALL) {
            const int want = (2 * left + d) / (2 * d);
            r.fill = want < per ? want : per;
            skip = (skip + r.fill) % behind;
            left -= r.fill * d;
            if (r.fill == want) {
                from = (from + skip) & 255;
                behind = ALL;
                skip = 0;
            }
        }
        r.from2 = (from + skip) & 255;
        if (r.fill < per) {
            skip = (skip + per - r.fill) & 255;
            last = d;
        }
        return r;
    }
};

// a workgroup's tiles of one expert: at, while that is below the expert's number of tiles, then next()
struct Turns {
    int at, fill, behind, second;
    constexpr Turns(const Record& r, int my) : at(0), fill(r.fill), behind(r.behind), second(r.fill + ((my - r.from2) & 255))
    {
        const int place = (my - r.from) & 255, turn = place - r.skip, first = turn < 0 ? turn + r.behind : turn;
        at = place < r.behind && first < r.fill ? first : second;
    }
    constexpr void next()
    {
        if (at < fill) {
            at += behind;
            if (at >= fill) at = second;
        } else {
            at += ALL;
        }
    }
};

// The workgroups' loads as differences, add(w, d): from workgroup w on d more.

// d more for `count` workgroups from `from` on, in the circle of them
template <typename Add>
constexpr void add_arc(int from, int count, int d, Add add)
{
    if (count == 0) return;
    add(from, d);
    if (from + count < ALL) add(from + count, -d);
    if (from + count > ALL) {
        add(0, d);
        add(from + count - ALL, -d);
    }
}

// of an expert's `per` tiles of depth d
template <typename Add>
constexpr void add_by_depth(const Record& r, int d, int per, Add add)
{
    if (r.fill) {
        const int each = r.fill / r.behind, more = r.fill - each * r.behind;
        add_arc(r.from, r.behind, each * d, add);
        // places skip .. skip + more - 1, counted round the workgroups behind
        const int end = r.skip + more < r.behind ? r.skip + more : r.behind;
        add_arc((r.from + r.skip) & 255, end - r.skip, d, add);
        add_arc(r.from, r.skip + more - end, d, add);
    }
    add(0, (per - r.fill) / ALL * d);
    add_arc(r.from2, (per - r.fill) % ALL, d, add);
}

// of tiles e per .. (e + 1) per - 1, tile v to workgroup v % 256
template <typename Add>
constexpr void add_by_number(int e, int d, int per, Add add)
{
    add(0, per / ALL * d);
    add_arc((int)((unsigned)e * (unsigned)per & 255u), per % ALL, d, add);
}

// by number the last round's tile whole + i, whole rounds before it, goes to this workgroup instead of i: an eighth of them to each of 8 dies
constexpr int last_of(int i) { return (i & 7) * 32 + (i >> 3); }

}  // namespace amoe_deal
