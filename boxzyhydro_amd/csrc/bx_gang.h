// bx_gang.h -- how the cells of a tube are divided among the workgroups of a
// gang (bx_batch.hip).  Integers only.
#pragma once

namespace bx {

constexpr int kSegOut = 60;  // output cells per wave row

// The range of segments and cells a workgroup takes of a tube.
struct Range {
    int nseg, s0, s1;      // segments [s0, s1) of nseg
    int c_lo, c_hi;        // cells [c_lo, c_hi) of [0, nx); the first and last ranges hold the ghosts too
    bool left, right;      // whether another member holds the segment before / after
};

// Member `member` of p of a tube of nx cells (p = 1: the whole tube).  Equal
// shares of whole segments, rounded up: with 13 segments, say, five of six
// members hold them all, so the member with the last segment need not be the
// last member, and the ones behind it have no cells.
__host__ __device__ inline Range tube_range(int nx, int member, int p)
{
    Range r;
    r.nseg = (nx - 4 + kSegOut - 1) / kSegOut;
    const int per = (r.nseg + p - 1) / p;
    r.s0 = member * per < r.nseg ? member * per : r.nseg;
    r.s1 = r.s0 + per < r.nseg ? r.s0 + per : r.nseg;
    r.left = r.s0 > 0 && r.s0 < r.s1;
    r.right = r.s1 < r.nseg;
    r.c_lo = r.s0 == 0 ? 0 : (r.s0 == r.nseg ? nx : r.s0 * kSegOut + 2);
    r.c_hi = r.s1 == r.nseg ? nx : r.s1 * kSegOut + 2;
    return r;
}

}  // namespace bx
