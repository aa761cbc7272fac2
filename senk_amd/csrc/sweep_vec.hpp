// Host-side account of the two vectors through which the single-launch solves on caller
// arrays publish their rows (trsv_csr.hip).
#pragma once

#include <algorithm>
#include <cstddef>

namespace senk_amd {

// `clean` leading elements of `width` bytes held the sentinel before its last use as the
// output, which wrote the first `dirty` of them (0: reset since).
struct SweepVec {
    void *p = nullptr;
    size_t bytes = 0, clean = 0, dirty = 0;
    int width = 0;
};

// A solve of n rows publishes in out() and resets the first n elements of next() to the
// sentinel; the two then change places.  The account changes only when a kernel that does
// this was launched (solved): a solve refused before its launch leaves it as it was.
struct SweepVecs {
    SweepVec v[2];
    int cur = 0;
    SweepVec &out() { return v[cur]; }
    SweepVec &next() { return v[cur ^ 1]; }
    // whether out() must be filled with the sentinel before a solve of n elements
    bool needs_fill(size_t n, int width) const {
        return v[cur].width != width || v[cur].dirty || v[cur].clean < n;
    }
    void filled(size_t n, int width) {
        SweepVec &u = out();
        u.width = width;
        u.clean = n;
        u.dirty = 0;
    }
    void solved(size_t n, int width) {
        out().dirty = n;
        SweepVec &o = next();  // clean beyond n where its last solve was no longer
        o.clean = o.width == width && n >= o.dirty ? std::max(o.clean, n) : n;
        o.width = width;
        o.dirty = 0;
        cur ^= 1;
    }
    // a launch failed: neither vector is known to hold the sentinel
    void spoiled() {
        for (SweepVec &u : v) u.clean = u.dirty = 0;
    }
};

}  // namespace senk_amd
