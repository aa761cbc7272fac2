// Random sequences of solves (taken, refused before the launch, failed at it) over
// SweepVecs, on a model of the two vectors' bytes: every solve that runs must find all of
// its elements holding the sentinel of its width.
#include <cstdio>
#include <random>
#include <vector>

#include "sweep_vec.hpp"

using senk_amd::SweepVecs;

namespace {
constexpr int kMax = 24;
using Mem = std::vector<int>;  // per byte: 16 * width + place in the element, or -1
bool sentinel(const Mem &m, int i, int w) {
    for (int b = 0; b < w; b++)
        if (m[i * w + b] != 16 * w + b) return false;
    return true;
}
void put(Mem &m, int n, int w, bool value) {
    for (int i = 0; i < n; i++)
        for (int b = 0; b < w; b++) m[i * w + b] = value ? -1 : 16 * w + b;
}
}  // namespace

int main(int argc, char **) {
    std::mt19937 g(1);
    for (int trial = 0; trial < 4000; trial++) {
        SweepVecs s;
        Mem mem[2] = {Mem(8 * kMax, -1), Mem(8 * kMax, -1)};
        for (int step = 0; step < 30; step++) {
            const int n = 1 + (int)(g() % kMax), w = g() % 3 ? 8 : 4, what = (int)(g() % 6);
            if (what == 0) {                // refused: no vector is asked for
                if (argc > 1) s.solved(n, w);  // (the account of a solve that never ran)
                continue;
            }
            const int u = s.cur;
            if (s.needs_fill(n, w)) {
                put(mem[u], n, w, false);
                s.filled(n, w);
            }
            for (int i = 0; i < n; i++)
                if (!sentinel(mem[u], i, w)) {
                    std::printf("trial %d step %d: element %d of %d is not clean\n", trial, step, i, n);
                    return 1;
                }
            const bool failed = what == 1, ran = !failed || g() % 2;
            if (ran) {
                put(mem[u], n, w, true);
                put(mem[u ^ 1], n, w, false);
            }
            if (failed) s.spoiled();
            else s.solved(n, w);
        }
    }
    return 0;
}
