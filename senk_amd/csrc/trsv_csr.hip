// Single-launch triangular solves on the caller's own CSR / BCSR factors (the colored,
// planned and block entry points and the driver twins; factors held by a preconditioner
// handle use the sliced layout of trsv_sell.hip).
//
// One launch solves a whole triangle: a row's value is published in a context-owned vector
// z that starts all-sentinel (sweep.hpp), a gather waits until the row it reads is
// published, and the value also goes to the caller's y with a plain store.  The launch
// resets the context's other vector to the sentinel for the next solve, so no fill kernel
// runs.  x may alias y: only a row's own x is read, before its y is written.
//
// A launch's workgroups are numbered by ticket, 0, 1, ...: ticket 8 j + x solves part j of
// stream x, the x-th eighth of every level (in an ABMC order a band of the domain), level by
// level.  Two ways to number them:
//  - by workgroup number (a context that is alone on its device): ticket b runs on the XCD that
//    the dispatcher hands workgroup b to, b mod 8, so most gathers are served by the XCD's own
//    L2.  Progress needs every dispatcher to hand out its workgroups in increasing order and
//    no other waiting kernel beside this one: the unfinished row of the lowest level then waits
//    on nothing unfinished, and its workgroup is resident or next.
//  - drawn from the context's counter in the order of arrival (SweepWait::ticket), as soon as
//    another context lives on the device: its waiting workgroups could fill one XCD and ours
//    another, each waiting for a workgroup that finds no room where the other waits.  A drawn
//    ticket waits on lower tickets only (in a plan: see k_csr_rows), which are drawn too and
//    running or done, so a launch ends whatever runs beside it and however they arrive.  The draws
//    cost 10-15 ns each, all on one address: 64^3 grid, blocks of 8, GMRES(30) 25.8 -> 31.8
//    ms; 61x64x67 plans 557 -> 673 us; block solve of 45^3 elasticity 151 -> 161 us.
// Any other order ends in the bounded poll, which raises the context's time-out word, not in a
// hang.
//
// Per row the operations and their order are the sequential solve's: the same bits.
#include "sweep.hpp"

#include <algorithm>
#include <mutex>
#include <type_traits>

namespace senk_amd {

// Levels of a schedule in solve order (a kernel argument): first ticket, first unit (row or
// block) and unit count of each.
constexpr int kSweepMaxLevels = 256;
struct SweepLevels {
    int n;
    int ticket[kSweepMaxLevels], unit0[kSweepMaxLevels], units[kSweepMaxLevels];
};
// What a launch's waits need: the context's time-out word, the launch's number, which a wait
// that gives up writes there, and the polls after which it does.  The other waits of the
// launch then give up as well; those of later launches, whatever the word still holds, do not.
// ticket: the counter that the workgroups draw from and its value before the launch (null:
// tickets are workgroup numbers).
struct SweepWait {
    unsigned *err, tag;
    int limit;
    unsigned *ticket, base;
};

namespace {
constexpr int kCsrWaves = 4;  // waves per workgroup, each with rows (and staged entries) of its own
// How often (in polls, a power of two) a wait looks whether another wait has already given up.
constexpr int kCsrSpinCheck = 1 << 12;

// Waits until every row cc[q] (on[q]) is published in z, its bits in yb.  While a wave waits
// it polls one row only, the last one still missing of its first waiting lane (the latest
// color); when that one is there it reads all the missing ones again.  (Polling all of them,
// up to 64 x CH lines a poll from every resident wave, slows down the rows waited for:
// GMRES(30) of a 64^3 system 39.7 against 36.6 ms.)  Every other poll
// is a plain load, which the CU's own cache may answer with the sentinel, so it only thins out
// the polls at the device-coherent level: without it GMRES(30) of the 64^3 system takes 26.0
// instead of 25.6 ms, the block solve of 45^3 elasticity 153 instead of 157 us.  The limit is
// on the device-coherent ones, so that many round trips bound the wait from below.
template <typename T, int CH>
__device__ __forceinline__ void await_rows(const T *z, const int (&cc)[CH], const bool (&on)[CH],
                                           typename Bits<T>::U (&yb)[CH], SweepWait wt) {
    int want = -1;  // the last missing row of this lane
#pragma unroll
    for (int q = 0; q < CH; q++)
        if (on[q] && yb[q] == Bits<T>::kSentinel) want = cc[q];
    unsigned long long b = __ballot(want >= 0);
    for (int spin = 0; b;) {
        const T *p = z + __builtin_amdgcn_readlane(want, __ffsll((long long)b) - 1);
        while ((spin & 1 ? load_local(p) : load_agent(p)) == Bits<T>::kSentinel) {
            spin++;
            if ((spin >> 1) >= wt.limit ||
                ((spin & (kCsrSpinCheck - 1)) == 0 &&
                 __hip_atomic_load(wt.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) == wt.tag)) {
                __hip_atomic_store(wt.err, wt.tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                return;
            }
            __builtin_amdgcn_s_sleep(1);
        }
#pragma unroll
        for (int q = 0; q < CH; q++)
            if (on[q] && yb[q] == Bits<T>::kSentinel) yb[q] = load_agent(ixp<true>(z, cc[q]));
        want = -1;
#pragma unroll
        for (int q = 0; q < CH; q++)
            if (on[q] && yb[q] == Bits<T>::kSentinel) want = cc[q];
        b = __ballot(want >= 0);
    }
}

// The ticket of workgroup `number` of the `n` that solve; -1: the counter is out of step with
// the host's count (the launch then reports a time-out).
__device__ __forceinline__ int draw_ticket(const SweepWait &wt, int number, int n) {
    if (!wt.ticket) return number;
    __shared__ int tk;
    if (threadIdx.x == 0) {
        const unsigned t =
            __hip_atomic_fetch_add(wt.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - wt.base;
        tk = t < (unsigned)n ? (int)t : -1;
        if (tk < 0) __hip_atomic_store(wt.err, wt.tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(tk);
}

// Level of ticket j (uniform): the last l with ticket[l] <= j.
__device__ __forceinline__ int level_of(const SweepLevels &lv, int j) {
    int lo = 0, hi = lv.n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (lv.ticket[mid] <= j) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}
// The wave's slice (of `per` units) of its stream's band of level l, or -1.
__device__ __forceinline__ int band_slice(const SweepLevels &lv, int l, int j, int xs, int per) {
    const int ns = (lv.units[l] + per - 1) / per;
    const int lo = (int)((long long)ns * xs / kXcds), end = (int)((long long)ns * (xs + 1) / kXcds);
    const int sl = lo + (j - lv.ticket[l]) * kCsrWaves + (int)(threadIdx.x >> 6);
    return sl < end ? sl : -1;
}

// ------------------------------------------------------------------ CSR, colored
// One lane per row, the BS rows of a block in consecutive lanes (BS | 64).  The wave copies
// its rows' slice of the factor into LDS with coalesced loads (a slice of more than
// kCsrCap entries is read in place), then per row: the entries outside the block in rounds
// of 8 gathers, then BS steps inside the block, each finished row broadcast in the wave.
// Bound by the levels' dependent chain (publish, poll, in-block steps), not by bytes.
template <typename T>
constexpr int kCsrCap = 10 * 1024 / (int)(sizeof(T) + sizeof(int));

template <typename T, int BS, bool UPPER, typename FC, typename FV>
__device__ __forceinline__ T solve_row(T t, int s, int e, bool active, int base, const T *z, SweepWait wt, FC C,
                                       FV V) {
    using U = typename Bits<T>::U;
    constexpr int CH = 8;
    const int r = (int)(threadIdx.x & 63) % BS;
    T dinv = 0;
    if (UPPER && active) dinv = V(s);
    int k = UPPER ? e - 1 : s;
    bool go = active;
    while (__ballot(go)) {
        int cc[CH];
        bool on[CH];
        T vv[CH];
        U yb[CH];
        int cnt = 0;
#pragma unroll
        for (int q = 0; q < CH; q++) {
            const int i = UPPER ? k - q : k + q;
            const bool in = go && (UPPER ? i > s : i < e);
            cc[q] = in ? C(i) : 0;
            on[q] = in && (UPPER ? cc[q] >= base + BS : cc[q] < base) && (q == 0 || on[q > 0 ? q - 1 : 0]);
            if (on[q]) {
                vv[q] = V(i);
                cnt++;
            }
        }
#pragma unroll
        for (int q = 0; q < CH; q++)
            if (on[q]) yb[q] = load_local(ixp<true>(z, cc[q]));
        await_rows<T, CH>(z, cc, on, yb, wt);
#pragma unroll
        for (int q = 0; q < CH; q++)
            if (on[q]) t -= vv[q] * __builtin_bit_cast(T, yb[q]);
        k += UPPER ? -cnt : cnt;
        go = on[CH - 1];
    }
    if constexpr (BS == 1) {
        if (UPPER) t = t * dinv;
    } else if constexpr (BS <= 16) {
        // mask of the in-block columns (ascending for L, descending for U); the entry of
        // column c is then found by counting, so every value is read before the steps
        unsigned mk = 0;
        bool more = active;
        int prev = UPPER ? BS : -1;
#pragma unroll
        for (int q = 0; q < BS; q++) {
            const int i = UPPER ? k - q : k + q;
            const int c = more && (UPPER ? i > s : i < e) ? C(i) - base : (UPPER ? BS : -1);
            more = more && (UPPER ? (c < prev && c >= 0) : (c > prev && c < BS));
            if (more) mk |= 1u << c;
            prev = c;
        }
        T iv[BS];
#pragma unroll
        for (int c = 0; c < BS; c++) {
            const unsigned before = UPPER ? mk >> (c + 1) : mk & ((1u << c) - 1);
            const int p = __popc(before);
            iv[c] = (mk >> c) & 1 ? V(UPPER ? k - p : k + p) : T(0);
        }
#pragma unroll
        for (int i = 0; i < BS; i++) {
            const int c = UPPER ? BS - 1 - i : i;
            if (UPPER && r == c) t = t * dinv;
            const T yc = block_bcast<BS>(t, c);
            if ((mk >> c) & 1) t -= iv[c] * yc;
        }
    } else {
        // the next in-block entry, loaded one ahead of the step that takes it
        const int lim = UPPER ? s : e;
        auto has = [&](int i) { return active && (UPPER ? i > lim : i < lim); };
        int nc = has(k) ? C(k) : -1;
        T nv = has(k) ? V(k) : T(0);
#pragma unroll
        for (int i = 0; i < BS; i++) {
            const int c = UPPER ? BS - 1 - i : i;
            if (UPPER && r == c) t = t * dinv;
            const T yc = block_bcast<BS>(t, c);
            if (nc == base + c) {
                t -= nv * yc;
                k += UPPER ? -1 : 1;
                nc = has(k) ? C(k) : -1;
                nv = has(k) ? V(k) : T(0);
            }
        }
    }
    return t;
}

template <typename T, int BS, bool UPPER>
__global__ __launch_bounds__(64 * kCsrWaves) void k_csr_sweep(SweepLevels lv, const int *__restrict__ rptr,
                                                              const int *__restrict__ cind,
                                                              const T *__restrict__ val, const T *x, T *y, T *z,
                                                              T *reset, const double *__restrict__ in_scale,
                                                              SweepWait wt, const int *__restrict__ stop) {
    __shared__ T sv[kCsrWaves][kCsrCap<T>];
    __shared__ int sc[kCsrWaves][kCsrCap<T>];
    const int tk = draw_ticket(wt, (int)blockIdx.x, (int)gridDim.x);
    if (tk < 0) return;
    const int xs = tk % kXcds, j = tk / kXcds;
    const int l = level_of(lv, j), sl = __builtin_amdgcn_readfirstlane(band_slice(lv, l, j, xs, 64));
    if (sl < 0) return;
    const int wv = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63);
    const int r0 = lv.unit0[l] + sl * 64, nr = min(64, lv.units[l] - sl * 64);
    const int row = r0 + lane;
    const bool active = lane < nr;
    const int stopped = stop ? *stop : 0;
    int s = 0, e = 0;
    T t = 0;
    if (active) {
        s = rptr[row];
        e = rptr[row + 1];
        t = x[row];
        reset[row] = __builtin_bit_cast(T, Bits<T>::kSentinel);
    }
    if (stopped) return;
    if (!UPPER && in_scale && active) t = (T)((double)t * *in_scale);
    const int e0 = __builtin_amdgcn_readlane(s, 0), e1 = __builtin_amdgcn_readlane(e, nr - 1);
    const int base = row - lane % BS;
    if (e1 - e0 <= kCsrCap<T>) {
        const int n = e1 - e0;
        for (int q0 = lane; q0 < n; q0 += 64 * 4) {
            T v[4];
            int c[4];
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (q0 + 64 * u < n) {
                    v[u] = val[e0 + q0 + 64 * u];
                    c[u] = cind[e0 + q0 + 64 * u];
                }
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (q0 + 64 * u < n) {
                    sv[wv][q0 + 64 * u] = v[u];
                    sc[wv][q0 + 64 * u] = c[u];
                }
        }
        wave_lds_sync();
        t = solve_row<T, BS, UPPER>(t, s - e0, e - e0, active, base, z, wt, [&](int i) { return sc[wv][i]; },
                                    [&](int i) { return sv[wv][i]; });
    } else {
        t = solve_row<T, BS, UPPER>(t, s, e, active, base, z, wt, [&](int i) { return cind[i]; },
                                    [&](int i) { return val[i]; });
    }
    if (active) {
        store_agent(z + row, canonical(t));
        y[row] = t;
    }
}

// ------------------------------------------------------------------ CSR, planned (level lists)
// Rows of a level schedule (bsize 1): ticket t takes the rows seq[64 t + lane] (-1: none).
// Rows of several levels may share a wave, so no lane waits for another: every lane polls for
// its own entries, and a lane whose round is complete subtracts it and goes on or publishes its
// row, whatever the others wait for.  A wave's rows are 64 consecutive ones of one stream, and a
// ticket's begin at most one wave of its stream past the level in which a higher ticket's begin.
// So of the waves that have drawn a ticket, at most two a stream cannot finish before one that
// has not drawn: they fill no XCD, and the next workgroup finds room.
// Rows are published by their place in seq (pos), not by row: the rows that a level's
// consecutive rows wait for are then close together, and a poll touches a few lines instead
// of one per entry (published by row, every resident wave's polls kept the memory system
// busy: 61x64x67 7-point grid, 190 levels, L + U in FP64 1352 us, 581 by place; one launch
// per level 1748).  Every poll is at the device-coherent level: a plain load may be answered
// with the sentinel by the CU's own cache (every other poll plain 581 us, none 551; 27-point
// 38^3 1332 and 1249).  What is left is one publish-and-poll round trip per level, about 1.45 us.
template <typename T, bool UPPER, int CH>
__global__ __launch_bounds__(64) void k_csr_rows(int waves, int xcds, const int *__restrict__ seq,
                                                 const int *__restrict__ pos,
                                                 const int *__restrict__ rptr, const int *__restrict__ cind,
                                                 const T *__restrict__ val, const T *x, T *y, T *z, T *reset,
                                                 const double *__restrict__ in_scale, SweepWait wt,
                                                 const int *__restrict__ stop) {
    using U = typename Bits<T>::U;
    const int xcd = (int)(blockIdx.x % kXcds), number = (int)(blockIdx.x / kXcds) * xcds + xcd;
    if (xcd >= xcds) return;
    const int tk = draw_ticket(wt, number, waves);
    if (tk < 0) return;
    const int mine = tk * 64 + (int)(threadIdx.x & 63);
    const int row = seq[mine];
    const int stopped = stop ? *stop : 0;
    bool act = row >= 0;
    int s = 0, e = 0, k = 0;
    T t = 0, dinv = 0;
    if (act) {
        s = rptr[row];
        e = rptr[row + 1];
        t = x[row];
    }
    reset[mine] = __builtin_bit_cast(T, Bits<T>::kSentinel);
    if (stopped) return;
    if (act) {
        if (UPPER) dinv = val[s];
        else if (in_scale) t = (T)((double)t * *in_scale);
        k = UPPER ? e - 1 : s;
    }
    int cc[CH];
    bool on[CH];
    T vv[CH];
    U yb[CH];
    auto round = [&]() {
#pragma unroll
        for (int q = 0; q < CH; q++) {
            const int i = UPPER ? k - q : k + q;
            const bool in = act && (UPPER ? i > s : i < e);
            cc[q] = in ? cind[i] : 0;
            vv[q] = in ? val[i] : T(0);
            on[q] = in && (UPPER ? cc[q] > row : cc[q] < row) && (q == 0 || on[q > 0 ? q - 1 : 0]);
        }
#pragma unroll
        for (int q = 0; q < CH; q++) cc[q] = on[q] ? pos[cc[q]] : 0;
#pragma unroll
        for (int q = 0; q < CH; q++) yb[q] = on[q] ? load_local(z + cc[q]) : U(0);
    };
    round();
    for (int spin = 0; __ballot(act); spin++) {
        bool pend = false;
#pragma unroll
        for (int q = 0; q < CH; q++) pend |= on[q] && yb[q] == Bits<T>::kSentinel;
        if (__ballot(act && !pend)) {
            spin = 0;
            if (act && !pend) {
                int cnt = 0;
#pragma unroll
                for (int q = 0; q < CH; q++)
                    if (on[q]) {
                        t -= vv[q] * __builtin_bit_cast(T, yb[q]);
                        cnt++;
                    }
                k += UPPER ? -cnt : cnt;
                if (on[CH - 1]) {
                    round();
                } else {
                    if (UPPER) t = t * dinv;
                    store_agent(z + mine, canonical(t));
                    y[row] = t;
                    act = false;
                }
            }
            continue;
        }
        if (spin >= wt.limit ||
            ((spin & (kCsrSpinCheck - 1)) == kCsrSpinCheck - 1 &&
             __hip_atomic_load(wt.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) == wt.tag)) {
            // give up: publish a NaN so that the rows behind this one end too
            if (act) {
                __hip_atomic_store(wt.err, wt.tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                t = __builtin_nan("");
                store_agent(z + mine, canonical(t));
                y[row] = t;
            }
            return;
        }
        __builtin_amdgcn_s_sleep(1);
#pragma unroll
        for (int q = 0; q < CH; q++)
            if (act && on[q] && yb[q] == Bits<T>::kSentinel)
                yb[q] = load_agent(z + cc[q]);
    }
}

// ------------------------------------------------------------------ BCSR, colored
// One lane per row.  A wave takes bpw whole schedule blocks of bsize rows (bsize <= 64), or one
// larger block in parts of at most 64 rows one after the other (a later part gathers the
// earlier ones like any other row).  Per row, in the order of the sequential solve
// (senk_sparse.hpp:399-415, 436-464): first the entries of BNL x BNW blocks outside the
// part, in rounds of about 8 gathers, then the in-part columns step by step, each finished row
// broadcast in the wave; the lane's next in-part blocks wait in LDS, requested before the
// first wait, one block read ahead of its step (in registers instead of LDS the queue spills:
// 181-604 us).  Bound by the levels' chain (publish, poll, in-part steps).  Elasticity 45^3,
// blocks of 48, 11 colors, L + U in FP64: 150 us; one lane per schedule block walking its rows,
// one launch per color (518 lanes in flight), 3187 us.
template <typename T, int BNL, int BNW, bool UPPER>
__global__ __launch_bounds__(64 * kCsrWaves) void k_bcsr_sweep(
    SweepLevels lv, const int *__restrict__ blk_list, int bsize, int part, int bpw, const int *__restrict__ brptr,
    const int *__restrict__ bcind, const T *__restrict__ bval, const T *x, T *y, T *z, T *reset, SweepWait wt) {
    using U = typename Bits<T>::U;
    constexpr int BS = BNL * BNW, BREM = BNL / BNW;
    constexpr int CB = BNW >= 8 ? 1 : (8 + BNW - 1) / BNW;  // blocks per round
    constexpr int QB = BNW == 1 ? 8 : 4;                    // in-part blocks held in LDS
    __shared__ int qc[kCsrWaves][QB][64];
    __shared__ T qv[kCsrWaves][QB][BNW][64];
    const int tk = draw_ticket(wt, (int)blockIdx.x, (int)gridDim.x);
    if (tk < 0) return;
    const int xs = tk % kXcds, j = tk / kXcds;
    const int l = level_of(lv, j), sl = __builtin_amdgcn_readfirstlane(band_slice(lv, l, j, xs, bpw));
    if (sl < 0) return;
    const int lane = (int)(threadIdx.x & 63), wv = (int)(threadIdx.x >> 6);
    const int nb = min(bpw, lv.units[l] - sl * bpw);  // blocks of this wave
    const int slot = bpw > 1 ? lane / bsize : 0;
    const bool has = slot < nb;
    const int bu = lv.unit0[l] + sl * bpw + (has ? slot : 0);
    const int blk = blk_list ? blk_list[bu] : bu;
    const int nparts = (bsize + part - 1) / part;
    for (int pq = 0; pq < nparts; pq++) {
        const int p = UPPER ? nparts - 1 - pq : pq;
        const int rows = min(part, bsize - p * part);
        const int r = lane - slot * bsize;  // row in the part (bpw > 1: a whole block)
        const bool active = has && r < rows;
        const int base = blk * bsize + p * part, end = base + rows;
        const int row = base + (active ? r : 0), g = row / BNL, kk = row % BNL;
        const int lbase = slot * bsize;  // lane of the part's first row
        T t = 0;
        int first = 0, cnt = 0;          // the row's blocks outside its own diagonal (U), in solve order
        T dg[BNL] = {};
        if (active) {
            t = x[row];
            reset[row] = __builtin_bit_cast(T, Bits<T>::kSentinel);
            const int b0 = brptr[g], b1 = brptr[g + 1];
            if (UPPER) {
                first = b1 - 1;
                cnt = b1 - (b0 + BREM);
#pragma unroll
                for (int d = 0; d < BNL; d++)
                    dg[d] = d >= kk ? bval[(size_t)(b0 + d / BNW) * BS + (d % BNW) * BNL + kk] : T(0);
            } else {
                first = b0;
                cnt = b1 - b0;
            }
        }
        auto at = [&](int i) { return UPPER ? first - i : first + i; };
        // the place of the first in-part block, and whether the columns run strictly in solve order
        int in0 = cnt, prev = UPPER ? 0x7fffffff : -1;
        bool ordered = true;
        for (int i0 = 0; __ballot(i0 < cnt); i0 += 8) {
            int c[8];
#pragma unroll
            for (int q = 0; q < 8; q++)
                if (i0 + q < cnt) c[q] = bcind[at(i0 + q)] * BNW;
#pragma unroll
            for (int q = 0; q < 8; q++)
                if (i0 + q < cnt) {
                    ordered = ordered && (UPPER ? c[q] < prev : c[q] > prev);
                    prev = c[q];
                    if (UPPER ? c[q] < end : c[q] >= base) in0 = min(in0, i0 + q);
                }
        }
        const bool slow = __ballot(!ordered) != 0;
        const int outside = slow ? cnt : in0;  // blocks to look at for rows outside the part
        // in-part columns: the lane's next QB blocks wait in LDS, requested before the wait below;
        // the block after the current one is read ahead of its step
        auto refill = [&](int i0) {
            int c[QB];
            T v[QB][BNW];
#pragma unroll
            for (int q = 0; q < QB; q++) {
                c[q] = -1;
                if (i0 + q < cnt) {
                    const int b = at(i0 + q);
                    c[q] = bcind[b] * BNW - base;
                    const T *vb = bval + (size_t)b * BS + kk;
#pragma unroll
                    for (int m = 0; m < BNW; m++) v[q][m] = vb[m * BNL];
                }
            }
#pragma unroll
            for (int q = 0; q < QB; q++) {
                qc[wv][q][lane] = c[q];
#pragma unroll
                for (int m = 0; m < BNW; m++)
                    if (i0 + q < cnt) qv[wv][q][m][lane] = v[q][m];
            }
        };
        refill(in0);
        // outside the part
        for (int i0 = 0; __ballot(i0 < outside); i0 += CB) {
            int cc[CB * BNW];
            bool on[CB * BNW];
            T vv[CB * BNW];
            U yb[CB * BNW];
#pragma unroll
            for (int q = 0; q < CB; q++) {
                const bool have = i0 + q < outside;
                const int c = have ? bcind[at(i0 + q)] * BNW : 0;
                const bool out = have && (UPPER ? c >= end : c < base);
#pragma unroll
                for (int m = 0; m < BNW; m++) {
                    cc[q * BNW + m] = c + m;
                    on[q * BNW + m] = out;
                    if (out) vv[q * BNW + m] = (bval + (size_t)at(i0 + q) * BS + kk)[m * BNL];
                }
            }
#pragma unroll
            for (int q = 0; q < CB * BNW; q++)
                if (on[q]) yb[q] = load_local(ixp<true>(z, cc[q]));
            await_rows<T, CB * BNW>(z, cc, on, yb, wt);
#pragma unroll
            for (int q = 0; q < CB * BNW; q++)
                if (on[q]) t -= vv[q] * __builtin_bit_cast(T, yb[q]);
        }
        auto bcast = [&](int i) {  // row i of every block's part
            if (bpw == 1) {
                if constexpr (sizeof(T) == 4) {
                    return __builtin_bit_cast(T, __builtin_amdgcn_readlane(__builtin_bit_cast(int, t), i));
                } else {
                    const unsigned long long u = __builtin_bit_cast(unsigned long long, t);
                    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, i);
                    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), i);
                    return __builtin_bit_cast(T, ((unsigned long long)hi << 32) | lo);
                }
            }
            return __shfl(t, (lbase + i) & 63, 64);
        };
        int nq = 0, nc = -1;
        T nv[BNW];
        auto next = [&]() {
            nc = qc[wv][nq][lane];
#pragma unroll
            for (int m = 0; m < BNW; m++) nv[m] = qv[wv][nq][m][lane];
        };
        next();
        // The rows that hold the column block at c0 subtract it; value(m): column c0 + m.  A
        // block of L may lie in its rows' own group, where column m is final only once the
        // columns before it are subtracted: value(m) is asked for in that order.
        auto take = [&](int c0, auto &&value) {
            if (slow) {  // columns not in order: every block of the row is looked at
                for (int m = 0; m < BNW; m++) {
                    const T yc = value(m);
                    for (int i = 0; i < cnt; i++) {
                        const int b = at(i);
                        if (bcind[b] * BNW - base == c0) t -= bval[(size_t)b * BS + m * BNL + kk] * yc;
                    }
                }
                return;
            }
            const bool mine = nc == c0;
            if (!__ballot(mine)) return;
#pragma unroll
            for (int m = 0; m < BNW; m++) {
                const T yc = value(m);
                if (mine) t -= nv[m] * yc;
            }
            if (mine) {
                if (++nq == QB) {
                    in0 += QB;
                    refill(in0);
                    nq = 0;
                }
                next();
            }
        };
        if (!UPPER) {
            for (int c0 = 0; c0 < rows; c0 += BNW) take(c0, [&](int m) { return bcast(c0 + m); });
        } else {
            for (int g0 = rows - BNL; g0 >= 0; g0 -= BNL) {
                // the group's own triangle, its diagonal inverted
                T yd[BNL];
#pragma unroll
                for (int d = BNL - 1; d >= 0; d--) {
                    if (r == g0 + d) t = t * dg[d];
                    yd[d] = bcast(g0 + d);
                    if (r >= g0 && r < g0 + d) t -= dg[d] * yd[d];
                }
#pragma unroll
                for (int q = BREM - 1; q >= 0; q--)
                    take(g0 + q * BNW, [&](int m) {
                        T v = yd[q * BNW];
#pragma unroll
                        for (int w = 1; w < BNW; w++) v = m == w ? yd[q * BNW + w] : v;
                        return v;
                    });
            }
        }
        if (active) {
            store_agent(z + row, canonical(t));
            y[row] = t;
        }
    }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_fill_sentinel2(size_t n, T *p) {
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock)
        p[i] = __builtin_bit_cast(T, Bits<T>::kSentinel);
}
}  // namespace

// ------------------------------------------------------------------ host side
// The sweep vectors of the next solve of n rows: *z all-sentinel (filled here where the
// last solves left less than that), *reset the vector the launch must fill in its first n
// rows; SweepLaunch::done follows the launch.  false: no memory (the caller takes its
// launch-per-level path).
template <typename T>
static int sweep_vectors(Ctx *c, size_t n, T **z, T **reset, bool *ok) {
    SweepVec *v = c->sweep.v;
    *ok = false;
    const size_t bytes = n * sizeof(T);
    if (!c->sweep_err || bytes >= (size_t)1 << 32) return SENK_OK;  // z is addressed by 32-bit offsets
    if (v[0].bytes < bytes) {
        // grown while nothing of this context runs on it; allowed during a stream capture
        // of the calling thread (the context's stream is never captured)
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        SENK_HIP(hipThreadExchangeStreamCaptureMode(&mode));
        int st = hipStreamSynchronize(c->stream) == hipSuccess ? SENK_OK : SENK_ERR_HIP;
        bool got = st == SENK_OK;
        for (int i = 0; i < 2 && got; i++) {
            if (v[i].p) (void)hipFree(v[i].p);
            v[i] = SweepVec{};
            got = hipMalloc(&v[i].p, bytes) == hipSuccess;
            if (!got) v[i].p = nullptr;
        }
        if (!got) {
            (void)hipGetLastError();
            for (int i = 0; i < 2; i++) {
                if (v[i].p) (void)hipFree(v[i].p);
                v[i] = SweepVec{};
            }
        } else {
            v[0].bytes = v[1].bytes = bytes;
        }
        SENK_HIP(hipThreadExchangeStreamCaptureMode(&mode));
        if (st) return st;
        if (!got) return SENK_OK;
    }
    SweepVec &u = c->sweep.out();
    if (c->sweep.needs_fill(n, (int)sizeof(T))) {
        k_fill_sentinel2<T><<<(int)std::min<size_t>((n + kBlock - 1) / kBlock, 2048), kBlock, 0, c->stream>>>(
            n, (T *)u.p);
        SENK_LAUNCH_CHECK();
        c->sweep.filled(n, (int)sizeof(T));
    }
    *z = (T *)u.p;
    *reset = (T *)c->sweep.next().p;
    *ok = true;
    return SENK_OK;
}
// Held while a sweep is launched: which way its tickets are numbered depends on the contexts
// that live on the device, and senk_ctx_create waits, once its own is counted, for what was
// launched under the former count.
struct SweepLaunch {
    Ctx *c;
    std::lock_guard<std::mutex> held;
    SweepWait wt;
    explicit SweepLaunch(Ctx *ctx) : c(ctx), held(device_contexts(ctx->device).m) {
        if (++c->sweep_tag == 0) c->sweep_tag = 1;  // 0: nothing gave up
        const bool draw = c->sweep_tickets < 0 ? device_contexts(c->device).n > 1 : c->sweep_tickets != 0;
        wt = SweepWait{c->sweep_err_d, c->sweep_tag, c->sweep_polls, draw ? c->sweep_ticket : nullptr, c->sweep_base};
    }
    // The status of the launch, which took the vectors of sweep_vectors<T>(n) and whose `tickets`
    // workgroups solve.
    template <typename T>
    int done(size_t n, int tickets) {
        const hipError_t e = hipGetLastError();
        if (e == hipSuccess) {
            c->sweep.solved(n, (int)sizeof(T));
            if (wt.ticket) c->sweep_base += (unsigned)tickets;
            return SENK_OK;
        }
        c->sweep.spoiled();
        (void)hipMemsetAsync(c->sweep_ticket, 0, sizeof(unsigned), c->stream);
        c->sweep_base = 0;
        SENK_HIP(e);
        return SENK_OK;
    }
};

// Average rows per level below which a plan's rows go through one stream, i.e. one XCD: a
// thin level has no use for the others' bandwidth, and its waits stay on one die.  L + U in
// FP64, one / eight streams: 7-point 12^3 (51 rows a level) 73 / 96 us, 24^3 (197) 160 /
// 194, 40^3 (542) 309 / 334, 48^3 (776) 404 / 405, 61x64x67 (1377) 663 / 551; 27-point 38^3
// (209) 1263 / 1352.
constexpr double kPlanOneStream = 800;
void sweep_sequence(const Schedule &s, const std::vector<int> &blk, bool upper, int *streams, int *waves,
                    std::vector<int> &out) {
    const size_t n = blk.size();
    const int S = s.nlev > 0 && (double)n / s.nlev < kPlanOneStream ? 1 : kXcds;
    // the rows of every stream, level by level, and the level of every wave's first row
    std::vector<int> row[kXcds], first[kXcds];
    for (int step = 0; step < s.nlev; step++) {
        const int l = upper ? s.nlev - 1 - step : step;
        const long long a = s.lev_ptr[l], k = s.lev_ptr[l + 1] - a;
        for (int x = 0; x < S; x++)
            for (long long i = a + k * x / S; i < a + k * (x + 1) / S; i++) {
                if (row[x].size() % 64 == 0) first[x].push_back(step);
                row[x].push_back(blk[i]);
            }
    }
    // Rounds of one wave a stream.  A stream whose next wave begins in a later level than another
    // stream's passes (an empty wave), unless its last one does not: it is at most one ahead.
    std::vector<int> order[kXcds];  // wave of the stream per round, or -1
    size_t at[kXcds] = {};
    for (;;) {
        int low = s.nlev;
        for (int x = 0; x < S; x++)
            if (at[x] < first[x].size()) low = std::min(low, first[x][at[x]]);
        if (low == s.nlev) break;
        for (int x = 0; x < S; x++) {
            const size_t i = at[x];
            const bool take = i < first[x].size() && (first[x][i] <= low || i == 0 || first[x][i - 1] <= low);
            order[x].push_back(take ? (int)i : -1);
            at[x] += take;
        }
    }
    const size_t w = order[0].size() * S;
    *streams = S;
    *waves = (int)w;
    // blk, then the sequence, then each row's place in it
    out.assign(n + w * 64 + n, -1);
    std::copy(blk.begin(), blk.end(), out.begin());
    int *seq = out.data() + n, *pos = seq + w * 64;
    for (size_t t = 0; t < w; t++) {
        const std::vector<int> &r = row[t % S];
        const int k = order[t % S][t / S];
        if (k < 0) continue;
        for (size_t i = (size_t)k * 64; i < std::min(r.size(), (size_t)k * 64 + 64); i++) {
            const size_t p = t * 64 + i % 64;
            seq[p] = r[i];
            pos[r[i]] = (int)p;
        }
    }
}

// The level table of a schedule in solve order; units of a level: rows or blocks, `per` of
// them in a wave's slice.
static bool sweep_levels(const Schedule &s, bool upper, int scale, int per, SweepLevels *lv, int *tickets) {
    lv->n = 0;
    int tk = 0;
    for (int step = 0; step < s.nlev; step++) {
        const int l = upper ? s.nlev - 1 - step : step;
        const int nb = s.lev_ptr[l + 1] - s.lev_ptr[l];
        if (nb < 0) return false;
        if (nb == 0) continue;
        if (lv->n >= kSweepMaxLevels) return false;
        lv->ticket[lv->n] = tk;
        lv->unit0[lv->n] = s.lev_ptr[l] * scale;
        lv->units[lv->n] = nb * scale;
        lv->n++;
        const int ns = (nb * scale + per - 1) / per;
        int most = 0;
        for (int x = 0; x < kXcds; x++)
            most = std::max(most, (int)((long long)ns * (x + 1) / kXcds - (long long)ns * x / kXcds));
        tk += (most + kCsrWaves - 1) / kCsrWaves;
    }
    *tickets = tk;
    return lv->n > 0;
}

template <typename T>
int launch_csr_sweep(Ctx *c, const Schedule &s, bool upper, int N, const int *rptr, const int *cind, const T *val,
                     const T *x, T *y, const double *in_scale, const int *stop, bool *done) {
    *done = false;
    const int BS = s.bsize;
    if (N <= 0 || BS < 1 || BS > 64 || 64 % BS || s.lev_ptr.empty() || s.lev_ptr[0] != 0 ||
        (long long)s.lev_ptr[s.nlev] * BS != N)
        return SENK_OK;
    T *z = nullptr, *reset = nullptr;
    if (s.dblk) {
        if (BS != 1 || !s.dseq || !s.dpos || s.seq_upper != upper) return SENK_OK;
        const size_t nz = (size_t)s.seq_waves * 64;
        bool ok = false;
        SENK_TRY(sweep_vectors<T>(c, nz, &z, &reset, &ok));
        if (!ok) return SENK_OK;
        const int grid = s.seq_waves / s.streams * kXcds;
        SweepLaunch sl(c);
        // rounds of 4 where no row has more entries, else of 16: a second round costs its own
        // chain of dependent loads after the last row of the first is there
#define SENK_CSR_ROWS(UP, CH)                                                                                     \
    k_csr_rows<T, UP, CH><<<grid, 64, 0, c->stream>>>(s.seq_waves, s.streams, s.dseq, s.dpos, rptr, cind, val, x, \
                                                      y, z, reset, UP ? nullptr : in_scale, sl.wt, stop)
        if (upper && s.max_ext <= 4) SENK_CSR_ROWS(true, 4);
        else if (upper) SENK_CSR_ROWS(true, 16);
        else if (s.max_ext <= 4) SENK_CSR_ROWS(false, 4);
        else SENK_CSR_ROWS(false, 16);
#undef SENK_CSR_ROWS
        SENK_TRY(sl.done<T>(nz, s.seq_waves));
        *done = true;
        return SENK_OK;
    }
    SweepLevels lv;
    int tickets = 0;
    if (!sweep_levels(s, upper, BS, 64, &lv, &tickets)) return SENK_OK;
    bool ok = false;
    SENK_TRY(sweep_vectors<T>(c, (size_t)N, &z, &reset, &ok));
    if (!ok) return SENK_OK;
    const int grid = kXcds * tickets;
    SweepLaunch sl(c);
#define SENK_CSR_SWEEP(B)                                                                                        \
    case B:                                                                                                      \
        if (upper)                                                                                               \
            k_csr_sweep<T, B, true><<<grid, 64 * kCsrWaves, 0, c->stream>>>(lv, rptr, cind, val, x, y, z, reset, \
                                                                            nullptr, sl.wt, stop);              \
        else                                                                                                     \
            k_csr_sweep<T, B, false><<<grid, 64 * kCsrWaves, 0, c->stream>>>(lv, rptr, cind, val, x, y, z,       \
                                                                             reset, in_scale, sl.wt,             \
                                                                             stop);                              \
        break;
    switch (BS) {
        SENK_CSR_SWEEP(1)
        SENK_CSR_SWEEP(2)
        SENK_CSR_SWEEP(4)
        SENK_CSR_SWEEP(8)
        SENK_CSR_SWEEP(16)
        SENK_CSR_SWEEP(32)
        SENK_CSR_SWEEP(64)
        default: return SENK_ERR_UNSUPPORTED;  // not reached: BS divides 64
    }
#undef SENK_CSR_SWEEP
    SENK_TRY(sl.done<T>((size_t)N, kXcds * tickets));
    *done = true;
    return SENK_OK;
}
template int launch_csr_sweep<double>(Ctx *, const Schedule &, bool, int, const int *, const int *, const double *,
                                      const double *, double *, const double *, const int *, bool *);
template int launch_csr_sweep<float>(Ctx *, const Schedule &, bool, int, const int *, const int *, const float *,
                                     const float *, float *, const double *, const int *, bool *);

template <typename T, int BNL, int BNW>
static void bcsr_sweep(Ctx *c, const SweepWait &wt, const SweepLevels &lv, int tickets, const Schedule &s,
                       bool upper, int part, int bpw, const int *brptr, const int *bcind, const T *bval, const T *x,
                       T *y, T *z, T *reset) {
    const int grid = kXcds * tickets;
    if (upper)
        k_bcsr_sweep<T, BNL, BNW, true><<<grid, 64 * kCsrWaves, 0, c->stream>>>(
            lv, s.dblk, s.bsize, part, bpw, brptr, bcind, bval, x, y, z, reset, wt);
    else
        k_bcsr_sweep<T, BNL, BNW, false><<<grid, 64 * kCsrWaves, 0, c->stream>>>(
            lv, s.dblk, s.bsize, part, bpw, brptr, bcind, bval, x, y, z, reset, wt);
}
template <typename T>
int launch_bcsr_sweep(Ctx *c, const Schedule &s, bool upper, int N, int bnl, int bnw, const int *brptr,
                      const int *bcind, const T *bval, const T *x, T *y, bool *done) {
    *done = false;
    if (bnl < 1 || bnw < 1 || bnl % bnw || s.bsize % bnl || s.lev_ptr.empty() || s.lev_ptr[0] != 0 ||
        (long long)s.lev_ptr[s.nlev] * s.bsize != N)
        return SENK_OK;
    const int part = s.bsize <= 64 ? s.bsize : 64 / bnl * bnl;
    const int bpw = s.bsize <= 64 ? 64 / s.bsize : 1;
    SweepLevels lv;
    int tickets = 0;
    if (!sweep_levels(s, upper, 1, bpw, &lv, &tickets)) return SENK_OK;
    decltype(&bcsr_sweep<T, 1, 1>) launch = nullptr;
#define SENK_BCSR_SWEEP(A, B) \
    case 16 * A + B: launch = bcsr_sweep<T, A, B>; break
    switch (16 * bnl + bnw) {
        SENK_BCSR_SWEEP(1, 1);
        SENK_BCSR_SWEEP(2, 1);
        SENK_BCSR_SWEEP(2, 2);
        SENK_BCSR_SWEEP(3, 1);
        SENK_BCSR_SWEEP(3, 3);
        SENK_BCSR_SWEEP(4, 1);
        SENK_BCSR_SWEEP(4, 2);
        SENK_BCSR_SWEEP(4, 4);
        SENK_BCSR_SWEEP(8, 1);
        SENK_BCSR_SWEEP(8, 2);
        SENK_BCSR_SWEEP(8, 4);
        SENK_BCSR_SWEEP(8, 8);
        default: return SENK_ERR_UNSUPPORTED;  // as the launch per level
    }
#undef SENK_BCSR_SWEEP
    T *z = nullptr, *reset = nullptr;
    bool ok = false;
    SENK_TRY(sweep_vectors<T>(c, (size_t)N, &z, &reset, &ok));
    if (!ok) return SENK_OK;
    SweepLaunch sl(c);
    launch(c, sl.wt, lv, tickets, s, upper, part, bpw, brptr, bcind, bval, x, y, z, reset);
    SENK_TRY(sl.done<T>((size_t)N, kXcds * tickets));
    *done = true;
    return SENK_OK;
}
template int launch_bcsr_sweep<double>(Ctx *, const Schedule &, bool, int, int, int, const int *, const int *,
                                       const double *, const double *, double *, bool *);
template int launch_bcsr_sweep<float>(Ctx *, const Schedule &, bool, int, int, int, const int *, const int *,
                                      const float *, const float *, float *, bool *);

}  // namespace senk_amd
