// Device helpers of the single-launch triangular sweeps: in-wave row broadcasts, and the
// sentinel protocol by which one row waits for another.
#pragma once

#include "dev_common.hpp"

#include <type_traits>

namespace senk_amd {

// number of set bits of b in the lanes below this one
__device__ __forceinline__ int lanes_below(unsigned long long b) {
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(b >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)b, 0u));
}

// Row c of every block of BS consecutive lanes, broadcast to the block's lanes (the
// source row of an in-block step), without the LDS crossbar of a general shuffle: DPP
// inside rows of 16 lanes (quad_perm for blocks of 2 and 4, row_newbcast for 8 and 16)
// and v_readlane for 32 and 64.  c is a compile-time constant once the in-block loop is
// unrolled, so each switch folds to one instruction.  Every lane of the wave must be
// active (the in-block loop runs in uniform control flow).
template <int CTRL>
__device__ __forceinline__ int dpp_mov(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, false);
}
__device__ __forceinline__ int row_bcast16(int v, int n) {
    switch (n) {
        case 0: return dpp_mov<0x150>(v);
        case 1: return dpp_mov<0x151>(v);
        case 2: return dpp_mov<0x152>(v);
        case 3: return dpp_mov<0x153>(v);
        case 4: return dpp_mov<0x154>(v);
        case 5: return dpp_mov<0x155>(v);
        case 6: return dpp_mov<0x156>(v);
        case 7: return dpp_mov<0x157>(v);
        case 8: return dpp_mov<0x158>(v);
        case 9: return dpp_mov<0x159>(v);
        case 10: return dpp_mov<0x15a>(v);
        case 11: return dpp_mov<0x15b>(v);
        case 12: return dpp_mov<0x15c>(v);
        case 13: return dpp_mov<0x15d>(v);
        case 14: return dpp_mov<0x15e>(v);
        default: return dpp_mov<0x15f>(v);
    }
}
template <int BS>
__device__ __forceinline__ int block_bcast32(int v, int c) {
    const int lane = threadIdx.x & 63;
    if constexpr (BS == 2) {  // quad_perm [c, c, 2 + c, 2 + c]
        return c == 0 ? dpp_mov<0xa0>(v) : dpp_mov<0xf5>(v);
    } else if constexpr (BS == 4) {  // quad_perm [c, c, c, c]
        switch (c) {
            case 0: return dpp_mov<0x00>(v);
            case 1: return dpp_mov<0x55>(v);
            case 2: return dpp_mov<0xaa>(v);
            default: return dpp_mov<0xff>(v);
        }
    } else if constexpr (BS == 8) {
        const int a = row_bcast16(v, c), b = row_bcast16(v, c + 8);
        return (lane & 8) ? b : a;
    } else if constexpr (BS == 16) {
        return row_bcast16(v, c);
    } else if constexpr (BS == 32) {
        const int a = __builtin_amdgcn_readlane(v, c), b = __builtin_amdgcn_readlane(v, 32 + c);
        return lane < 32 ? a : b;
    } else {
        return __builtin_amdgcn_readlane(v, c);
    }
}
template <int BS, typename T>
__device__ __forceinline__ T block_bcast(T v, int c) {
    if constexpr (sizeof(T) == 4) {
        return __builtin_bit_cast(T, block_bcast32<BS>(__builtin_bit_cast(int, v), c));
    } else {
        const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
        const unsigned lo = (unsigned)block_bcast32<BS>((int)(unsigned)u, c);
        const unsigned hi = (unsigned)block_bcast32<BS>((int)(unsigned)(u >> 32), c);
        return __builtin_bit_cast(T, ((unsigned long long)hi << 32) | lo);
    }
}

// ------------------------------------------------------------ single-launch sweep
// In the sweep every row of the output starts as a sentinel: a signalling NaN, which
// no arithmetic produces (results are canonicalised before they are stored, so an
// input holding the pattern cannot leak through either).  A gather of an earlier row
// that still reads the sentinel polls again; a row's value is stored once, so the
// first non-sentinel value read is the final one.  Stores of the output and the polls
// go to the device-coherent level (every XCD has its own L2, which a row written on
// another XCD does not update).
template <typename T>
struct Bits {
    using U = unsigned;
    static constexpr U kSentinel = 0x7fa5a5a5u;
};
template <>
struct Bits<double> {
    using U = unsigned long long;
    static constexpr U kSentinel = 0x7ff4a5a5a5a5a5a5ull;
};
template <typename T>
__device__ __forceinline__ typename Bits<T>::U load_agent(const T *p) {
    using U = typename Bits<T>::U;
    return __hip_atomic_load((const U *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// First read of a gathered row: through the XCD's L2 (workgroup scope).  At the start of
// a launch no cache holds an older value of any row (the sentinels were written by an
// earlier launch), and within the launch a row changes once, from the sentinel to its
// final value; so this read gives the final value or the sentinel, and only a sentinel
// is polled again at device scope.
template <typename T>
__device__ __forceinline__ typename Bits<T>::U load_local(const T *p) {
    using U = typename Bits<T>::U;
    return __hip_atomic_load((const U *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <typename T>
__device__ __forceinline__ void store_agent(T *p, T v) {
    using U = typename Bits<T>::U;
    __hip_atomic_store((U *)p, __builtin_bit_cast(U, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float canonical(float v) { return __builtin_canonicalizef(v); }
__device__ __forceinline__ double canonical(double v) { return __builtin_canonicalize(v); }
// p + i; with O32 addressed as p's (uniform) base plus a 32-bit byte offset, one address
// register per access instead of a 64-bit pair (the launch checks that every array of the
// layout and every vector fits: i * sizeof(P) < 2^32)
template <bool O32, typename P>
__device__ __forceinline__ P *ixp(P *p, size_t i) {
    if constexpr (O32) {
        using Ch = typename std::conditional<std::is_const<P>::value, const char, char>::type;
        return reinterpret_cast<P *>(reinterpret_cast<Ch *>(p) + (size_t)((unsigned)i * (unsigned)sizeof(P)));
    } else {
        return p + i;
    }
}

// polls of one pending gather before the wave gives up and raises the time-out flag;
// a poll takes about a microsecond, so this bounds a wait at a few seconds
constexpr int kSweepSpinLimit = 1 << 22;

}  // namespace senk_amd
