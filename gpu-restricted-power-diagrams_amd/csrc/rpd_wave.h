// rpd_wave.h -- wave64 primitives for gfx950 (CDNA4): lane ids, ballots,
// lane reads of uniform values, scans and reductions across one wavefront.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>
#include <type_traits>

namespace rpd {

constexpr int kWave = 64;

__device__ __forceinline__ int lane_id() {
    return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
}

// The lanes where p holds.  (Of one comparison it is the comparison's own
// mask; a compound condition costs a select and another comparison, so
// conditions are combined as masks: ballot(x) & ballot(y) & m.)
__device__ __forceinline__ uint64_t ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }

// whether this lane's bit of the wave-uniform mask m is set
__device__ __forceinline__ bool in_mask(uint64_t m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

// base plus the number of set bits of m strictly below this lane
__device__ __forceinline__ int mbcnt(uint64_t m, int base = 0) {
    return __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), uint32_t(base)));
}

__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ uint32_t uni(uint32_t v) { return uint32_t(__builtin_amdgcn_readfirstlane(int(v))); }
__device__ __forceinline__ uint64_t uni(uint64_t v) {
    const uint32_t lo = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(v))));
    const uint32_t hi = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(v >> 32))));
    return (uint64_t(hi) << 32) | lo;
}
__device__ __forceinline__ double uni(double v) {
    return __longlong_as_double((long long)uni(uint64_t(__double_as_longlong(v))));
}

// value of v in lane l (l wave-uniform)
__device__ __forceinline__ int rlane(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ uint32_t rlane(uint32_t v, int l) { return uint32_t(__builtin_amdgcn_readlane(int(v), l)); }
__device__ __forceinline__ float rlane(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double rlane(double v, int l) {
    const long long b = __double_as_longlong(v);
    const uint32_t lo = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(b)), l));
    const uint32_t hi = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(uint64_t(b) >> 32)), l));
    return __longlong_as_double((long long)((uint64_t(hi) << 32) | lo));
}
__device__ __forceinline__ uint64_t rlane(uint64_t v, int l) {
    const uint32_t lo = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(v)), l));
    const uint32_t hi = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(v >> 32)), l));
    return (uint64_t(hi) << 32) | lo;
}

// ---- DPP (data-parallel primitives of the gfx9 VALU): row shifts inside a
// row of 16 lanes and row broadcasts of lanes 15 / 31 give a 64-lane
// inclusive scan in 6 steps without an LDS round trip.  Lanes a step does not
// write keep the identity element passed as `old`.
constexpr int kDppRowShr1 = 0x111, kDppRowShr2 = 0x112, kDppRowShr4 = 0x114, kDppRowShr8 = 0x118;
constexpr int kDppRowBcast15 = 0x142, kDppRowBcast31 = 0x143;

template <int CTRL, int ROW = 0xf, int BANK = 0xf>
__device__ __forceinline__ int dpp_i(int old, int v) {
    return __builtin_amdgcn_update_dpp(old, v, CTRL, ROW, BANK, false);
}
template <int CTRL, int ROW = 0xf, int BANK = 0xf>
__device__ __forceinline__ float dpp_f(float old, float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(v), CTRL, ROW, BANK, false));
}
template <int CTRL, int ROW = 0xf, int BANK = 0xf>
__device__ __forceinline__ double dpp_d(double old, double v) {
    const long long o = __double_as_longlong(old), b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(int(uint32_t(o)), int(uint32_t(b)), CTRL, ROW, BANK, false);
    const int hi = __builtin_amdgcn_update_dpp(int(uint32_t(uint64_t(o) >> 32)), int(uint32_t(uint64_t(b) >> 32)),
                                               CTRL, ROW, BANK, false);
    return __longlong_as_double((long long)((uint64_t(uint32_t(hi)) << 32) | uint32_t(lo)));
}

// inclusive scan with operator OP over the 64 lanes; ID is OP's identity
template <typename T, typename OP>
__device__ __forceinline__ T wave_incl_scan_op(T x, T id, OP op) {
    if constexpr (sizeof(T) == 8) {
        x = op(x, dpp_d<kDppRowShr1>(id, x));
        x = op(x, dpp_d<kDppRowShr2>(id, x));
        x = op(x, dpp_d<kDppRowShr4>(id, x));
        x = op(x, dpp_d<kDppRowShr8>(id, x));
        x = op(x, dpp_d<kDppRowBcast15, 0xa>(id, x));
        x = op(x, dpp_d<kDppRowBcast31, 0xc>(id, x));
    } else if constexpr (std::is_same<T, float>::value) {
        x = op(x, dpp_f<kDppRowShr1>(id, x));
        x = op(x, dpp_f<kDppRowShr2>(id, x));
        x = op(x, dpp_f<kDppRowShr4>(id, x));
        x = op(x, dpp_f<kDppRowShr8>(id, x));
        x = op(x, dpp_f<kDppRowBcast15, 0xa>(id, x));
        x = op(x, dpp_f<kDppRowBcast31, 0xc>(id, x));
    } else {
        x = op(x, dpp_i<kDppRowShr1>(id, x));
        x = op(x, dpp_i<kDppRowShr2>(id, x));
        x = op(x, dpp_i<kDppRowShr4>(id, x));
        x = op(x, dpp_i<kDppRowShr8>(id, x));
        x = op(x, dpp_i<kDppRowBcast15, 0xa>(id, x));
        x = op(x, dpp_i<kDppRowBcast31, 0xc>(id, x));
    }
    return x;
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
    return rlane(wave_incl_scan_op(v, T(0), [](T a, T b) { return a + b; }), 63);
}
template <typename T>
__device__ __forceinline__ T wave_max(T v) {
    return rlane(wave_incl_scan_op(v, T(-INFINITY), [](T a, T b) { return a > b ? a : b; }), 63);
}
template <typename T>
__device__ __forceinline__ T wave_min(T v) {
    return rlane(wave_incl_scan_op(v, T(INFINITY), [](T a, T b) { return a < b ? a : b; }), 63);
}
// Sums over the wave of four values at once: the lanes of row 0 (lanes 0-15)
// return that of x, of row 1 y, of row 2 z, of row 3 w.  The cross-row swaps
// fold two values into one register, so that the last four steps serve all of
// them: about 25 VALU instructions where four scans take 80.
__device__ __forceinline__ double fold_rows(double lo, double hi, bool half) {
    const uint64_t a = uint64_t(__double_as_longlong(lo)), b = uint64_t(__double_as_longlong(hi));
    uint64_t u, v;
    if (half) {
        const auto l = __builtin_amdgcn_permlane32_swap(uint32_t(a), uint32_t(b), false, false);
        const auto h = __builtin_amdgcn_permlane32_swap(uint32_t(a >> 32), uint32_t(b >> 32), false, false);
        u = (uint64_t(h[0]) << 32) | l[0];
        v = (uint64_t(h[1]) << 32) | l[1];
    } else {
        const auto l = __builtin_amdgcn_permlane16_swap(uint32_t(a), uint32_t(b), false, false);
        const auto h = __builtin_amdgcn_permlane16_swap(uint32_t(a >> 32), uint32_t(b >> 32), false, false);
        u = (uint64_t(h[0]) << 32) | l[0];
        v = (uint64_t(h[1]) << 32) | l[1];
    }
    return __longlong_as_double((long long)u) + __longlong_as_double((long long)v);
}
__device__ __forceinline__ double wave_sum4(double x, double y, double z, double w) {
    // lanes 0-31 x (y), 32-63 z (w); then rows x, y, z, w
    double r = fold_rows(fold_rows(x, z, true), fold_rows(y, w, true), false);
    r += dpp_d<0x128>(0.0, r);  // row_ror 8, 4, 2, 1
    r += dpp_d<0x124>(0.0, r);
    r += dpp_d<0x122>(0.0, r);
    r += dpp_d<0x121>(0.0, r);
    return r;
}

// Maximum over the wave of values >= 0 (their bits order as unsigned integers,
// whose maximum takes one DPP instruction a step).
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t x) {
    x = max(x, uint32_t(__builtin_amdgcn_update_dpp(0, int(x), kDppRowShr1, 0xf, 0xf, true)));
    x = max(x, uint32_t(__builtin_amdgcn_update_dpp(0, int(x), kDppRowShr2, 0xf, 0xf, true)));
    x = max(x, uint32_t(__builtin_amdgcn_update_dpp(0, int(x), kDppRowShr4, 0xf, 0xf, true)));
    x = max(x, uint32_t(__builtin_amdgcn_update_dpp(0, int(x), kDppRowShr8, 0xf, 0xf, true)));
    x = max(x, uint32_t(__builtin_amdgcn_update_dpp(0, int(x), kDppRowBcast15, 0xa, 0xf, true)));
    x = max(x, uint32_t(__builtin_amdgcn_update_dpp(0, int(x), kDppRowBcast31, 0xc, 0xf, true)));
    return rlane(x, 63);
}
__device__ __forceinline__ float wave_max_pos(float v) { return __uint_as_float(wave_max_u32(__float_as_uint(v))); }
__device__ __forceinline__ double wave_max_pos(double v) { return wave_max(v); }

// exclusive prefix sum across the wave
__device__ __forceinline__ int wave_excl_scan(int v) {
    return wave_incl_scan_op(v, 0, [](int a, int b) { return a + b; }) - v;
}

// Value of v in lane (lane ^ J), J a power of two below 64, on the VALU
// rather than the LDS crossbar: DPP quad permutes (J = 1, 2), row rotations
// by 4/12 and 8 within 16-lane rows (J = 4, 8), and the gfx950 cross-row
// swaps v_permlane16_swap / v_permlane32_swap (J = 16, 32).
template <int J>
__device__ __forceinline__ uint32_t xor_lane(uint32_t v) {
    static_assert(J == 1 || J == 2 || J == 4 || J == 8 || J == 16 || J == 32, "xor_lane");
    if constexpr (J == 1) {
        return uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0xB1, 0xf, 0xf, false));  // quad_perm 1,0,3,2
    } else if constexpr (J == 2) {
        return uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0x4E, 0xf, 0xf, false));  // quad_perm 2,3,0,1
    } else if constexpr (J == 4) {
        const uint32_t up = uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0x12C, 0xf, 0xf, false));  // row_ror 12
        const uint32_t dn = uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0x124, 0xf, 0xf, false));  // row_ror 4
        return (lane_id() & 4) ? dn : up;
    } else if constexpr (J == 8) {
        return uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0x128, 0xf, 0xf, false));  // row_ror 8
    } else if constexpr (J == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return (lane_id() & 16) ? r[0] : r[1];
    } else {
        const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        return (lane_id() & 32) ? r[0] : r[1];
    }
}
// same, J known only after loop unrolling
__device__ __forceinline__ uint32_t xor_lane(uint32_t v, int j) {
    switch (j) {
        case 1: return xor_lane<1>(v);
        case 2: return xor_lane<2>(v);
        case 4: return xor_lane<4>(v);
        case 8: return xor_lane<8>(v);
        case 16: return xor_lane<16>(v);
        default: return xor_lane<32>(v);
    }
}
__device__ __forceinline__ uint64_t xor_lane(uint64_t v, int j) {
    return (uint64_t(xor_lane(uint32_t(v >> 32), j)) << 32) | xor_lane(uint32_t(v), j);
}
// Value of v in lane - 1 (DPP wave_shr:1); lane 0 gets `first`.
__device__ __forceinline__ uint32_t shr_lane1(uint32_t v, uint32_t first) {
    return uint32_t(__builtin_amdgcn_update_dpp(int(first), int(v), 0x138, 0xf, 0xf, false));
}
__device__ __forceinline__ uint64_t shr_lane1(uint64_t v, uint64_t first) {
    return (uint64_t(shr_lane1(uint32_t(v >> 32), uint32_t(first >> 32))) << 32) | shr_lane1(uint32_t(v), uint32_t(first));
}

// index of the lowest set bit (m != 0)
__device__ __forceinline__ int lowest_bit(uint64_t m) { return __ffsll((long long)m) - 1; }

// Sum of the totals of the tiles before `tile`, found by one wave of the tile's
// workgroup (decoupled lookback).  state: a zeroed word per tile, which becomes
// (1, total), then (2, sum up to and with the tile), value in the low half:
// one 64-bit word, so nothing else is ordered by it.  Tiles are numbered by a
// ticket that a workgroup takes when it starts: the tiles before it have
// started too, and post their totals without waiting for anyone, so every wait
// ends.
__device__ __forceinline__ int tile_prefix(unsigned long long *state, int tile, int total) {
    const int lane = lane_id();
    auto post = [&](unsigned long long kind, int v) {
        if (lane == 0)
            __hip_atomic_store(state + tile, (kind << 32) | uint32_t(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    post(tile == 0 ? 2 : 1, total);
    int before = 0;
    for (int j0 = tile - 1; j0 >= 0; j0 -= 64) {
        const int j = j0 - lane;
        unsigned long long v = 2ull << 32;  // before the first tile: nothing
        if (j >= 0)
            while (((v = __hip_atomic_load(state + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) >> 32) == 0)
                __builtin_amdgcn_s_sleep(1);
        const uint64_t whole = ballot((v >> 32) == 2);
        const int last = whole ? lowest_bit(whole) : 63;
        before += wave_sum(lane <= last ? int(uint32_t(v)) : 0);
        if (whole) break;
    }
    if (tile > 0) post(2, before + total);
    return before;
}

}  // namespace rpd
