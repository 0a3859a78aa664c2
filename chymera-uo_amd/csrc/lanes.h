// Values of the neighbouring lane of a wavefront through DPP (a VALU move,
// no LDS round trip as for __shfl_up / __shfl_down):
//   lane_prev(x): x of lane i-1 (DPP wave_shr:1), 0 on lane 0;
//   lane_next(x): x of lane i+1 (DPP wave_shl:1), 0 on lane 63.
// Equal to __shfl_up(x, 1) / __shfl_down(x, 1) on every lane whose
// neighbour lies in its group; callers replace the values of the lanes at a
// group's edge, as they do for the shuffles.
#pragma once

#include <hip/hip_runtime.h>

namespace chy {

constexpr int kDppWaveShl1 = 0x130;  // lane i reads lane i+1
constexpr int kDppWaveShr1 = 0x138;  // lane i reads lane i-1
constexpr int kDppRowShl = 0x100;    // + n: lane i reads lane i+n of its row of 16 (0 past the row)
constexpr int kDppRowShr = 0x110;    // + n: lane i reads lane i-n of its row of 16 (0 past the row)

template <int CTRL>
__device__ __forceinline__ int dpp_move(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}

template <int CTRL>
__device__ __forceinline__ double dpp_move(double x)
{
    const long long v = __double_as_longlong(x);
    const int lo = dpp_move<CTRL>((int)(v & 0xffffffffll)), hi = dpp_move<CTRL>((int)(v >> 32));
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

template <int CTRL>
__device__ __forceinline__ float dpp_move(float x)
{
    return __int_as_float(dpp_move<CTRL>(__float_as_int(x)));
}

template <typename T>
__device__ __forceinline__ T lane_prev(T x)
{
    return dpp_move<kDppWaveShr1>(x);
}

template <typename T>
__device__ __forceinline__ T lane_next(T x)
{
    return dpp_move<kDppWaveShl1>(x);
}

// x of the lane at byte address addr (4 * lane, modulo the wavefront) through
// the LDS crossbar
__device__ __forceinline__ int crossbar_word(int v, int addr) { return __builtin_amdgcn_ds_bpermute(addr, v); }

// f applied to both words of x (double: low, then high)
template <typename F>
__device__ __forceinline__ double by_word(double x, F f)
{
    const long long v = __double_as_longlong(x);
    const int lo = f((int)(v & 0xffffffffll)), hi = f((int)(v >> 32));
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// a DPP move within a row of 16 lanes, 0 where it reads past the row
template <int CTRL>
__device__ __forceinline__ double row_move(double x)
{
    return by_word(x, [](int v) { return __builtin_amdgcn_mov_dpp(v, CTRL, 0xF, 0xF, true); });
}

// x of lane i ^ S, S = 4 or 8 (within a row of 16 lanes): a shift either way,
// the second written to its own half only
template <int S>
__device__ __forceinline__ double row_swap(double x)
{
    static_assert(S == 4 || S == 8, "halves of 8 or 16 lanes");
    return by_word(x, [](int v) {
        const int up = __builtin_amdgcn_mov_dpp(v, kDppRowShr + S, 0xF, 0xF, true);
        // the banks of 4 lanes that read upwards
        return __builtin_amdgcn_update_dpp(up, v, kDppRowShl + S, 0xF, S == 4 ? 0x5 : 0x3, false);
    });
}

// v of both halves of a pair of rows (S = 16) or of the wavefront (S = 32) on
// both: even is the first half's value, odd the second's, of the lane at the
// same place in its half
template <int S>
__device__ __forceinline__ void half_pair(int v, int &even, int &odd)
{
    if constexpr (S == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
        even = (int)r[0];
        odd = (int)r[1];
    } else {
        const auto r = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
        even = (int)r[0];
        odd = (int)r[1];
    }
}

}  // namespace chy
