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
__device__ __forceinline__ double crossbar(double x, int addr)
{
    const long long v = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_ds_bpermute(addr, (int)(v & 0xffffffffll));
    const int hi = __builtin_amdgcn_ds_bpermute(addr, (int)(v >> 32));
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// x of lane i ^ S, S a power of two; lane4 = 4 * lane.  Within a row of 16
// lanes by DPP: quad permutations for 1 and 2, for 4 and 8 a shift either way,
// the second written to its own half only.
template <int S>
__device__ __forceinline__ int lane_swap_word(int v)
{
    if constexpr (S == 1) return __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, false);  // quad [1,0,3,2]
    if constexpr (S == 2) return __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, false);  // quad [2,3,0,1]
    constexpr int lower = S == 4 ? 0x5 : 0x3;  // banks of 4 lanes that read upwards
    const int up = __builtin_amdgcn_update_dpp(0, v, kDppRowShr + S, 0xF, 0xF, false);
    return __builtin_amdgcn_update_dpp(up, v, kDppRowShl + S, 0xF, lower, false);
}

template <int S>
__device__ __forceinline__ double lane_swap(double x, int lane4)
{
    if constexpr (S <= 8) {
        const long long v = __double_as_longlong(x);
        const int lo = lane_swap_word<S>((int)(v & 0xffffffffll)), hi = lane_swap_word<S>((int)(v >> 32));
        return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
    } else {
        return crossbar(x, lane4 ^ (4 * S));
    }
}

}  // namespace chy
