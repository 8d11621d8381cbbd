// gdr_solve.hpp -- what the two chunked prefill kernels share: the 16 x 16
// unit lower triangular inverse by forward substitution, and the workgroup ->
// (sequence and head, rows) map.
#pragma once

#include <utility>

#include "gdr_device.hpp"

namespace rhz {

// a from lane R of each row of 16 lanes (DPP row_newbcast) times t, and the
// same added to acc: one VALU instruction each.  a is only ever written by LDS
// loads, so the DPP source needs no wait states.
template <int R>
__device__ __forceinline__ float bcast_mul(float a, float t) {
    float r;
    asm("v_mul_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "=v"(r) : "v"(a), "v"(t), "i"(R));
    return r;
}
template <int R>
__device__ __forceinline__ float bcast_fma(float a, float t, float acc) {
    asm("v_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(a), "v"(t), "i"(R));
    return acc;
}
// Forward substitution t_R = -sum_{s<R} A[R][s] t_s in column order: once t_S
// is final it is folded into the partial sums of every later row R > S, with
// A[R][S] broadcast from the lane that holds row R.  Each row still sums its
// terms in increasing s, but the rows' sums advance together, so the
// dependent chain is one multiply-add per row instead of one per term.
template <int R>
__device__ __forceinline__ void t_diag_init(float* acc, const float* a, const float* t) {
    acc[R] = bcast_mul<R>(a[0], t[0]);
}
template <int S, int R>
__device__ __forceinline__ void t_diag_fold(float* acc, const float* a, const float* t) {
    acc[R] = bcast_fma<R>(a[S], t[S], acc[R]);
}
template <int S, int... R>
__device__ __forceinline__ void t_diag_col(float* t, float* acc, const float* a, int col,
                                           std::integer_sequence<int, R...>) {
    if (S > col) t[S] = -acc[S];
    (t_diag_fold<S, S + 1 + R>(acc, a, t), ...);
}
template <int... S>
__device__ __forceinline__ void t_diag_solve(float* t, const float* a, int col, std::integer_sequence<int, S...>) {
    float acc[16];
    (t_diag_init<S + 1>(acc, a, t), ...);
    (t_diag_col<S + 1>(t, acc, a, col, std::make_integer_sequence<int, 14 - S>{}), ...);
}

// Workgroup -> (unit = seq-order index * H + h, tile).  Consecutive
// workgroup ids go round-robin to the 8 XCDs, so the tiles of one unit are
// placed 8 ids apart and share that XCD's L2 (every tile of a unit reads the
// same K, Q and gates).
__device__ __forceinline__ void map_block(int bid, int units, int nt, int& unit, int& tile) {
    const int full = (units / 8) * 8 * nt;
    if (bid < full) {
        const int xcd = bid & 7, slot = bid >> 3;
        tile = slot % nt;
        unit = (slot / nt) * 8 + xcd;
    } else {
        const int rem = bid - full;
        unit = (units / 8) * 8 + rem / nt;
        tile = rem % nt;
    }
}

}  // namespace rhz
