// Epilogue of the prefill GEMMs whose lanes hold 8 consecutive product columns of a row.
#pragma once
#include "sc_common.h"

namespace sc {

// Bias of the lane's columns n .. n + 7 of the launch (product columns c .. c + 7) as bf16
// pairs.  SWIGLU: columns 2j, 2j + 1 are gate j and up j.
template <bool SWIGLU>
__device__ __forceinline__ void load_bias8(uint32_t (&bb)[4], const uint16_t *bias, int c, int n, int N, int swiglu_i) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int c0 = SWIGLU ? (c >> 1) + e : c + 2 * e, c1 = SWIGLU ? swiglu_i + c0 : c0 + 1;
        bb[e] = n < N ? bias[c0] | (uint32_t)bias[c1] << 16 : 0u;
    }
}

// o: the lane's columns rounded to bf16; yr: the output row.  The bias, if there is one, is
// added to the rounded values and rounded again.  SWIGLU: the row receives silu(gate) * up.
// N is a multiple of 8, so the columns lie all inside the matrix or all outside, and rows are
// aligned for 16-byte (SwiGLU: 8-byte) stores.  INNER: all inside, no bias.
template <bool INNER, bool SWIGLU>
__device__ __forceinline__ void store_cols8(uint32_t (&o)[4], uint16_t *yr, int c, int n, int N, bool has_bias,
                                            const uint32_t (&bb)[4]) {
    if (!INNER && n >= N) return;
    if (!INNER && has_bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            o[e] = cvt_pk_bf16(bf2f(o[e] & 0xFFFFu) + bf2f(bb[e] & 0xFFFFu), bf2f(o[e] >> 16) + bf2f(bb[e] >> 16));
    }
    if (SWIGLU) {
        float s[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] = silu_mul_f(bf2f(o[e] & 0xFFFFu), bf2f(o[e] >> 16));
        *reinterpret_cast<uint2 *>(yr + (c >> 1)) = make_uint2(cvt_pk_bf16(s[0], s[1]), cvt_pk_bf16(s[2], s[3]));
    } else {
        *reinterpret_cast<uint4 *>(yr + c) = make_uint4(o[0], o[1], o[2], o[3]);
    }
}

// Whether an output of N columns (SwiGLU: 2 swiglu_half) is laid out for store_cols8.  Element
// stores (2 bytes a lane, rows apart) cost 14 us a round of 256 x 256 tiles, more than these
// kernels gain on most such products.
inline bool wide_rows(const uint16_t *y, int N, int swiglu_half) {
    return swiglu_half ? swiglu_half % 4 == 0 && (uintptr_t)y % 8 == 0 : N % 8 == 0 && (uintptr_t)y % 16 == 0;
}

}  // namespace sc
