// Epilogue of the prefill GEMMs whose lanes hold 8 consecutive product columns of a row.
#pragma once
#include "sc_common.h"

namespace sc {

// o: columns n .. n + 7 of the launch (product columns c .. c + 7) rounded to bf16; yr: the
// output row.  The bias is added to the rounded values and rounded again.  SWIGLU: columns
// 2j, 2j + 1 are gate j and up j and the row receives silu(gate) * up.  FAST: all 8 columns
// lie inside the matrix, rows are aligned for 16-byte (SwiGLU: 8-byte) stores, no bias.
template <bool FAST, bool SWIGLU>
__device__ __forceinline__ void store_cols8(uint32_t (&o)[4], uint16_t *yr, int c, int n, int N, const uint16_t *bias,
                                            int swiglu_i) {
    if (!FAST && bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int c0 = SWIGLU ? (c >> 1) + e : c + 2 * e, c1 = SWIGLU ? swiglu_i + c0 : c0 + 1;
            if (n + 2 * e < N)
                o[e] = cvt_pk_bf16(bf2f(o[e] & 0xFFFFu) + bf2f(bias[c0]),
                                   bf2f(o[e] >> 16) + (n + 2 * e + 1 < N ? bf2f(bias[c1]) : 0.f));
        }
    }
    if (SWIGLU) {
        float s[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] = silu_mul_f(bf2f(o[e] & 0xFFFFu), bf2f(o[e] >> 16));
        uint16_t *d = yr + (c >> 1);
        if (FAST) {
            *reinterpret_cast<uint2 *>(d) = make_uint2(cvt_pk_bf16(s[0], s[1]), cvt_pk_bf16(s[2], s[3]));
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n + 2 * e < N) d[e] = (uint16_t)f2bf(s[e]);
        }
    } else if (FAST) {
        *reinterpret_cast<uint4 *>(yr + c) = make_uint4(o[0], o[1], o[2], o[3]);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (n + 2 * e < N) yr[c + 2 * e] = (uint16_t)o[e];
            if (n + 2 * e + 1 < N) yr[c + 2 * e + 1] = (uint16_t)(o[e] >> 16);
        }
    }
}

}  // namespace sc
