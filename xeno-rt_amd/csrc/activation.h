// The activation of a gated product, out = act(a . w_gate) * (a . w_up): one code, one formula, here.
// A product's mode carries the code in its bits from 8 up (mode 2 alone is the gated product with SiLU).
// Another activation is another code and another case below; every kernel with a gated epilogue
// takes the code as an argument and calls gate_activation.
#pragma once
#include "common.h"

#include "xrt_hip.h"

enum { XRT_ACT_COUNT = 1 };          // codes XRT_ACT_* of xrt_hip.h below this are known

inline int mode_of(int mode) { return mode & 255; }
inline int activation_of(int mode) { return mode >> 8; }

// 1 / (1 + e) for e = exp(something), 0 to infinity: correctly rounded, in six instructions where a division takes twelve. The
// hardware's reciprocal, a unit in the last place off, and one Newton step; both scaled by 2^-24, because the reciprocal has no
// denormal results (those of e beyond 2^126 are rounded twice so); infinity goes to 0. Compared with the division for every
// float32 e on gfx950: no normal result differs.
__device__ __forceinline__ float one_over_one_plus(float e) {
    const float scaled = fmaf(e, 0x1p-24f, 0x1p-24f), guess = __builtin_amdgcn_rcpf(scaled);
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-scaled, guess, 1.0f), guess, guess), scaled, 1.0f) * 0x1p-24f;
}

// QUICK: the exponential by the hardware's own instruction (a few units in the last place of a float32), for results that are
// rounded to bfloat16 anyway; the division is as exact as the other's. (A prefill's gate/up product of 2048 rows, 28672 rows
// of w and k = 4096, with the bare reciprocal, so and with a division: 324, 328 and 332 us.)
template <bool QUICK = false>
__device__ __forceinline__ float gate_activation(float z, int activation) {
    switch (activation) {
        case XRT_ACT_SILU:
        default:                                    // silu(z) = z / (1 + exp(-z)): crates/xrt-kernels/src/cpu/silu.rs:1-3 of the reference
            if constexpr (QUICK) return z * one_over_one_plus(__expf(-z));
            else return z / (1.0f + expf(-z));
    }
}
