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

// QUICK: the exponential by the hardware's own instruction (a few units in the last place of a float32), for results that are
// rounded to bfloat16 anyway. The division is the exact one: the hardware's reciprocal is a unit in the last place off and
// has no denormal results, which takes the sigmoid of gates below -87 away, and scaled so that they stay it takes the gates
// below 2^-102. (A prefill's gate/up product of 2048 rows, 28672 rows of w and k = 4096: 331 us, with that reciprocal 324.)
template <bool QUICK = false>
__device__ __forceinline__ float gate_activation(float z, int activation) {
    switch (activation) {
        case XRT_ACT_SILU:
        default:                                    // silu(z) = z / (1 + exp(-z)): crates/xrt-kernels/src/cpu/silu.rs:1-3 of the reference
            if constexpr (QUICK) return z * __frcp_rn(1.0f + __expf(-z));
            else return z / (1.0f + expf(-z));
    }
}
