// The SiLU gate of an MLP, one element.
#pragma once

#include <hip/hip_runtime.h>

namespace berth {

// silu(g) * u with every step rounded to fp16: e = exp(-g); s = 1 + e; r = 1 / s;
// t = g * r; out = t * u (crates/berth-kernels/csrc/ops/act.cu:35-69 and its fixture)
__device__ __forceinline__ _Float16 silu_mul_h(_Float16 g, _Float16 u)
{
    _Float16 e = (_Float16)expf(-(float)g);
    _Float16 s = (_Float16)1.0f + e;
    _Float16 r = (_Float16)(1.0f / (float)s);
    _Float16 t = g * r;
    return t * u;
}

}  // namespace berth
