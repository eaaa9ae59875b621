// Half-spectrum step of a real row of n = 2 m samples read as m complex ones
// (kernels_real.hip has the formulas), one bin at a time.
#pragma once
#include "cplx.hpp"

namespace tope {

// X[k] from a = Z[k], bc = Z[m - k], w = W_n^k
template <typename R>
__device__ __forceinline__ cpx<R> r2c_bin(cpx<R> a, cpx<R> bc, cpx<R> w)
{
    const cpx<R> b{bc.x, -bc.y};
    const cpx<R> e{R(0.5) * (a.x + b.x), R(0.5) * (a.y + b.y)};
    // O = (a - b) / (2i) = (Im(a-b), -Re(a-b)) / 2
    const cpx<R> o{R(0.5) * (a.y - b.y), R(-0.5) * (a.x - b.x)};
    const cpx<R> wo = cmul(w, o);
    return cpx<R>{e.x + wo.x, e.y + wo.y};
}

// Z[k] from a = X[k], bc = X[m - k], w = W_n^k, scaled by s
template <typename R>
__device__ __forceinline__ cpx<R> c2r_bin(cpx<R> a, cpx<R> bc, cpx<R> w, R s)
{
    const cpx<R> b{bc.x, -bc.y};
    const cpx<R> e{R(0.5) * (a.x + b.x), R(0.5) * (a.y + b.y)};
    const cpx<R> d{R(0.5) * (a.x - b.x), R(0.5) * (a.y - b.y)};
    const cpx<R> o = cmulc(d, w);  // d * conj(W^k)
    // Z = E + i O
    return cpx<R>{s * (e.x - o.y), s * (e.y + o.x)};
}

}  // namespace tope
