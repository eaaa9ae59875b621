// The mixed-radix kernels of one precision and one direction, for real type
// MIXED_R and sign MIXED_SIGN: compiled once for each of the four.
#include "mixed_kernel.hpp"

namespace tope {

template <typename R, int SIGN, int NT, bool COL, bool POST, int E = MIXED_E>
static void launch(const void *in, void *out, const MixedArgs &a, unsigned grid, hipStream_t st)
{
    const size_t slots = (size_t)mixed_slots<COL>(a.n, a.tb, a.tbp);
    hipLaunchKernelGGL((mixed_kernel<R, SIGN, NT, COL, POST, E>), dim3(grid), dim3(NT), slots * sizeof(cpx<R>), st,
                       static_cast<const cpx<R> *>(in), static_cast<cpx<R> *>(out), a);
}

template <typename R, int SIGN, int NT>
static void launch_nt(const void *in, void *out, const MixedArgs &a, unsigned grid, hipStream_t st)
{
    if constexpr (NT == 1024 && sizeof(R) == 4)
        if (a.e == MIXED_WIDE) {
            if (a.pt_n) launch<R, SIGN, NT, true, true, MIXED_WIDE>(in, out, a, grid, st);
            else launch<R, SIGN, NT, true, false, MIXED_WIDE>(in, out, a, grid, st);
            return;
        }
    const bool col = a.is != 1 || a.ois != 1;  // the planner's post-twiddle passes are strided
    // (in this order in the code object too, whose layout moves a pass by 1 to 2 %:
    // 100^3 64.0 us with the post-twiddle form first, 63.4 so, 1000^2 51.1 and 50.6)
    if (col && !a.pt_n) launch<R, SIGN, NT, true, false>(in, out, a, grid, st);
    else if (a.pt_n) launch<R, SIGN, NT, true, true>(in, out, a, grid, st);
    else if constexpr (NT <= 512) launch<R, SIGN, NT, false, false>(in, out, a, grid, st);
}

template <typename R, int SIGN>
hipError_t launch_mixed_t(const void *in, void *out, const MixedArgs &a, unsigned grid, hipStream_t st)
{
    if (a.nst == 1) {
        const cpx<R> *i = static_cast<const cpx<R> *>(in);
        cpx<R> *o = static_cast<cpx<R> *>(out);
        if (a.nt == MIXED_ROWS)
            hipLaunchKernelGGL((mixed_rows_kernel<R, SIGN>), dim3(grid), dim3(MIXED_ROWS),
                               (size_t)MIXED_ROWS * (a.n | 1) * sizeof(cpx<R>), st, i, o, a);
        else
            hipLaunchKernelGGL((mixed_one_kernel<R, SIGN>), dim3(grid), dim3(256), 0, st, i, o, a);
        return hipGetLastError();
    }
    switch (a.nt) {
    case 256: launch_nt<R, SIGN, 256>(in, out, a, grid, st); break;
    case 512: launch_nt<R, SIGN, 512>(in, out, a, grid, st); break;
    case 1024: launch_nt<R, SIGN, 1024>(in, out, a, grid, st); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <typename R, int SIGN>
hipError_t launch_mixed_real_t(const void *in, void *out, const MixedArgs &a, const MixedReal &h, unsigned grid,
                               hipStream_t st)
{
    const size_t bytes = (size_t)a.n * a.tb * sizeof(cpx<R>);
    const cpx<R> *i = static_cast<const cpx<R> *>(in);
    cpx<R> *o = static_cast<cpx<R> *>(out);
    if (a.nt == 256) hipLaunchKernelGGL((mixed_real_kernel<R, SIGN, 256>), dim3(grid), dim3(256), bytes, st, i, o, a, h);
    else hipLaunchKernelGGL((mixed_real_kernel<R, SIGN, 512>), dim3(grid), dim3(512), bytes, st, i, o, a, h);
    return hipGetLastError();
}

template hipError_t launch_mixed_t<MIXED_R, MIXED_SIGN>(const void *, void *, const MixedArgs &, unsigned, hipStream_t);
template hipError_t launch_mixed_real_t<MIXED_R, MIXED_SIGN>(const void *, void *, const MixedArgs &, const MixedReal &,
                                                             unsigned, hipStream_t);

}  // namespace tope
