// Instantiations of the persistent uneven-batch kernel.
#include "internal.hpp"
#include "many_kernel.hpp"

namespace tope {

template <typename R, int NT>
static hipError_t launch_many_t(const void *in, void *out, const void *args, int grid, int sign, hipStream_t s)
{
    const ManyArgs<R> &a = *static_cast<const ManyArgs<R> *>(args);
    const cpx<R> *i = static_cast<const cpx<R> *>(in);
    cpx<R> *o = static_cast<cpx<R> *>(out);
    // arrays that outgrow the 256 MB Infinity Cache twice over stream their
    // stores (streamed lines skip that cache too): 20000 FP64 transforms of 64 ..
    // 16384 points (1.2 GB) 513 -> 486 us; 2000 of them (115 MB) over and over on
    // one array would go from 62 to 66
    const bool stream = a.elems * (long long)sizeof(cpx<R>) >= 512LL << 20;
    if (sign < 0) {
        if (stream) hipLaunchKernelGGL((many_kernel<R, -1, NT, true>), dim3(grid), dim3(NT), 0, s, i, o, a);
        else hipLaunchKernelGGL((many_kernel<R, -1, NT, false>), dim3(grid), dim3(NT), 0, s, i, o, a);
    } else {
        if (stream) hipLaunchKernelGGL((many_kernel<R, 1, NT, true>), dim3(grid), dim3(NT), 0, s, i, o, a);
        else hipLaunchKernelGGL((many_kernel<R, 1, NT, false>), dim3(grid), dim3(NT), 0, s, i, o, a);
    }
    return hipGetLastError();
}

hipError_t launch_many(int prec, int threads, const void *in, void *out, const void *args, int grid, int sign,
                       hipStream_t s)
{
    const bool d = prec == PREC_F64;
    switch (threads) {
    case MANY_SMALL_THREADS:
        return d ? launch_many_t<double, MANY_SMALL_THREADS>(in, out, args, grid, sign, s)
                 : launch_many_t<float, MANY_SMALL_THREADS>(in, out, args, grid, sign, s);
    case MANY_THREADS:
        return d ? launch_many_t<double, MANY_THREADS>(in, out, args, grid, sign, s)
                 : launch_many_t<float, MANY_THREADS>(in, out, args, grid, sign, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace tope
