// Non-power-of-two axes by Bluestein's chirp-z identity on top of the
// power-of-two passes.  The reference runs 1D non-powers of two as an O(n^2)
// DFT (src/fft1d.c:148-232, src/kernels1D.cl:549-573) and rejects them in
// 2D/3D (src/fft2d.c:355-362, src/fft3d.c:522-533).
//
// With c[k] = W_2n^(k^2) (k^2 reduced mod 2n in integers, so the phase is
// exact) and jk = (j^2 + k^2 - (j-k)^2) / 2:
//   X[j] = c[j] sum_k (x[k] c[k]) conj(c[j-k]),
// a linear convolution of a[k] = x[k] c[k] with b[m] = conj(c[m]),
// |m| < n, evaluated as a circular one of power-of-two length M >= 2n - 1:
// A = FFT_M(a zero-padded), C = IFFT_M(A * FFT_M(b wrapped)), X[j] = c[j] C[j].
// The inverse transform uses conj(c) throughout.  Every line of an axis is
// padded into its own row of M elements of a scratch array, so the two inner
// FFTs are contiguous row passes.  Up to M = CHIRP_MAX_M a line's whole
// convolution runs in one workgroup instead (chirp_line_kernel), contiguous
// lines up to M = CHIRP_ROWS_M take three passes (chirp_cols_kernel).
#include "internal.hpp"

namespace tope {

__device__ __forceinline__ cpx<double> chirp(long long k, long long n, int inverse)
{
    // W_2n^(k^2): k^2 mod 2n in 64-bit integers (k < n <= 2^31)
    const unsigned long long m2 = 2ULL * (unsigned long long)n;
    const unsigned long long e = ((unsigned long long)k * (unsigned long long)k) % m2;
    double s, c;
    sincospi((double)e / (double)n, &s, &c);  // angle 2 pi e / 2n = pi e / n
    return cpx<double>{c, inverse ? s : -s};
}

// b (length M): b[m] = conj(c[m]) for m < n, b[M - m] = conj(c[m]) for
// 0 < m < n, zero elsewhere (c conjugated for the inverse's filter).
__global__ void chirp_filter_kernel(cpx<double> *b, long long n, long long M, int inverse)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= M) return;
    long long m = -1;
    if (i < n) m = i;
    else if (i > M - n) m = M - i;
    cpx<double> v{0.0, 0.0};
    if (m >= 0) {
        const cpx<double> c = chirp(m, n, inverse);
        v = cpx<double>{c.x, -c.y};
    }
    b[i] = v;
}

// c[k] = W_2n^(k^2), k < n, forward sign.
__global__ void chirp_table_kernel(cpx<double> *c, long long n)
{
    const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) c[k] = chirp(k, n, 0);
}

// One axis of lines of length n, M = N >= 2n - 1, in one launch: a block
// takes TB lines, multiplies them by the chirp as it loads them, runs the
// forward FFT_M, the product with the transformed filter and the inverse
// FFT_M in registers with LDS exchanges (run_stages), and stores the n
// outputs times the chirp.  In place, no padded array: an element is read
// and written once, where the separate passes moved 2 + 8 M/n elements per
// element through memory and evaluated a sincospi at both ends.  2D
// 1009 x 1009 (M = 2048): 133 us in ten launches -> 36 us in two.
//
// Each thread holds elements p + P e (P = N/16): n <= M/2, so those with
// e >= 8 are padding on the way in and unused on the way out.  Rows put the
// P threads of a line on neighbouring lanes; strided axes put TB adjacent
// lines there.  The real and imaginary parts are exchanged in turn, which
// halves the LDS of a tile, except in rows of M >= 2048, which fit four
// blocks per CU whole (1999 x 251: 52.1 -> 51.3 us, both for a forward and an
// inverse transform).  What bounds it now is the latency of its two serial
// transforms at two to three waves per SIMD (160-190 VGPRs): four waves
// (128 VGPRs) measured slower, 63 -> 82 us at 251 x 1999 and 52 -> 71 us at
// 1999 x 251, and leaving out the additions of the zero half changed nothing.
template <int N, int TB, bool CFAST>
__global__ void __launch_bounds__(TB *(N / 16))
chirp_line_kernel(const cpx<double> *in, cpx<double> *out, const ChirpLineArgs a)
{
    using R = double;
    constexpr int E = 16, P = N / E, H = E / 2;
    constexpr bool SPLIT = CFAST || N < 2048;
    __shared__ __align__(16) unsigned char lds[Exchange<R, N, E, TB, CFAST, SPLIT>::BYTES];
    const int tid = threadIdx.x;
    const int t = CFAST ? tid % TB : tid / P;
    const int p = CFAST ? tid / TB : tid % P;
    const cpx<R> *tw = static_cast<const cpx<R> *>(a.tw);
    const cpx<R> *ct = static_cast<const cpx<R> *>(a.chirp);
    const cpx<R> *fl = static_cast<const cpx<R> *>(a.filter);

    const long long blk = xcd_block(CFAST ? 1 : 0);
    const long long o = blk / a.tiles;
    const long long c = (blk - o * a.tiles) * TB + t;
    const bool valid = c < a.g.C;
    const long long at = o * a.g.os + c * a.g.cs;

    cpx<R> v[E];
#pragma unroll
    for (int e = 0; e < H; ++e) {
        const int k = p + P * e;
        v[e] = valid && k < a.n ? in[at + k * a.g.is] : cpx<R>{0, 0};
    }
#pragma unroll
    for (int e = 0; e < H; ++e) {
        const int k = p + P * e;
        const cpx<R> w = ct[k < a.n ? k : 0];
        v[e] = a.inverse ? cmulc(v[e], w) : cmul(v[e], w);
    }
#pragma unroll
    for (int e = H; e < E; ++e) v[e] = cpx<R>{0, 0};

    run_stages<R, N, E, TB, CFAST, SPLIT, -1, 0>(v, p, t, tw, lds);
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = cmul(v[e], fl[p + P * e]);
    __syncthreads();  // the forward transform's last exchange has been read
    run_stages<R, N, E, TB, CFAST, SPLIT, 1, 0>(v, p, t, tw, lds);

    if (!valid) return;
#pragma unroll
    for (int e = 0; e < H; ++e) {
        const int k = p + P * e;
        if (k < a.n) {
            const cpx<R> w = ct[k];
            const cpx<R> r = a.inverse ? cmulc(v[e], w) : cmul(v[e], w);
            out[at + k * a.g.is] = cpx<R>{r.x * a.scale, r.y * a.scale};
        }
    }
}

// Longer contiguous lines, M = n1 n2, element i = i1 n2 + i2 of a row of the
// padded array, bin k = k1 + n1 k2.  The forward transform's second half and the
// inverse's first half work on the same n2 contiguous elements (one k1), so a
// line's convolution is three passes and the bins are never put in order:
//   chirp_cols_kernel<PRE>   chirp, transforms over i1, W_M^(i2 k1)
//   chirp_mid_kernel         transform over i2, filter (kept in this order),
//                            inverse transform over k2
//   chirp_cols_kernel<POST>  W_M^-(i2 k1), inverse over k1, chirp, 1/M
// What bounds it: launches and latency at one line, else the memory of the
// padded rows, written twice and read twice (seven passes wrote them six
// times, with a sincospi for every element at both ends).
// A forward and an inverse transform: 3001 points 55 -> 23 us, 20011 55 -> 26,
// 300007 135 -> 68, 1000003 210 -> 116, 100 lines of 32771 954 -> 410.  Eight
// elements a thread; sixteen take 28, 29, 70, 111 and 467 us.
constexpr int CR_E = 8;
// v[e] *= W_M^(b (p + P e)) (SIGN < 0) or its conjugate: four table values
// and at most three products to a factor.
template <int SIGN>
__device__ __forceinline__ void chirp_twiddle(cpx<double> (&v)[CR_E], int b, int p, int P, const ChirpRowsArgs &a)
{
    const cpx<double> *lo = static_cast<const cpx<double> *>(a.lo), *hi = static_cast<const cpx<double> *>(a.hi);
    auto at = [&](int k) { return pt_lookup((long long)b * k, lo, hi, (long long)a.M, a.shift); };
    const cpx<double> s1 = at(P), s2 = at(2 * P), s4 = at(4 * P);
    cpx<double> w[4];
    w[0] = at(p);
    w[1] = cmul(w[0], s1);
    w[2] = cmul(w[0], s2);
    w[3] = cmul(w[1], s2);
#pragma unroll
    for (int e = 0; e < CR_E; ++e) v[e] = twmul<SIGN>(v[e], e < 4 ? w[e & 3] : cmul(w[e & 3], s4));
}

template <int N, int TB, bool POST>
__global__ void __launch_bounds__(TB *(N / CR_E))
chirp_cols_kernel(const cpx<double> *in, cpx<double> *out, const ChirpRowsArgs a)
{
    using R = double;
    constexpr int E = CR_E, P = N / E, H = E / 2;  // n <= M / 2: e >= H is padding
    __shared__ __align__(16) unsigned char lds[Exchange<R, N, E, TB, true, true>::BYTES];
    const int tid = threadIdx.x, t = tid % TB, p = tid / TB;
    const cpx<R> *tw = static_cast<const cpx<R> *>(a.tw1);
    const cpx<R> *ct = static_cast<const cpx<R> *>(a.chirp);

    const long long blk = xcd_block(1);
    const int tiles = a.n2 / TB;
    const long long l = blk / tiles;
    const int i2 = (int)(blk - l * tiles) * TB + t;
    const long long o = l / a.g.C, c = l - o * a.g.C;
    const long long at = o * a.g.os + c * a.g.cs, row = l * a.M;

    cpx<R> v[E];
    if constexpr (!POST) {
#pragma unroll
        for (int e = 0; e < H; ++e) {
            const int i = (p + P * e) * a.n2 + i2;
            v[e] = i < a.n ? in[at + i] : cpx<R>{0, 0};
        }
#pragma unroll
        for (int e = 0; e < H; ++e) {
            const int i = (p + P * e) * a.n2 + i2;
            const cpx<R> w = ct[i < a.n ? i : 0];
            v[e] = a.inverse ? cmulc(v[e], w) : cmul(v[e], w);
        }
#pragma unroll
        for (int e = H; e < E; ++e) v[e] = cpx<R>{0, 0};
        run_stages<R, N, E, TB, true, true, -1, 0>(v, p, t, tw, lds);
        chirp_twiddle<-1>(v, i2, p, P, a);
#pragma unroll
        for (int e = 0; e < E; ++e) out[row + (p + P * e) * a.n2 + i2] = v[e];
    } else {
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = in[row + (p + P * e) * a.n2 + i2];
        chirp_twiddle<1>(v, i2, p, P, a);
        run_stages<R, N, E, TB, true, true, 1, 0>(v, p, t, tw, lds);
#pragma unroll
        for (int e = 0; e < H; ++e) {
            const int i = (p + P * e) * a.n2 + i2;
            if (i < a.n) {
                const cpx<R> w = ct[i];
                const cpx<R> r = a.inverse ? cmulc(v[e], w) : cmul(v[e], w);
                out[at + i] = cpx<R>{r.x * a.scale, r.y * a.scale};
            }
        }
    }
}

template <int N, int TB>
__global__ void __launch_bounds__(TB *(N / CR_E)) chirp_mid_kernel(cpx<double> *S, const ChirpRowsArgs a)
{
    using R = double;
    constexpr int E = CR_E, P = N / E;
    __shared__ __align__(16) unsigned char lds[Exchange<R, N, E, TB, false, true>::BYTES];
    const int tid = threadIdx.x, t = tid / P, p = tid % P;
    const cpx<R> *tw = static_cast<const cpx<R> *>(a.tw2);
    const long long row = xcd_block(0) * TB + t;
    cpx<R> *s = S + row * N;
    const cpx<R> *fl = static_cast<const cpx<R> *>(a.filter) + (row & (a.n1 - 1)) * N;

    cpx<R> v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = s[p + P * e];
    run_stages<R, N, E, TB, false, true, -1, 0>(v, p, t, tw, lds);
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = cmul(v[e], fl[p + P * e]);
    __syncthreads();  // the forward transform's last exchange has been read
    run_stages<R, N, E, TB, false, true, 1, 0>(v, p, t, tw, lds);
#pragma unroll
    for (int e = 0; e < E; ++e) s[p + P * e] = v[e];
}

// out[k1 n2 + k2] = in[k1 + n1 k2]
__global__ void chirp_order_kernel(const cpx<double> *in, cpx<double> *out, int n1, int n2)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n1 * n2) out[i] = in[i / n2 + n1 * (i % n2)];
}

// Element k of line l (o = l / C, c = l % C) of the axis: o os + c cs + k is.
// Threads run along k when the axis is contiguous (is = 1), else along the
// lines (adjacent lines are adjacent in memory for the strided axes).
__device__ __forceinline__ void line_of(long long idx, const ChirpGeo &g, long long span, long long &l, long long &k)
{
    if (g.is == 1) {
        l = idx / span;
        k = idx % span;
    } else {
        const long long lines = g.O * g.C;
        k = idx / lines;
        l = idx % lines;
    }
}

__device__ __forceinline__ long long elem_of(long long l, long long k, const ChirpGeo &g)
{
    return (l / g.C) * g.os + (l % g.C) * g.cs + k * g.is;
}

// S[l M + k] = x_l[k] c[k] (k < n), 0 (n <= k < M)
__global__ void chirp_pre_kernel(const cpx<double> *__restrict__ x, cpx<double> *__restrict__ S, const ChirpGeo g,
                                 long long n, long long M, int inverse)
{
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= g.O * g.C * M) return;
    long long l, k;
    line_of(idx, g, M, l, k);
    cpx<double> v{0.0, 0.0};
    if (k < n) v = cmul(x[elem_of(l, k, g)], chirp(k, n, inverse));
    S[l * M + k] = v;
}

// S[l M + k] *= B[k] (the transformed filter of the direction)
__global__ void chirp_mul_kernel(cpx<double> *__restrict__ S, const cpx<double> *__restrict__ B, long long M,
                                 long long total)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < total) S[i] = cmul(S[i], B[i % M]);
}

// x_l[j] = c[j] S[l M + j] s (j < n)
__global__ void chirp_post_kernel(const cpx<double> *__restrict__ S, cpx<double> *__restrict__ x, const ChirpGeo g,
                                  long long n, long long M, double s, int inverse)
{
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= g.O * g.C * n) return;
    long long l, j;
    line_of(idx, g, n, l, j);
    const cpx<double> v = cmul(S[l * M + j], chirp(j, n, inverse));
    x[elem_of(l, j, g)] = cpx<double>{v.x * s, v.y * s};
}

template <int N, int TB, bool CFAST>
static hipError_t launch_line_t(const void *in, void *out, ChirpLineArgs a, hipStream_t st)
{
    a.tiles = (a.g.C + TB - 1) / TB;
    const long long grid = a.g.O * a.tiles;
    if (grid < 1 || grid > 0x7fffffffLL) return hipErrorInvalidValue;
    hipLaunchKernelGGL((chirp_line_kernel<N, TB, CFAST>), dim3((unsigned)grid), dim3(TB * (N / 16)), 0, st,
                       static_cast<const cpx<double> *>(in), static_cast<cpx<double> *>(out), a);
    return hipGetLastError();
}

// Rows: 64 to 256 threads a block.  Strided axes: tiles of WIDE adjacent
// lines, or NARROW ones where the wide tiles would leave CUs with no more than
// one block.  Up to M = 512 wide tiles gain a little (4096 x 251: 51.9 us, 53.8
// narrow; 8192 x 127 58.1 and 60.8); longer lines take one width, as more
// blocks of fewer waves hide their serial stages better than wider segments
// help: 4096 x 509 82 us in four lines, 90 in eight; 4096 x 1021 151 in two,
// 180 in four; 4096 x 2039 343 in two, 373 in four, whose 1024 threads leave
// 128 registers each and spill 24 (forward and inverse).
template <int N, int ROW, int WIDE, int NARROW>
static hipError_t launch_line_n(const void *in, void *out, const ChirpLineArgs &a, hipStream_t st)
{
    if (a.g.is == 1) return launch_line_t<N, ROW, false>(in, out, a, st);
    if (a.g.O * ((a.g.C + WIDE - 1) / WIDE) < 512) return launch_line_t<N, NARROW, true>(in, out, a, st);
    return launch_line_t<N, WIDE, true>(in, out, a, st);
}

hipError_t launch_chirp_lines(const void *in, void *out, const ChirpLineArgs &a, hipStream_t st)
{
    if (a.n < 1 || 2LL * a.n - 1 > a.M) return hipErrorInvalidValue;
    switch (a.M) {
    case 32: return launch_line_n<32, 32, 32, 32>(in, out, a, st);
    case 64: return launch_line_n<64, 16, 16, 16>(in, out, a, st);
    case 128: return launch_line_n<128, 16, 16, 8>(in, out, a, st);
    case 256: return launch_line_n<256, 8, 16, 4>(in, out, a, st);
    case 512: return launch_line_n<512, 4, 8, 4>(in, out, a, st);
    case 1024: return launch_line_n<1024, 2, 4, 4>(in, out, a, st);
    case 2048: return launch_line_n<2048, 1, 2, 2>(in, out, a, st);
    case 4096: return launch_line_n<4096, 1, 2, 2>(in, out, a, st);
    default: return hipErrorInvalidValue;
    }
}

template <int N, int TB>
static hipError_t launch_cols_t(int op, const void *in, void *out, const ChirpRowsArgs &a, hipStream_t st)
{
    const long long grid = a.g.O * a.g.C * (a.n2 / TB);
    if (grid < 1 || grid > 0x7fffffffLL || a.n2 % TB) return hipErrorInvalidValue;
    const cpx<double> *i = static_cast<const cpx<double> *>(in);
    cpx<double> *o = static_cast<cpx<double> *>(out);
    if (op == CHIRP_PRE)
        hipLaunchKernelGGL((chirp_cols_kernel<N, TB, false>), dim3((unsigned)grid), dim3(TB * (N / CR_E)), 0, st, i, o, a);
    else
        hipLaunchKernelGGL((chirp_cols_kernel<N, TB, true>), dim3((unsigned)grid), dim3(TB * (N / CR_E)), 0, st, i, o, a);
    return hipGetLastError();
}

template <int N, int TB>
static hipError_t launch_mid_t(void *S, const ChirpRowsArgs &a, hipStream_t st)
{
    const long long rows = a.g.O * a.g.C * a.n1, grid = rows / TB;
    if (grid < 1 || grid > 0x7fffffffLL || rows % TB) return hipErrorInvalidValue;
    hipLaunchKernelGGL((chirp_mid_kernel<N, TB>), dim3((unsigned)grid), dim3(TB * (N / CR_E)), 0, st,
                       static_cast<cpx<double> *>(S), a);
    return hipGetLastError();
}

hipError_t launch_chirp_rows(int op, const void *in, void *out, const ChirpRowsArgs &a, hipStream_t st)
{
    if (a.n < 1 || 2LL * a.n - 1 > a.M || a.g.is != 1 || (long long)a.n1 * a.n2 != a.M || a.M > CHIRP_ROWS_M)
        return hipErrorInvalidValue;
    if (op == CHIRP_MUL) {
        switch (a.n2) {  // 64 threads or one row a block
        case 128: return launch_mid_t<128, 4>(out, a, st);
        case 256: return launch_mid_t<256, 2>(out, a, st);
        case 512: return launch_mid_t<512, 1>(out, a, st);
        case 1024: return launch_mid_t<1024, 1>(out, a, st);
        case 2048: return launch_mid_t<2048, 1>(out, a, st);
        case 4096: return launch_mid_t<4096, 1>(out, a, st);
        default: return hipErrorInvalidValue;
        }
    }
    switch (a.n1) {  // 64- to 128-byte row segments while 1024 threads hold them
    case 64: return launch_cols_t<64, 8>(op, in, out, a, st);
    case 128: return launch_cols_t<128, 4>(op, in, out, a, st);
    case 256: return launch_cols_t<256, 4>(op, in, out, a, st);
    case 512: return launch_cols_t<512, 4>(op, in, out, a, st);
    case 1024: return launch_cols_t<1024, 4>(op, in, out, a, st);
    case 2048: return launch_cols_t<2048, 4>(op, in, out, a, st);
    case 4096: return launch_cols_t<4096, 2>(op, in, out, a, st);
    default: return hipErrorInvalidValue;
    }
}

hipError_t gen_chirp_order(const void *in, void *out, int n1, int n2, hipStream_t st)
{
    hipLaunchKernelGGL(chirp_order_kernel, dim3((unsigned)((n1 * n2 + 255) / 256)), dim3(256), 0, st,
                       static_cast<const cpx<double> *>(in), static_cast<cpx<double> *>(out), n1, n2);
    return hipGetLastError();
}

hipError_t gen_chirp_table(void *out, long long n, hipStream_t st)
{
    hipLaunchKernelGGL(chirp_table_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                       static_cast<cpx<double> *>(out), n);
    return hipGetLastError();
}

static unsigned grid_of(long long count) { return (unsigned)((count + 255) / 256); }

hipError_t launch_chirp(int op, const void *in, void *out, const void *table, const ChirpGeo &g, long long n,
                        long long M, double s, int inverse, hipStream_t st)
{
    const cpx<double> *i = static_cast<const cpx<double> *>(in);
    cpx<double> *o = static_cast<cpx<double> *>(out);
    const long long lines = g.O * g.C;
    if ((lines * M + 255) / 256 > 0x7fffffffLL) return hipErrorInvalidValue;
    switch (op) {
    case CHIRP_FILTER:
        hipLaunchKernelGGL(chirp_filter_kernel, dim3(grid_of(M)), dim3(256), 0, st, o, n, M, inverse);
        break;
    case CHIRP_PRE:
        hipLaunchKernelGGL(chirp_pre_kernel, dim3(grid_of(lines * M)), dim3(256), 0, st, i, o, g, n, M, inverse);
        break;
    case CHIRP_MUL:
        hipLaunchKernelGGL(chirp_mul_kernel, dim3(grid_of(lines * M)), dim3(256), 0, st, o,
                           static_cast<const cpx<double> *>(table), M, lines * M);
        break;
    case CHIRP_POST:
        hipLaunchKernelGGL(chirp_post_kernel, dim3(grid_of(lines * n)), dim3(256), 0, st, i, o, g, n, M, s, inverse);
        break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace tope
