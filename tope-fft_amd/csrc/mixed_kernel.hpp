// Mixed-radix axis pass for lengths n = 2^a 3^b 5^c 7^d <= 4096 (FP64, and
// complex64 storage with FP32 arithmetic and the tables rounded once).
// The reference runs such 1D sizes as an O(n^2) DFT (src/fft1d.c:148-232,
// src/kernels1D.cl:549-573) and rejects them in 2D/3D (src/fft2d.c:355-362,
// src/fft3d.c:522-533).
//
// Self-sorting Stockham, decimation in time, with a runtime list of radices
// 2 .. 16: stage s of radix r at span Ns treats butterfly j < n/r, reads
// j + m n/r (m < r), multiplies element m by W_{Ns r}^{(j mod Ns) m} and
// writes output m of its r-point DFT to (j / Ns) Ns r + (j mod Ns) + m Ns;
// starting at Ns = 1 the result is in natural order.  A block owns whole
// lines: its first stage reads them from memory, its last stage writes them
// back, so the pass is in place, and the stages in between exchange through
// one LDS buffer.  The twiddles are entries of a table per stage (exponents
// 1, 2, 4, 8; the others are products of those) and the constants inside a
// radix are correctly rounded literals, so no device sin/cos is evaluated.
//
// What bounds it: the latency of a stage -- one exchange, its barriers and
// its twiddles -- so the radices are as few as possible (mixed_schedule), the
// composite ones (6, 10, 12, 14, 15) are prime-factor DFTs without inner
// twiddles, and a thread keeps its butterflies in registers over the
// exchange, which leaves one LDS buffer instead of two and so twice the
// blocks on a CU.
// A forward and an inverse transform, against radices 2, 3, 4, 5, 7, 8, 16
// between two LDS buffers with roots from a two-level table: 3000^2 648 ->
// 321 us (rows 160 -> 68 us, 4.2 TB/s; columns 172 -> 99 us: a tile of three
// lines fills the LDS, so one block per CU alternates between memory and
// arithmetic), 100^3 85 -> 63.5 us, 1000^2 51 us, complex64 100^3 45 us.
// Twiddles read ahead of the barrier before their stage: 1-3 % of that.
#pragma once
#include "internal.hpp"
#include "real_bins.hpp"

namespace tope {


// Integer division by a runtime divisor without the emulated divide: a
// float reciprocal estimate, exact to +-1 for the operands here (< 2^24),
// then one correction.
struct Div32 {
    int d;
    float r;
};
__device__ __forceinline__ int divmod(int a, const Div32 &d, int &rem)
{
    int q = (int)((float)a * d.r);
    int r = a - q * d.d;
    if (r >= d.d) {
        ++q;
        r -= d.d;
    } else if (r < 0) {
        --q;
        r += d.d;
    }
    rem = r;
    return q;
}
// The same for 64-bit line numbers (< 2^40) through a double reciprocal.
struct Div64 {
    long long d;
    double r;
};
__device__ __forceinline__ long long divmod64(long long a, const Div64 &d, long long &rem)
{
    long long q = (long long)((double)a * d.r);
    long long r = a - q * d.d;
    if (r >= d.d) {
        ++q;
        r -= d.d;
    } else if (r < 0) {
        --q;
        r += d.d;
    }
    rem = r;
    return q;
}

// cos(2 pi m / r) and sin(2 pi m / r), m < r, for the odd radices: FP64
// values correctly rounded from 50-digit evaluations (complex64 rounds them
// once more).
template <int r>
__device__ __forceinline__ double odd_cos(int m)
{
    constexpr double c3[3] = {0x1p+0, -0x1p-1, -0x1p-1};
    constexpr double c5[5] = {0x1p+0, 0x1.3c6ef372fe950p-2, -0x1.9e3779b97f4a8p-1, -0x1.9e3779b97f4a8p-1,
                              0x1.3c6ef372fe950p-2};
    constexpr double c7[7] = {0x1p+0,
                              0x1.3f3a0e28bedd1p-1,
                              -0x1.c7b90e3024582p-3,
                              -0x1.cd4bca9cb5c71p-1,
                              -0x1.cd4bca9cb5c71p-1,
                              -0x1.c7b90e3024582p-3,
                              0x1.3f3a0e28bedd1p-1};
    return r == 3 ? c3[m] : r == 5 ? c5[m] : c7[m];
}
template <int r>
__device__ __forceinline__ double odd_sin(int m)
{
    constexpr double s3[3] = {0.0, 0x1.bb67ae8584caap-1, -0x1.bb67ae8584caap-1};
    constexpr double s5[5] = {0.0, 0x1.e6f0e134454ffp-1, 0x1.2cf2304755a5ep-1, -0x1.2cf2304755a5ep-1,
                              -0x1.e6f0e134454ffp-1};
    constexpr double s7[7] = {0.0,
                              0x1.904c37505de4bp-1,
                              0x1.f329c0558e969p-1,
                              0x1.bc4c04d71abc1p-2,
                              -0x1.bc4c04d71abc1p-2,
                              -0x1.f329c0558e969p-1,
                              -0x1.904c37505de4bp-1};
    return r == 3 ? s3[m] : r == 5 ? s5[m] : s7[m];
}

// Odd prime radix r by the conjugate-pair form: with a_j = x_j + x_{r-j},
// b_j = x_j - x_{r-j} and W_r^{jk} = c + i s,
//   y_k = A_k + i B_k, y_{r-k} = A_k - i B_k,
//   A_k = x_0 + sum_{j=1}^{(r-1)/2} a_j c_jk, B_k = sum b_j s_jk.
template <int r, int SIGN, typename R>
__device__ __forceinline__ void dft_odd(cpx<R> (&x)[r])
{
    constexpr int h = (r - 1) / 2;
    cpx<R> a[h], b[h];
#pragma unroll
    for (int j = 1; j <= h; ++j) {
        a[j - 1] = x[j] + x[r - j];
        b[j - 1] = x[j] - x[r - j];
    }
    const cpx<R> x0 = x[0];
#pragma unroll
    for (int j = 0; j < h; ++j) x[0] = x[0] + a[j];
#pragma unroll
    for (int k = 1; k <= h; ++k) {
        cpx<R> A = x0, B{0, 0};
#pragma unroll
        for (int j = 1; j <= h; ++j) {
            const R c = (R)odd_cos<r>((j * k) % r);
            const R s = (R)(SIGN < 0 ? -odd_sin<r>((j * k) % r) : odd_sin<r>((j * k) % r));
            A = fmac(a[j - 1], c, A);
            if (j == 1) B = scale(b[0], s);
            else B = fmac(b[j - 1], s, B);
        }
        // i B
        x[k] = cpx<R>{A.x - B.y, A.y + B.x};
        x[r - k] = cpx<R>{A.x + B.y, A.y - B.x};
    }
}

// 9-point DFT as 3 x 3: columns over n1 (x[n2 + 3 n1]), W_9^{n2 k1}, rows
// over n2 to X[k1 + 3 k2]; W_9^1, W_9^2, W_9^4 correctly rounded.
template <int SIGN, typename R>
__device__ __forceinline__ void dft9(cpx<R> (&x)[9])
{
    cpx<R> y[3][3];
#pragma unroll
    for (int n2 = 0; n2 < 3; ++n2) {
        cpx<R> c[3] = {x[n2], x[n2 + 3], x[n2 + 6]};
        dft_odd<3, SIGN>(c);
#pragma unroll
        for (int k = 0; k < 3; ++k) y[k][n2] = c[k];
    }
    y[1][1] = rotc<SIGN>(y[1][1], (R)0x1.8836fa2cf5039p-1, (R)0x1.491b7523c161dp-1);
    y[1][2] = rotc<SIGN>(y[1][2], (R)0x1.63a1a7e0b738ap-3, (R)0x1.f838b8c811c17p-1);
    y[2][1] = rotc<SIGN>(y[2][1], (R)0x1.63a1a7e0b738ap-3, (R)0x1.f838b8c811c17p-1);
    y[2][2] = rotc<SIGN>(y[2][2], (R)-0x1.e11f642522d1cp-1, (R)0x1.5e3a8748a0bf5p-2);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        dft_odd<3, SIGN>(y[k]);
#pragma unroll
        for (int m = 0; m < 3; ++m) x[k + 3 * m] = y[k][m];
    }
}

template <int r, int SIGN, typename R>
__device__ __forceinline__ void dft_mixed(cpx<R> (&x)[r]);

// r = a b, coprime (Good-Thomas): input b n1 + a n2 mod r, output k at
// (k mod a, k mod b); no twiddles between the a- and b-point DFTs.
template <int a, int b, int SIGN, typename R>
__device__ __forceinline__ void dft_pfa(cpx<R> (&x)[a * b])
{
    cpx<R> y[a][b];
#pragma unroll
    for (int i = 0; i < a; ++i) {
#pragma unroll
        for (int j = 0; j < b; ++j) y[i][j] = x[(b * i + a * j) % (a * b)];
        dft_mixed<b, SIGN>(y[i]);
    }
#pragma unroll
    for (int j = 0; j < b; ++j) {
        cpx<R> c[a];
#pragma unroll
        for (int i = 0; i < a; ++i) c[i] = y[i][j];
        dft_mixed<a, SIGN>(c);
#pragma unroll
        for (int i = 0; i < a; ++i) y[i][j] = c[i];
    }
#pragma unroll
    for (int k = 0; k < a * b; ++k) x[k] = y[k % a][k % b];
}

template <int r, int SIGN, typename R>
__device__ __forceinline__ void dft_mixed(cpx<R> (&x)[r])
{
    if constexpr (r == 3 || r == 5 || r == 7) dft_odd<r, SIGN>(x);
    else if constexpr (r == 6) dft_pfa<2, 3, SIGN>(x);
    else if constexpr (r == 9) dft9<SIGN>(x);
    else if constexpr (r == 10) dft_pfa<2, 5, SIGN>(x);
    else if constexpr (r == 12) dft_pfa<4, 3, SIGN>(x);
    else if constexpr (r == 14) dft_pfa<2, 7, SIGN>(x);
    else if constexpr (r == 15) dft_pfa<3, 5, SIGN>(x);
    else dft<r, SIGN>(x);
}

// Registers: a thread holds up to E = MIXED_E elements (MIXED_WIDE in some
// complex64 columns, see mixed_schedule), as E / r butterflies of radix r
// (butterfly b, element m in v[b r + m]).
constexpr int MIXED_E = 16, MIXED_WIDE = 32;

// A stage of the block: radix-r butterfly bi < count is butterfly j of line
// t; neighbouring lanes take neighbouring j (BYLINE false) or lines.
struct Stage {
    int r, nb, Ns;      // nb = n / r
    Div32 dnb, dns;
    const void *tw;     // row a: W_{Ns r}^{kk 2^a}, kk < Ns
};

template <bool BYLINE>
__device__ __forceinline__ void stage_at(int bi, const Stage &st, const Div32 &dtb, int &t, int &j)
{
    if constexpr (BYLINE) j = divmod(bi, dtb, t);
    else t = divmod(bi, st.dnb, j);
}

// LDS slot of element i of line t: lines back to back, or (COL) element by
// element with the tile's lines side by side, tbp slots from one element to
// the next.
// Both are linear in i, so the r slots of a butterfly are one base and a
// uniform stride.  Reads are contiguous over the lanes and so are the writes
// but a first stage's, r slots apart: mixed_schedule puts a radix first that
// has few factors of two.
template <bool COL>
__device__ __forceinline__ int slot_of(int t, int i, int n, int tbp)
{
    if constexpr (COL) return i * tbp + t;
    else return t * n + i;
}
template <bool COL>
__host__ __device__ __forceinline__ int mixed_slots(int n, int tb, int tbp) { return COL ? n * tbp : n * tb; }

// LDS to registers and back.
template <int r, typename R, int NT, bool COL, int E>
__device__ __forceinline__ void stage_get(cpx<R> (&v)[E], const cpx<R> *lds, const Stage &st, int n, int tb,
                                          int tbp, const Div32 &dtb, int tid)
{
    const int step = COL ? st.nb * tbp : st.nb;
#pragma unroll
    for (int b = 0; b < E / r; ++b) {
        const int bi = tid + b * NT;
        if (bi < tb * st.nb) {
            int t, j;
            stage_at<COL>(bi, st, dtb, t, j);
            const int s = slot_of<COL>(t, j, n, tbp);
#pragma unroll
            for (int m = 0; m < r; ++m) v[b * r + m] = lds[s + m * step];
        }
    }
}

template <int r, typename R, int NT, bool COL, int E>
__device__ __forceinline__ void stage_put(const cpx<R> (&v)[E], cpx<R> *lds, const Stage &st, int n, int tb,
                                          int tbp, const Div32 &dtb, bool byline, int tid)
{
    const int step = COL ? st.Ns * tbp : st.Ns;
#pragma unroll
    for (int b = 0; b < E / r; ++b) {
        const int bi = tid + b * NT;
        if (bi < tb * st.nb) {
            int t, j, kk;
            if (COL && byline) stage_at<true>(bi, st, dtb, t, j);
            else stage_at<false>(bi, st, dtb, t, j);
            const int jn = divmod(j, st.dns, kk);
            const int s = slot_of<COL>(t, jn * st.Ns * r + kk, n, tbp);
#pragma unroll
            for (int m = 0; m < r; ++m) lds[s + m * step] = v[b * r + m];
        }
    }
}

// Twiddles of a thread's butterflies: exponents 1, 2, 4, 8 below r, read
// ahead of the barrier that the stage's LDS reads wait behind.
template <int r>
constexpr int mixed_ntw() { return r <= 2 ? 1 : r <= 4 ? 2 : r <= 8 ? 3 : 4; }
template <int r, typename R, int NT, bool COL, int BF>
__device__ __forceinline__ void stage_tw(cpx<R> (&w)[BF][mixed_ntw<r>()], const Stage &st, int tb,
                                         const Div32 &dtb, int tid)
{
#pragma unroll
    for (int b = 0; b < BF; ++b) {
        const int bi = tid + b * NT;
        if (bi < tb * st.nb) {
            int t, j, kk;
            stage_at<COL>(bi, st, dtb, t, j);
            divmod(j, st.dns, kk);
            const cpx<R> *tw = static_cast<const cpx<R> *>(st.tw) + kk;
#pragma unroll
            for (int a = 0; a < mixed_ntw<r>(); ++a) w[b][a] = tw[a * st.Ns];
        }
    }
}

// The butterflies of a stage, in registers; stage_run_tw with twiddles.
template <int r, int SIGN, typename R, int NT, int E>
__device__ __forceinline__ void stage_run(cpx<R> (&v)[E], const Stage &st, int tb, int tid)
{
#pragma unroll
    for (int b = 0; b < E / r; ++b) {
        if (tid + b * NT < tb * st.nb) {
            cpx<R> x[r];
#pragma unroll
            for (int m = 0; m < r; ++m) x[m] = v[b * r + m];
            dft_mixed<r, SIGN>(x);
#pragma unroll
            for (int m = 0; m < r; ++m) v[b * r + m] = x[m];
        }
    }
}
template <int r, int SIGN, typename R, int NT, int E, int BF>
__device__ __forceinline__ void stage_run_tw(cpx<R> (&v)[E], const cpx<R> (&wt)[BF][mixed_ntw<r>()],
                                             const Stage &st, int tb, int tid)
{
#pragma unroll
    for (int b = 0; b < BF; ++b) {
        if (tid + b * NT < tb * st.nb) {
            cpx<R> x[r], w[r];
#pragma unroll
            for (int m = 0; m < r; ++m) x[m] = v[b * r + m];
#pragma unroll
            for (int m = 1, a = 0; m < r; m <<= 1, ++a) w[m] = wt[b][a];
            apply_twiddles<SIGN>(x, w);
            dft_mixed<r, SIGN>(x);
#pragma unroll
            for (int m = 0; m < r; ++m) v[b * r + m] = x[m];
        }
    }
}

// Where the block's lines lie: line t of the block is line (o0, c0 + t) of
// the axis, carried into o past the C-th.
struct Lines {
    long long o0, c0, C;
    int left;  // lines of the block that the axis has
    double rC;
};
__device__ __forceinline__ void line_at(const Lines &g, int t, long long &o, long long &c)
{
    o = g.o0;
    c = g.c0 + t;
    if (c >= g.C) o += divmod64(c, Div64{g.C, g.rC}, c);
}

// First stage (Ns = 1): the input lines to registers (a line past the last
// reads the last one's elements; its results are not stored).
template <int r, typename R, int NT, int E>
__device__ __forceinline__ void stage_load(cpx<R> (&v)[E], const cpx<R> *in, const MixedArgs &a,
                                           const Lines &g, const Stage &st, const Div32 &dtb, bool byline, int tid)
{
#pragma unroll
    for (int b = 0; b < E / r; ++b) {
        const int bi = tid + b * NT;
        if (bi < a.tb * st.nb) {
            int t, j;
            if (byline) stage_at<true>(bi, st, dtb, t, j);
            else stage_at<false>(bi, st, dtb, t, j);
            long long o, c;
            line_at(g, min(t, g.left - 1), o, c);
            const cpx<R> *p = in + o * a.os + c * a.cs + j * a.is;
            const long long step = st.nb * a.is;
#pragma unroll
            for (int m = 0; m < r; ++m) v[b * r + m] = p[m * step];
        }
    }
}

// Last stage (Ns r = n, so butterfly j writes j + m Ns): registers to the
// output lines, scaled, with the four-step post-twiddle (POST).
template <int r, int SIGN, typename R, int NT, bool POST, int E>
__device__ __forceinline__ void stage_store(cpx<R> (&v)[E], cpx<R> *out, const MixedArgs &a,
                                            const Lines &g, const Stage &st, const Div32 &dtb, bool byline, int tid)
{
    const R sc = (R)a.scale;
#pragma unroll
    for (int b = 0; b < E / r; ++b) {
        const int bi = tid + b * NT;
        if (bi < a.tb * st.nb) {
            int t, j;
            if (byline) stage_at<true>(bi, st, dtb, t, j);
            else stage_at<false>(bi, st, dtb, t, j);
            if (t < g.left) {
                long long o, c;
                line_at(g, t, o, c);
                cpx<R> *p = out + o * a.oos + c * a.ocs + j * a.ois;
                const long long step = st.Ns * a.ois;
                if constexpr (POST) {
                    const int base = (int)(o * a.pt_o + c * a.pt_c);
                    const Div32 dsplit{a.pt_split, a.inv_split};
#pragma unroll
                    for (int m = 0; m < r; ++m) {  // the exponent base k stays below pt_n
                        // four lookups in flight: all r of them spill
                        if (m % 4 == 0) asm volatile("" ::: "memory");
                        int lo;
                        const int hi = divmod(base * (j + m * st.Ns), dsplit, lo);
                        v[b * r + m] = twmul<SIGN>(v[b * r + m], cmul(static_cast<const cpx<R> *>(a.pt_lo)[lo],
                                                                      static_cast<const cpx<R> *>(a.pt_hi)[hi]));
                    }
                }
                if (a.scale != 1.0) {
#pragma unroll
                    for (int m = 0; m < r; ++m) v[b * r + m] = scale(v[b * r + m], sc);
                }
#pragma unroll
                for (int m = 0; m < r; ++m) p[m * step] = v[b * r + m];
            }
        }
    }
}

// The thread's number, opaque to the optimiser: nothing that depends on the
// lane is hoisted out of a case of the switch, where the addresses of all
// thirteen radices would be live at once.
__device__ __forceinline__ int opaque_tid()
{
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    return tid;
}

// A case of the switch: the marks keep the optimiser from moving what ends
// (or starts) several cases alike -- the LDS writes -- behind (before) the
// switch, with the element arrays of all cases live there.
#define MIXED_CASE(r, CALL)                  \
    {                                        \
        asm volatile("; radix " #r);         \
        CALL(r);                             \
        asm volatile("; radix " #r " done"); \
    }
#define MIXED_SWITCH(rad, CALL)                \
    switch (rad) {                             \
    case 2: MIXED_CASE(2, CALL) break;      \
    case 3: MIXED_CASE(3, CALL) break;      \
    case 4: MIXED_CASE(4, CALL) break;      \
    case 5: MIXED_CASE(5, CALL) break;      \
    case 6: MIXED_CASE(6, CALL) break;      \
    case 7: MIXED_CASE(7, CALL) break;      \
    case 8: MIXED_CASE(8, CALL) break;      \
    case 9: MIXED_CASE(9, CALL) break;      \
    case 10: MIXED_CASE(10, CALL) break;    \
    case 12: MIXED_CASE(12, CALL) break;    \
    case 14: MIXED_CASE(14, CALL) break;    \
    case 15: MIXED_CASE(15, CALL) break;    \
    default: MIXED_CASE(16, CALL) break;     \
    }

// COL: tiles of strided lines, element-major in LDS, neighbouring lanes on
// neighbouring lines.  A stage is one case of a switch from its reads to its
// writes, barriers included (the radix is uniform), so that no registers
// are live from one case to another: carried over the switches, the element
// array spilled.
template <typename R, int SIGN, int NT, bool COL, bool POST, int E>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4)))
mixed_kernel(const cpx<R> *in, cpx<R> *out, const MixedArgs a)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    cpx<R> *lds = reinterpret_cast<cpx<R> *>(lds_raw);
    const int n = a.n, tb = a.tb, tbp = a.tbp;
    const Div32 dtb{tb, a.inv_tb};
    // strided lines share 128-byte segments with the neighbouring blocks'
    // lines: keep neighbours on one XCD (one L2)
    const long long l0 = xcd_block(COL ? 1 : 0) * tb;
    Lines g;
    g.left = (int)min((long long)tb, a.lines - l0);
    g.C = a.C;
    g.rC = a.inv_C;
    g.o0 = divmod64(l0, Div64{g.C, g.rC}, g.c0);
    const bool in_cols = COL && a.is != 1;

    auto stage = [&](int s) {
        const MixedStage &m = a.st[s];
        return Stage{m.r, m.nb, m.Ns, Div32{m.nb, m.inv_nb}, Div32{m.Ns, m.inv_Ns},
                     static_cast<const cpx<R> *>(a.tw) + m.tw};
    };
    const Stage first = stage(0);
#define MIXED_FIRST(r)                                                          \
    {                                                                           \
        cpx<R> v[E]{};                                                    \
        const int tid = opaque_tid();                                           \
        stage_load<r, R, NT>(v, in, a, g, first, dtb, in_cols, tid);            \
        stage_run<r, SIGN, R, NT>(v, first, tb, tid);                           \
        stage_put<r, R, NT, COL>(v, lds, first, n, tb, tbp, dtb, in_cols, tid);   \
    }
    MIXED_SWITCH(first.r, MIXED_FIRST)
    for (int s = 1; s < a.nst - 1; ++s) {
        const Stage st = stage(s);
#define MIXED_MID(r)                                                            \
    {                                                                           \
        cpx<R> v[E]{};                                                    \
        const int tid = opaque_tid();                                           \
        cpx<R> w[E / r][mixed_ntw<r>()]{};                              \
        stage_tw<r, R, NT, COL>(w, st, tb, dtb, tid);                           \
        __syncthreads();                                                        \
        stage_get<r, R, NT, COL>(v, lds, st, n, tb, tbp, dtb, tid);                  \
        __syncthreads();                                                        \
        stage_run_tw<r, SIGN, R, NT>(v, w, st, tb, tid);                        \
        stage_put<r, R, NT, COL>(v, lds, st, n, tb, tbp, dtb, COL, tid);             \
    }
        MIXED_SWITCH(st.r, MIXED_MID)
    }
    {
        const Stage st = stage(a.nst - 1);
#define MIXED_LAST(r)                                                           \
    {                                                                           \
        cpx<R> v[E]{};                                                    \
        const int tid = opaque_tid();                                           \
        cpx<R> w[E / r][mixed_ntw<r>()]{};                              \
        stage_tw<r, R, NT, COL>(w, st, tb, dtb, tid);                           \
        __syncthreads();                                                        \
        stage_get<r, R, NT, COL>(v, lds, st, n, tb, tbp, dtb, tid);                  \
        stage_run_tw<r, SIGN, R, NT>(v, w, st, tb, tid);                        \
        stage_store<r, SIGN, R, NT, POST>(v, out, a, g, st, dtb, COL, tid);     \
    }
        MIXED_SWITCH(st.r, MIXED_LAST)
    }
}

// Real rows of 2 n samples: the mixed-radix transform of a row read as n
// complex values and the half-spectrum step, in one pass.
//   R2C (SIGN = -1): the last stage leaves Z in the LDS and the block forms
//   each bin and its mirror from it; rows of n + 1 values, `pitch` apart.
//   C2R (SIGN = +1): the block forms Z from the bins in the LDS, where the
//   first stage reads it.
// What bounds it: memory, as the complex pass.  As two passes (the transform
// in place, then the step) every row was read and written twice: a forward
// and an inverse transform of 3000 x 3000 real values took 226 us, now 174
// (the step 25 us of each), 200 x 180 x 150 157 -> 129, 40 x 48 24 -> 19,
// complex64 3000 x 3000 155 -> 127.
template <typename R, int SIGN, int NT>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4)))
mixed_real_kernel(const cpx<R> *in, cpx<R> *out, const MixedArgs a, const MixedReal h)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    cpx<R> *lds = reinterpret_cast<cpx<R> *>(lds_raw);
    const int n = a.n, tb = a.tb, tbp = 1;
    const Div32 dtb{tb, a.inv_tb}, dpairs{n / 2 + 1, h.inv_pairs};
    const int count = tb * (n / 2 + 1);
    const cpx<R> *w = static_cast<const cpx<R> *>(h.w);
    const long long l0 = xcd_block(0) * tb;
    Lines g;
    g.left = (int)min((long long)tb, a.lines - l0);
    g.C = a.C;
    g.rC = a.inv_C;
    g.o0 = divmod64(l0, Div64{g.C, g.rC}, g.c0);

    auto stage = [&](int s) {
        const MixedStage &m = a.st[s];
        return Stage{m.r, m.nb, m.Ns, Div32{m.nb, m.inv_nb}, Div32{m.Ns, m.inv_Ns},
                     static_cast<const cpx<R> *>(a.tw) + m.tw};
    };
    constexpr int U = 4;  // pairs (k, n - k) of a thread in flight
    const Stage first = stage(0);
    if constexpr (SIGN < 0) {
#define REAL_FIRST(r)                                                     \
    {                                                                     \
        cpx<R> v[MIXED_E]{};                                              \
        const int tid = opaque_tid();                                     \
        stage_load<r, R, NT>(v, in, a, g, first, dtb, false, tid);        \
        stage_run<r, SIGN, R, NT>(v, first, tb, tid);                     \
        stage_put<r, R, NT, false>(v, lds, first, n, tb, tbp, dtb, false, tid); \
    }
        MIXED_SWITCH(first.r, REAL_FIRST)
    } else {
        const R sc = (R)h.scale;
        for (int i0 = threadIdx.x; i0 < count; i0 += U * NT) {
            cpx<R> xk[U], xm[U], wk[U], wm[U];
            int t[U], k[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                t[u] = divmod(min(i0 + u * NT, count - 1), dpairs, k[u]);
                const cpx<R> *X = in + (l0 + min(t[u], g.left - 1)) * h.pitch;
                xk[u] = X[k[u]];
                xm[u] = X[n - k[u]];
                wk[u] = w[k[u]];
                wm[u] = w[n - k[u]];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (i0 + u * NT >= count) continue;
                const int kk = k[u];
                if (h.pack && kk == 0) {  // column 0 holds X[0] + i X[n]
                    xm[u] = cpx<R>{xk[u].y, R(0)};
                    xk[u] = cpx<R>{xk[u].x, R(0)};
                }
                lds[t[u] * n + kk] = c2r_bin(xk[u], xm[u], wk[u], sc);
                if (kk > 0 && n - kk != kk) lds[t[u] * n + n - kk] = c2r_bin(xm[u], xk[u], wm[u], sc);
            }
        }
#define REAL_FIRST_LDS(r)                                                 \
    {                                                                     \
        cpx<R> v[MIXED_E]{};                                              \
        const int tid = opaque_tid();                                     \
        __syncthreads();                                                  \
        stage_get<r, R, NT, false>(v, lds, first, n, tb, tbp, dtb, tid);  \
        __syncthreads();                                                  \
        stage_run<r, SIGN, R, NT>(v, first, tb, tid);                     \
        stage_put<r, R, NT, false>(v, lds, first, n, tb, tbp, dtb, false, tid); \
    }
        MIXED_SWITCH(first.r, REAL_FIRST_LDS)
    }
    for (int s = 1; s < a.nst - (SIGN < 0 ? 0 : 1); ++s) {
        const Stage st = stage(s);
#define REAL_MID(r)                                                       \
    {                                                                     \
        cpx<R> v[MIXED_E]{};                                              \
        const int tid = opaque_tid();                                     \
        cpx<R> tw[MIXED_E / r][mixed_ntw<r>()]{};                       \
        stage_tw<r, R, NT, false>(tw, st, tb, dtb, tid);                  \
        __syncthreads();                                                  \
        stage_get<r, R, NT, false>(v, lds, st, n, tb, tbp, dtb, tid);     \
        __syncthreads();                                                  \
        stage_run_tw<r, SIGN, R, NT>(v, tw, st, tb, tid);                 \
        stage_put<r, R, NT, false>(v, lds, st, n, tb, tbp, dtb, false, tid); \
    }
        MIXED_SWITCH(st.r, REAL_MID)
    }
    if constexpr (SIGN > 0) {
        const Stage st = stage(a.nst - 1);
#define REAL_LAST(r)                                                      \
    {                                                                     \
        cpx<R> v[MIXED_E]{};                                              \
        const int tid = opaque_tid();                                     \
        cpx<R> tw[MIXED_E / r][mixed_ntw<r>()]{};                       \
        stage_tw<r, R, NT, false>(tw, st, tb, dtb, tid);                  \
        __syncthreads();                                                  \
        stage_get<r, R, NT, false>(v, lds, st, n, tb, tbp, dtb, tid);     \
        stage_run_tw<r, SIGN, R, NT>(v, tw, st, tb, tid);                 \
        stage_store<r, SIGN, R, NT, false>(v, out, a, g, st, dtb, false, tid); \
    }
        MIXED_SWITCH(st.r, REAL_LAST)
    } else {
        __syncthreads();
        const int here = g.left * (n / 2 + 1);
        for (int i0 = threadIdx.x; i0 < here; i0 += U * NT) {
            cpx<R> wk[U], wm[U];
            int t[U], k[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                t[u] = divmod(min(i0 + u * NT, here - 1), dpairs, k[u]);
                wk[u] = w[k[u]];
                wm[u] = w[n - k[u]];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (i0 + u * NT >= here) continue;
                const int kk = k[u];
                const cpx<R> zk = lds[t[u] * n + kk], zm = lds[t[u] * n + (kk ? n - kk : 0)];
                cpx<R> *X = out + (l0 + t[u]) * h.pitch;
                if (h.pack && kk == 0) {  // X[0] + i X[n] = (Re Z0 + Im Z0) + i (Re Z0 - Im Z0)
                    X[0] = cpx<R>{zk.x + zk.y, zk.x - zk.y};
                    continue;
                }
                X[kk] = r2c_bin(zk, zm, wk[u]);
                if (n - kk != kk) X[n - kk] = r2c_bin(zm, zk, wm[u]);
            }
        }
    }
}

// n <= 16: a radix of its own, one thread per line, no LDS.  (The factors of a
// four-step are never that short: 35 points is the least of any length.)
template <typename R, int SIGN>
__global__ void __launch_bounds__(256) mixed_one_kernel(const cpx<R> *in, cpx<R> *out, const MixedArgs a)
{
    const Div32 dtb{a.tb, a.inv_tb};
    const long long l0 = xcd_block(a.is != 1 ? 1 : 0) * a.tb;
    Lines g;
    g.left = (int)min((long long)a.tb, a.lines - l0);
    g.C = a.C;
    g.rC = a.inv_C;
    g.o0 = divmod64(l0, Div64{g.C, g.rC}, g.c0);
    const MixedStage &m = a.st[0];
    const Stage st{m.r, 1, 1, Div32{1, 1.0f}, Div32{1, 1.0f}, nullptr};
#define MIXED_ONE(r)                                                            \
    {                                                                           \
        cpx<R> v[MIXED_E]{};                                                    \
        const int tid = opaque_tid();                                           \
        stage_load<r, R, 256>(v, in, a, g, st, dtb, false, tid);                \
        stage_run<r, SIGN, R, 256>(v, st, a.tb, tid);                           \
        stage_store<r, SIGN, R, 256, false>(v, out, a, g, st, dtb, false, tid); \
    }
    MIXED_SWITCH(st.r, MIXED_ONE)
}

// The same for contiguous rows back to back: a block's rows go through LDS, so
// that neighbouring lanes move neighbouring elements; an odd pitch puts the
// lanes' rows on different banks.  What bounds it: memory.  A forward and an
// inverse transform of 10^6 rows, against a thread that reads its row from
// memory: FP64 3 points 40 -> 32 us, 7 points 112 -> 86, 12 points 212 -> 145,
// 15 points 337 -> 184 (5.2 TB/s), complex64 15 points 192 -> 93; 20000 rows of 15
// points 14.0 -> 9.0 us, 300 rows the same.  Blocks of 128 rows measure the same.
template <typename R, int SIGN>
__global__ void __launch_bounds__(MIXED_ROWS) mixed_rows_kernel(const cpx<R> *in, cpx<R> *out, const MixedArgs a)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    cpx<R> *lds = reinterpret_cast<cpx<R> *>(lds_raw);
    const long long l0 = xcd_block(0) * MIXED_ROWS;
    const int left = (int)min((long long)MIXED_ROWS, a.lines - l0);
    const R sc = (R)a.scale;
#define MIXED_ROW(r)                                                                  \
    {                                                                                 \
        constexpr int pitch = r | 1;                                                  \
        const int tid = opaque_tid();                                                 \
        const cpx<R> *p = in + l0 * r;                                                \
        cpx<R> *q = out + l0 * r;                                                     \
        cpx<R> x[r], *row = lds + tid * pitch;                                        \
        _Pragma("unroll") for (int m = 0; m < r; ++m)                                 \
        {                                                                             \
            const int i = tid + m * MIXED_ROWS;                                       \
            x[m] = i < left * r ? p[i] : cpx<R>{0, 0};                                \
        }                                                                             \
        _Pragma("unroll") for (int m = 0; m < r; ++m)                                 \
        {                                                                             \
            const int i = tid + m * MIXED_ROWS;                                       \
            lds[i / r * pitch + i % r] = x[m];                                        \
        }                                                                             \
        __syncthreads();                                                              \
        _Pragma("unroll") for (int m = 0; m < r; ++m) x[m] = row[m];                  \
        dft_mixed<r, SIGN>(x);                                                        \
        _Pragma("unroll") for (int m = 0; m < r; ++m) row[m] = scale(x[m], sc);       \
        __syncthreads();                                                              \
        _Pragma("unroll") for (int m = 0; m < r; ++m)                                 \
        {                                                                             \
            const int i = tid + m * MIXED_ROWS;                                       \
            if (i < left * r) q[i] = lds[i / r * pitch + i % r];                      \
        }                                                                             \
    }
    MIXED_SWITCH(a.n, MIXED_ROW)
}

// One launch of a precision and a direction (mixed_inst.hip holds one of
// each per object file).
template <typename R, int SIGN>
hipError_t launch_mixed_t(const void *in, void *out, const MixedArgs &a, unsigned grid, hipStream_t st);
template <typename R, int SIGN>
hipError_t launch_mixed_real_t(const void *in, void *out, const MixedArgs &a, const MixedReal &h, unsigned grid,
                               hipStream_t st);

}  // namespace tope
