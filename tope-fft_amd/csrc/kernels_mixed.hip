// Plans and launches of the mixed-radix axis pass (mixed_kernel.hpp).
#include <algorithm>
#include <vector>

#include "mixed_kernel.hpp"

namespace tope {

constexpr long long MIXED_LDS = 160 * 1024;  // of a CU

// The stage table: row a of stage s >= 1 (2^a < r) holds W_{Ns r}^{kk 2^a},
// gathered from W_n^i.
template <typename R>
__global__ void gen_mixed_kernel(cpx<R> *out, const cpx<R> *roots, const MixedArgs a)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.twsize) return;
    int s = 1;
    while (s + 1 < a.nst && i >= a.st[s + 1].tw) ++s;
    const int loc = i - a.st[s].tw, e = loc / a.st[s].Ns, kk = loc % a.st[s].Ns;
    out[i] = roots[(kk << e) * (a.n / (a.st[s].Ns * a.st[s].r))];
}

hipError_t gen_mixed_table(void *out, const void *roots, int prec, const MixedArgs &a, hipStream_t st)
{
    if (a.twsize < 1) return hipSuccess;
    const dim3 g((unsigned)((a.twsize + 255) / 256));
    if (prec == PREC_F64)
        hipLaunchKernelGGL(gen_mixed_kernel<double>, g, dim3(256), 0, st, static_cast<cpx<double> *>(out),
                           static_cast<const cpx<double> *>(roots), a);
    else
        hipLaunchKernelGGL(gen_mixed_kernel<float>, g, dim3(256), 0, st, static_cast<cpx<float> *>(out),
                           static_cast<const cpx<float> *>(roots), a);
    return hipGetLastError();
}

bool mixed_supported(long long n)
{
    if (n < 2 || n > MIXED_MAX_N) return false;
    for (long long p : {2, 3, 5, 7})
        while (n % p == 0) n /= p;
    return n == 1;
}

// Elements a thread can hold at radix r.
static int mixed_cap(int r, int e = MIXED_E) { return e / r * r; }

// Fewest radices of 2 .. 16 whose product is n; of those lists the one whose
// smallest mixed_cap is largest (more elements a thread), then the most
// balanced one.  Descending.
static std::vector<int> mixed_radices(int n)
{
    static const int kRadices[] = {16, 15, 14, 12, 10, 9, 8, 7, 6, 5, 4, 3, 2};
    std::vector<int> cur, best;
    auto cap = [](const std::vector<int> &v) {
        int c = MIXED_E;
        for (int r : v) c = std::min(c, mixed_cap(r));
        return c;
    };
    auto search = [&](auto &&self, int m, int from) -> void {
        if (m == 1) {
            if (best.empty() || cur.size() < best.size() ||
                (cur.size() == best.size() &&
                 (cap(cur) > cap(best) || (cap(cur) == cap(best) && cur[0] < best[0]))))
                best = cur;
            return;
        }
        if (!best.empty() && cur.size() + 1 > best.size()) return;
        for (int i = from; i < (int)(sizeof kRadices / sizeof kRadices[0]); ++i)
            if (m % kRadices[i] == 0) {
                cur.push_back(kRadices[i]);
                self(self, m / kRadices[i], i);
                cur.pop_back();
            }
    };
    search(search, n, 0);
    return best;
}

MixedArgs mixed_plan(long long n, long long O, long long os, long long C, long long cs, long long is)
{
    MixedArgs a{};
    a.n = (int)n;
    a.O = O;
    a.os = os;
    a.C = C;
    a.cs = cs;
    a.is = is;
    a.lines = O * C;
    a.scale = 1.0;
    a.oos = os;
    a.ocs = cs;
    a.ois = is;
    return a;
}

// Contiguous lines back to back, in and out.
static bool packed_rows(const MixedArgs &a)
{
    return a.is == 1 && a.ois == 1 && !a.pt_n && (a.C == 1 || (a.cs == a.n && a.ocs == a.n)) &&
           (a.O == 1 || (a.os == a.C * a.n && a.oos == a.C * a.n));
}

void mixed_schedule(MixedArgs &a, int prec)
{
    std::vector<int> rad = mixed_radices(a.n);
    a.nst = (int)rad.size();
    a.e = a.cap = MIXED_E;
    for (int r : rad) a.cap = std::min(a.cap, mixed_cap(r));

    // Tile: 256 threads, or as many more as a line (rows) or a 64-byte wide
    // tile (strided lines) needs.  Of the line counts that fit, the one whose
    // last wave of blocks leaves the least idle: a block costs its elements
    // plus a fixed latency worth about 1000 more, and 16 waves (four per SIMD at
    // 128 registers) or 160 KiB of LDS fill a CU.  Against the widest tile that
    // fits: 100^3 67.8 -> 63.5 us, 200 x 180 x 150 212 -> 200 us,
    // 48 x 60 x 56 40.0 -> 33.3 us (a forward and an inverse transform).
    // Strided lines take rows in segments of tb elements, and below 64 bytes
    // each costs more than its bytes: 2400 x 2400 takes 182 us in segments of
    // 64 bytes, 208 to 210 in 32 or 48 and 281 in 16 (its rows 88 of each);
    // complex64 115 in 32, 132 in 24, 137 in 16.  A
    // higher factor for 32 bytes loses where those tiles fill the chip better:
    // 900 x 900 50.7 us in 32 bytes, 55.5 in 16.
    const int eb = prec == PREC_F64 ? 16 : 8;
    const bool col = a.is != 1 || a.ois != 1;
    const int want = col ? 64 / eb : 1;
    a.tbp = 1;
    double best = 0;
    // The smallest column passes are one block: what the passes beside it wrote and
    // will read then stays in one L2.  complex64, in the blocks of least cost /
    // in one (forward and inverse, rows and columns): 64 x 20 15.9 / 14.3 us,
    // 16 x 24 14.3 / 12.6, FP64 64 x 18 16.1 / 15.3; even at 64 x 30 (16.8 /
    // 16.1, FP64 17.1 / 17.5), no gain from 64 x 36 on.
    const bool small = col && a.lines * a.n <= 2048;
    // the line count of least cost for threads of e elements
    auto tile = [&](int e, int cap, int nt, int most) {
        while (nt < (col ? 1024 : 512) && nt * cap < want * a.n) nt *= 2;
        most = std::max(1, std::min(nt * cap / a.n, most));
        for (int tb = most; tb >= 1; --tb) {
            if (tb != most && tb > want && tb % want) continue;  // whole 64-byte segments
            // an odd distance between a line's elements spreads the first
            // stage's writes over the banks; given up where the tile fits
            // only without (3600 x 3600, two lines for one: 570 -> 420 us)
            int tbp = tb | 1;
            if (col && (long long)a.n * tbp * eb > MIXED_LDS) tbp = tb;
            const long long bytes = (long long)eb * (col ? mixed_slots<true>(a.n, tb, tbp) : mixed_slots<false>(a.n, tb, tbp));
            if (bytes > MIXED_LDS) continue;
            const long long slots = 256 * std::min<long long>(MIXED_LDS / bytes, 1024 / nt);
            const long long blocks = (a.lines + tb - 1) / tb;
            const int seg = col ? tb * eb : 64;  // bytes of a row that a tile takes
            const double mem = seg < 24 ? 1.9 : seg < 32 ? 1.45 : seg < 64 ? 1.2 : 1.0;
            const double cost = (double)((blocks + slots - 1) / slots) * ((double)tb * a.n + 1000.0) * mem;
            if (best == 0 || cost < best) best = cost, a.tb = tb, a.tbp = tbp, a.nt = nt, a.e = e, a.cap = cap;
            if (small && tb >= a.lines) break;
        }
    };
    if (a.nst == 1) {
        a.nt = a.tb = packed_rows(a) ? MIXED_ROWS : 256;
    } else {
        tile(MIXED_E, a.cap, 256, 64);
        // complex64 columns of which 1024 threads hold fewer than four at 16
        // elements each (lengths above 2400 with radices that waste some):
        // 32 elements, three or four lines, where they cost less.  4000 x 4000
        // 354 -> 308 us, 1080 x 4000 155 -> 121, 600 x 3645 99 -> 72 (forward
        // and inverse); not 1050 x 2430, three lines of 16 elements a thread
        // 84, four of 32 95, nor 500 x 4000, 67 and 68.  Five and more lines, whose segments
        // straddle 32 bytes, lose: 3600^2 219 -> 247.
        if (prec == PREC_F32 && col && 4 * a.n > 1024 * a.cap) {
            int cap = MIXED_WIDE;
            for (int r : rad) cap = std::min(cap, mixed_cap(r, MIXED_WIDE));
            tile(MIXED_WIDE, cap, 1024, 4);
        }
    }
    if (a.tb > a.lines) {
        a.tb = (int)a.lines;
        a.tbp = a.tb | 1;
        if (col && (long long)a.n * a.tbp * eb > MIXED_LDS) a.tbp = a.tb;
    }
    a.inv_tb = 1.0f / (float)a.tb;
    a.inv_C = 1.0 / (double)a.C;
    a.inv_split = a.pt_split > 0 ? 1.0f / (float)a.pt_split : 0.0f;

    // Order: the largest radix first, which has no twiddles there; but where
    // neighbouring lanes write neighbouring butterflies r slots apart (rows,
    // narrow tiles), the one with the fewest factors of two (6000 x 2000, 80-
    // and 75-point tiles of 16 lines and more: 578 us, 596 us with that order
    // everywhere)
    if (a.tb < 8 || !col)
        std::stable_sort(rad.begin(), rad.end(), [](int x, int y) { return (x & -x) < (y & -y); });
    int Ns = 1, tw = 0;
    for (int s = 0; s < a.nst; ++s) {
        MixedStage &m = a.st[s];
        m.r = rad[s];
        m.nb = a.n / rad[s];
        m.Ns = Ns;
        m.inv_nb = 1.0f / (float)m.nb;
        m.inv_Ns = 1.0f / (float)Ns;
        m.tw = tw;
        if (s > 0)
            for (int e = 1; e < m.r; e <<= 1) tw += Ns;
        Ns *= m.r;
    }
    a.twsize = tw;
}

bool mixed4_split(long long n, long long *n1)
{
    if (n <= MIXED_MAX_N || n > (long long)MIXED_MAX_N * MIXED_MAX_N) return false;
    long long m = n;
    for (long long p : {2, 3, 5, 7})
        while (m % p == 0) m /= p;
    if (m != 1) return false;
    // the smallest divisor d >= sqrt(n) with d, n / d <= MIXED_MAX_N
    for (long long d = 1; d <= MIXED_MAX_N; ++d) {
        if (n % d || d * d < n || n / d > MIXED_MAX_N) continue;
        *n1 = d;
        return true;
    }
    return false;
}

unsigned mixed_grid(const MixedArgs &a) { return (unsigned)((a.lines + a.tb - 1) / a.tb); }

hipError_t launch_mixed(int prec, const void *in, void *out, const MixedArgs &a, int sign, hipStream_t st)
{
    const long long grid = (a.lines + a.tb - 1) / a.tb;
    const bool col = a.is != 1 || a.ois != 1;
    const long long bytes = (prec == PREC_F64 ? 16LL : 8LL) * (col ? mixed_slots<true>(a.n, a.tb, a.tbp) : mixed_slots<false>(a.n, a.tb, a.tbp));
    if (grid < 1 || grid > 0x7fffffffLL || a.nst < 1 || a.nst > MIXED_MAX_STAGES || a.tb < 1 ||
        (long long)a.tb * a.n > (long long)a.nt * a.cap || (a.nst > 1 && bytes > MIXED_LDS) ||
        (a.nt > 512 && !col) || (a.e != MIXED_E && (a.nt != 1024 || !col || prec != PREC_F32)) ||
        (col && a.nst > 1 && a.tbp < a.tb) || (a.nst == 1 && a.nt != (packed_rows(a) ? MIXED_ROWS : 256)) ||
        (a.pt_n && (!col || a.nst == 1)))
        return hipErrorInvalidValue;
    const unsigned g = (unsigned)grid;
    if (prec == PREC_F64)
        return sign < 0 ? launch_mixed_t<double, -1>(in, out, a, g, st) : launch_mixed_t<double, 1>(in, out, a, g, st);
    return sign < 0 ? launch_mixed_t<float, -1>(in, out, a, g, st) : launch_mixed_t<float, 1>(in, out, a, g, st);
}

// n <= 16 (one thread a line) has no LDS tile to form the bins in.
bool mixed_real_supported(long long n) { return n > 16 && mixed_supported(n); }

hipError_t launch_mixed_real(int prec, const void *in, void *out, const MixedArgs &a, MixedReal h, int sign,
                             hipStream_t st)
{
    const long long grid = (a.lines + a.tb - 1) / a.tb;
    const long long bytes = (prec == PREC_F64 ? 16LL : 8LL) * a.n * a.tb;
    if (grid < 1 || grid > 0x7fffffffLL || a.nst < 2 || a.nst > MIXED_MAX_STAGES || a.e != MIXED_E || a.tb < 1 || a.is != 1 ||
        a.ois != 1 || (a.nt != 256 && a.nt != 512) || (long long)a.tb * a.n > (long long)a.nt * a.cap ||
        bytes > MIXED_LDS || a.pt_n || h.pitch <= a.n || in == out)
        return hipErrorInvalidValue;
    h.inv_pairs = 1.0f / (float)(a.n / 2 + 1);
    const unsigned g = (unsigned)grid;
    if (prec == PREC_F64)
        return sign < 0 ? launch_mixed_real_t<double, -1>(in, out, a, h, g, st)
                        : launch_mixed_real_t<double, 1>(in, out, a, h, g, st);
    return sign < 0 ? launch_mixed_real_t<float, -1>(in, out, a, h, g, st)
                    : launch_mixed_real_t<float, 1>(in, out, a, h, g, st);
}

}  // namespace tope
