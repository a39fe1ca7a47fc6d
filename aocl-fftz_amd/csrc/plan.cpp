// GPU planner and executor.
//
// The reference's fixed-mode selector (selector/selector.c:509-789) walks a
// gate list -- pow2-iterative, four-step, batched CT-L1 direct, batched,
// N-D, Bluestein, direct, CT -- and builds a tree of CPU solvers.  On MI355X
// the same decisions collapse into a few shapes of LDS pass:
//
//   axis length n with all prime factors <= 13 and n <= single-pass limit
//       -> one pass along that axis (Stockham stages in LDS)
//   1-D n above the limit
//       -> four-step over p = 2 or 3 factors: column passes with the inter-pass
//          twiddle fused into their store (pow2_fourstep_solver_dft.c:700-763,
//          fused_twiddle_transpose_c.c:20-110), then a row pass whose store is
//          the transpose
//   axis length with a prime factor > 13
//       -> one fused Bluestein pass (bluestein_solver_dft.c:137-234)
//   R2C / C2R with even innermost n
//       -> real-packed pass with recombine / separate fused
//          (packed_solver_rdft.c:154-186)
//   N-D -> one pass per axis (ndim_solver_dft.c:96-121), batch = line axes.
#include "plan.h"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <sstream>
#include <thread>
#include <atomic>

namespace fftz {

// ---------------------------------------------------------------------------
// Device info
// ---------------------------------------------------------------------------
const DeviceInfo& device_info()
{
    static DeviceInfo info;
    static std::once_flag once;
    std::call_once(once, [] {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) return;
        hipDeviceProp_t prop;
        if (hipGetDeviceProperties(&prop, dev) != hipSuccess) return;
        info.cus = prop.multiProcessorCount;
        info.lds_per_block = prop.sharedMemPerBlock;
        info.warp = prop.warpSize;
        // Allow every kernel to use the full LDS of a workgroup.
        for (int prec : {4, 8})
            for (int rad : {kRadPow2, kRadAll, kRadLight, kRadTo8})
                for (KernelKind k : {KernelKind::Pass, KernelKind::Real, KernelKind::RealWide, KernelKind::Bluestein})
                    for (bool nt : {false, true})
                        for (int t : {256, 1024})
                            if (const void* f = kernel_symbol(k, prec, rad, nt, t))
                                (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                          (int)info.lds_per_block);
        for (int prec : {4, 8})
            for (int L = 64; L <= 4096; L *= 2)
                for (int t : {256, 512})
                    for (bool split : {false, true})
                        for (bool nt : {false, true})
                            if (const void* f = kernel_symbol_fixed(prec, L, t, split, nt))
                                (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                          (int)info.lds_per_block);
        for (int m : {kMfmaF32, kMfmaBf16x3, kMfmaF16x2})
            for (int L : {256, 4096})
                for (int nb : {2, 4})
                    (void)hipFuncSetAttribute(kernel_symbol_mfma(m, L, nb), hipFuncAttributeMaxDynamicSharedMemorySize,
                                              (int)info.lds_per_block);
    });
    return info;
}

// ---------------------------------------------------------------------------
// Roots of unity in double: exp(-2 pi i p / n), exact integer reduction and a
// fold onto [0, pi/4] before sin/cos.
// ---------------------------------------------------------------------------
struct d2 {
    double x, y;
};

// exp(-i theta) from u = (cos, sin) of theta's distance to the even end of its octant.
static d2 unfold(int64_t oct, d2 u)
{
    double ct, st;  // cos, sin of theta
    switch (oct) {
        case 0: ct = u.x; st = u.y; break;
        case 1: ct = u.y; st = u.x; break;
        case 2: ct = -u.y; st = u.x; break;
        case 3: ct = -u.x; st = u.y; break;
        case 4: ct = -u.x; st = -u.y; break;
        case 5: ct = -u.y; st = -u.x; break;
        case 6: ct = u.y; st = -u.x; break;
        default: ct = u.x; st = -u.y; break;
    }
    return {ct, -st};
}

static d2 root_fwd(int64_t p, int64_t n)
{
    p %= n;
    if (p < 0) p += n;
    // theta = (pi/4)(oct + rem/n), octant 0..7; below 2^60 in 64 bits.  The folded
    // angle counts from the octant's end in odd octants, so it stays <= pi/4.
    const bool narrow = n < ((int64_t)1 << 60);
    const int64_t oct = narrow ? 8 * p / n : (int64_t)((__int128)p * 8 / n);
    const int64_t rem = narrow ? 8 * p - oct * n : (int64_t)((__int128)p * 8 - (__int128)oct * n);
    const double a = (M_PI / 4.0) * ((double)(oct & 1 ? n - rem : rem) / (double)n);
    return unfold(oct, {cos(a), sin(a)});
}

// The n-th roots, root_fwd's values bit for bit.  Where 4 divides n the folded
// angles of all octants are those of the first, so only its n / 8 cosines and
// sines are computed.
class RootTable {
    const int64_t n_;
    std::vector<d2> u_;

public:
    explicit RootTable(int64_t n) : n_(n)
    {
        if (n % 4) return;
        u_.resize((size_t)(n / 8 + 1));
        for (int64_t p = 0; 8 * p <= n; p++) {
            const double a = (M_PI / 4.0) * ((double)(8 * p) / (double)n);
            u_[(size_t)p] = {cos(a), sin(a)};
        }
    }
    d2 operator()(int64_t p) const  // 0 <= p < n
    {
        if (u_.empty()) return root_fwd(p, n_);
        const int64_t oct = 8 * p / n_, q = n_ / 4;
        return unfold(oct, u_[(size_t)(oct & 1 ? (oct + 1) / 2 * q - p : p - oct / 2 * q)]);
    }
};

// ---------------------------------------------------------------------------
// Host FP64 FFT (recursive mixed radix) used only at setup, for the Bluestein
// spectrum table.  The roots of the top-level length are tabulated once
// (root_fwd, exact integer reduction); a sub-transform of length m reads
// root(j, m) as tab[j * (n / m)], which is the same double as root_fwd(j, m)
// (both reduce to the same correctly rounded fraction of the circle).
// ---------------------------------------------------------------------------
static void host_fft_rec(int64_t n, const d2* in, int64_t is, d2* out, const d2* tab, int64_t tstride)
{
    if (n == 1) { out[0] = in[0]; return; }
    int64_t r = 0;
    for (int64_t c : {4, 2, 3, 5, 7, 11, 13})
        if (n % c == 0) { r = c; break; }
    if (r == 0) {
        for (int64_t k = 0; k < n; k++) {
            d2 s = {0, 0};
            for (int64_t j = 0; j < n; j++) {
                const d2 w = tab[((j * k) % n) * tstride];
                const d2 x = in[j * is];
                s.x += x.x * w.x - x.y * w.y;
                s.y += x.x * w.y + x.y * w.x;
            }
            out[k] = s;
        }
        return;
    }
    const int64_t m = n / r;
    std::vector<d2> y((size_t)n);
    for (int64_t q = 0; q < r; q++) host_fft_rec(m, in + q * is, is * r, y.data() + q * m, tab, tstride * r);
    for (int64_t k1 = 0; k1 < m; k1++)
        for (int64_t k2 = 0; k2 < r; k2++) {
            d2 s = {0, 0};
            for (int64_t q = 0; q < r; q++) {
                const d2 w = tab[((q * (k1 + m * k2)) % n) * tstride];
                const d2 x = y[(size_t)(q * m + k1)];
                s.x += x.x * w.x - x.y * w.y;
                s.y += x.x * w.y + x.y * w.x;
            }
            out[k1 + m * k2] = s;
        }
}

static void host_fft(int64_t n, const d2* in, d2* out)
{
    std::vector<d2> tab((size_t)n);
    for (int64_t j = 0; j < n; j++) tab[(size_t)j] = root_fwd(j, n);
    host_fft_rec(n, in, 1, out, tab.data(), 1);
}

// ---------------------------------------------------------------------------
// Factorisation helpers
// ---------------------------------------------------------------------------
static const int kRadices[] = {16, 13, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2};

static bool smooth13(int64_t n)
{
    for (int64_t p : {2, 3, 5, 7, 11, 13})
        while (n % p == 0) n /= p;
    return n == 1;
}

// n as exactly S radices, the largest possible one first at each step.
static bool pick_radices(int n, int S, std::vector<int>& out)
{
    if (S == 0) return n == 1;
    for (int r : kRadices) {
        if (n % r) continue;
        int64_t most = 1;  // S - 1 radices reach at most 16^(S - 1)
        for (int s = 1; s < S; s++) most *= kRadices[0];
        if (n / r > most) continue;
        out.push_back(r);
        if (pick_radices(n / r, S - 1, out)) return true;
        out.pop_back();
    }
    return false;
}

// Fewest radix stages from kRadices (largest first on ties).
static bool factor_radices(int L, std::vector<int>& out)
{
    out.clear();
    if (L == 1) return true;
    if (!smooth13(L)) return false;
    for (int S = 1; !pick_radices(L, S, out); S++) {}
    std::sort(out.begin(), out.end(), std::greater<int>());
    // A radix-2 stage costs nearly as much LDS traffic and addressing as any
    // other: 16 16 16 2 becomes 16 16 8 4 (lines of 8192 points).  The lengths of
    // the fixed kernels keep their plan.
    if (out.size() >= 3 && out.back() == 2 && !((L & (L - 1)) == 0 && L <= 4096)) {
        std::vector<int> r = out;
        const size_t S = r.size();
        for (size_t i = 0; i + 1 < S && r[S - 1] == 2; i++)
            for (int f : {4, 3})
                if (r[S - 1] == 2 && r[i] % f == 0 && r[i] / f >= 3) {
                    r[i] /= f;
                    r[S - 1] *= f;
                }
        std::sort(r.begin(), r.end(), std::greater<int>());
        if (std::all_of(r.begin(), r.end(), [](int v) {
                return std::find(std::begin(kRadices), std::end(kRadices), v) != std::end(kRadices);
            }))
            out = r;
    }
    return (int)out.size() <= kMaxStages;
}

// A radix order the kernels can run: stages from kRadices whose product is L.
static bool radix_order_ok(int L, const std::vector<int>& r)
{
    if (r.empty() || (int)r.size() > kMaxStages) return false;
    int64_t prod = 1;
    for (int v : r) {
        if (std::find(std::begin(kRadices), std::end(kRadices), v) == std::end(kRadices)) return false;
        prod *= v;
    }
    return prod == L;
}

std::vector<std::vector<int>> radix_orders(int L, int maxn)
{
    // Multisets of radices with product L and at most one stage more than
    // the fewest; each in descending and ascending order.  The default order
    // (factor_radices) comes first.
    std::vector<std::vector<int>> out;
    std::vector<int> dflt;
    if (!factor_radices(L, dflt) || dflt.size() < 2) return out;
    out.push_back(dflt);
    const size_t smax = dflt.size() + 1;
    std::vector<std::vector<int>> sets;
    std::vector<int> cur;
    std::function<void(int64_t, size_t)> rec = [&](int64_t n, size_t from) {
        if (n == 1) {
            if (cur.size() >= 2) sets.push_back(cur);
            return;
        }
        if (cur.size() >= smax) return;
        for (size_t i = from; i < sizeof(kRadices) / sizeof(kRadices[0]); i++) {
            const int r = kRadices[i];
            if (n % r) continue;
            cur.push_back(r);
            rec(n / r, i);
            cur.pop_back();
        }
    };
    rec(L, 0);
    std::stable_sort(sets.begin(), sets.end(),
                     [](const std::vector<int>& a, const std::vector<int>& b) { return a.size() < b.size(); });
    for (const auto& m : sets) {
        std::vector<int> d = m, a = m;
        std::sort(d.begin(), d.end(), std::greater<int>());
        std::sort(a.begin(), a.end());
        for (const auto& o : {d, a})
            if ((int)out.size() < maxn && std::find(out.begin(), out.end(), o) == out.end()) out.push_back(o);
    }
    return out;
}

static int env_int(const char* name, int dflt)
{
    const char* v = getenv(name);
    return v ? atoi(v) : dflt;
}

static double radix_stage_cost(int r);

// Radices of a real-packed pass: the smallest goes to the stage that holds
// mirrored butterfly pairs (last for R2C, first for C2R).  Pairs above radix 10
// would double the kernel's VGPRs, so where the default plan has no smaller
// radix (16 x 16, 16 x 12, ...) the least-cost order that has one, with one
// more stage, is taken; products of 11s and 13s have none.
static std::vector<int> packed_radices(int L, std::vector<int> r, bool c2r)
{
    auto least = [](const std::vector<int>& o) { return *std::min_element(o.begin(), o.end()); };
    if (!r.empty() && least(r) > 10) {
        std::vector<std::vector<int>> sets = radix_orders(L, 1 << 20);
        if (L == 16) sets = {{8, 2}, {4, 4}};
        if (L == 12) sets = {{6, 2}, {4, 3}};
        double best = 1e300;
        for (auto& o : sets) {
            if (least(o) > 10) continue;
            double c = 0.0;
            for (int v : o) c += radix_stage_cost(v);
            if (c < best) {
                best = c;
                r = o;
            }
        }
    }
    std::sort(r.begin(), r.end());
    if (!c2r) std::reverse(r.begin(), r.end());
    return r;
}

static int next_pow2(int64_t v)
{
    int p = 1;
    while (p < v) p <<= 1;
    return p;
}

static int ilog2(int v)
{
    int l = 0;
    while ((1 << l) < v) l++;
    return l;
}

// ---------------------------------------------------------------------------
// Tables
// ---------------------------------------------------------------------------
struct TableBuilder {
    std::vector<unsigned char>& buf;
    int64_t add(const void* data, size_t bytes)
    {
        size_t off = (buf.size() + 255) & ~(size_t)255;
        buf.resize(off + bytes);
        memcpy(buf.data() + off, data, bytes);
        return (int64_t)off;
    }
    int64_t add_complex(const std::vector<d2>& v, int prec)
    {
        if (prec == 8) return add(v.data(), v.size() * sizeof(d2));
        std::vector<float> f(v.size() * 2);
        for (size_t i = 0; i < v.size(); i++) {
            f[2 * i] = (float)v[i].x;
            f[2 * i + 1] = (float)v[i].y;
        }
        return add(f.data(), f.size() * sizeof(float));
    }
};

// Stage twiddles of the fixed-length kernels: per stage, for c < ls, i in
// [1, R): w_{R ls}^{i c} -- the per-column layout of core/common/twiddle.c:46-66.
static int64_t stage_twiddles(TableBuilder& tb, int prec, const std::vector<int>& radix, int* twoff)
{
    std::vector<d2> tw;
    int ls = 1;
    for (size_t s = 0; s < radix.size(); s++) {
        const int R = radix[s];
        twoff[s] = (int)tw.size();
        const RootTable root((int64_t)R * ls);
        for (int c = 0; c < ls; c++)
            for (int i = 1; i < R; i++) tw.push_back(root((int64_t)i * c));
        ls *= R;
    }
    if (tw.empty()) tw.push_back({1.0, 0.0});
    return tb.add_complex(tw, prec);
}

// Threads per line of a generic pass: a power of two in [mint, maxt].  A stage
// runs ceil(nbl / TL) rounds of TL butterflies and lanes idle in its last one;
// the work of a choice is the sum over stages of rounds x TL x R x (cost per
// element).
//   * Wide enough that neighbouring lanes cover 64 bytes of a line, and a
//     column tile fills a wavefront (mint).
//   * At most 16 elements per thread where maxt allows it: beyond that too few
//     wavefronts fit next to the lines' LDS (1,000,000-point complex64, passes
//     of 100: 12 per thread 97 us, 25 per thread 104 us; 100 x 120 x 144
//     complex128 grid, 12 and 16 per thread 84.7 us, 25 to 32 per thread 87.1
//     us).  Column passes allow 20 before they double maxt, complex128 rows stop
//     at 256 threads where that keeps two workgroups on a CU (build_pass).
//   * Among the widths within 8% of the least work, short lines take the
//     narrowest (room for more lines) and long ones and pair stages the widest
//     (more loads in flight per line).
//   * Where the lines are too few for eight wavefronts per CU (two in
//     complex128), wider, up to 1.6 times the least
//     work: the launch is latency-bound.
// lines: how many there are; pair: the stage whose threads take two
// butterflies at a time, or -1.
static int line_threads(const std::vector<int>& radix, int L, int mint, int maxt, int pair, int64_t lines, int prec)
{
    int widest = 1;
    for (int r : radix) widest = std::max(widest, next_pow2(L / r));
    widest = std::min(widest, maxt);
    auto work = [&](int tl) {
        double w = 0.0;
        for (int s = 0; s < (int)radix.size(); s++) {
            const int r = radix[(size_t)s], per = s == pair ? 2 : 1;
            const int items = (L / r + per - 1) / per;
            w += (double)((items + tl - 1) / tl) * tl * per * r * radix_stage_cost(r);
        }
        return w;
    };
    int first = 1;
    while (first < widest && (first * 16 < L || first < mint)) first *= 2;
    double least = 1e300;
    for (int tl = first; tl <= widest; tl *= 2) least = std::min(least, work(tl));
    int tl = first;
    while (work(tl) > 1.08 * least) tl *= 2;
    if (L >= 1024 || pair >= 0) {
        tl = widest;
        while (work(tl) > 1.08 * least) tl /= 2;
    }
    const int64_t fill = 64 * (prec == 4 ? 2048 : 512);
    while (tl < widest && lines * tl < fill && work(tl * 2) <= 1.6 * least) tl *= 2;
    return tl;
}

// LDS layout, stage geometry and twiddles of a generic pass (kernels_body.h)
// of length L = product of radix, TL threads per line: fills the stage
// fields and the pitch LP of d (at least lp_min, odd, the padding within
// lp_max) and returns the table's offset.  Row k >= 1, column m of stage s: w_{Rs As}^{k m}, As = the product
// of the later radices.
//
// lst[0] is padded: consecutive lanes of the middle and last stages hold
// consecutive values of digit 0, which would otherwise sit a multiple of the
// later radices apart and meet in the same LDS banks.  The pad is the
// one of 0..7 with the fewest bank conflicts over the first wavefront's
// accesses of those stages (16 8-byte or 8 16-byte lanes per LDS cycle, banks
// of 128 bytes in all), the smallest on ties.
static int64_t digit_layout(TableBuilder& tb, int prec, const std::vector<int>& radix, int L, int TL, int lp_min,
                            int lp_max, PassDesc& d)
{
    const int S = (int)radix.size();
    d.nst = S;
    std::vector<d2> tw;
    int A = L;
    for (int s = 0; s < S; s++) {
        const int R = radix[(size_t)s];
        d.radix[s] = d.st[s].radix = R;
        d.st[s].nbl = L / R;
        A /= R;
        d.st[s].lst = A;
        d.st[s].mdiv = make_smalldiv((uint32_t)A);
        d.st[s].rdiv = make_smalldiv((uint32_t)R);
        d.st[s].twoff = (int)tw.size();
        if (s + 1 < S) {
            const RootTable root((int64_t)R * A);
            for (int k = 1; k < R; k++)
                for (int m = 0; m < A; m++) tw.push_back(root((int64_t)k * m));
        }
    }
    int LP = std::max(lp_min, L);
    if (S >= 2) {
        const int lanes = prec == 4 ? 16 : 8;  // lanes (and banks, in elements) per LDS cycle
        const int A0 = d.st[0].lst;
        // position of lane l in stage s: dig0 (A0 + pad) + rest + line pitch
        std::vector<int> dig0((size_t)(64 * S), -1), rest((size_t)(64 * S), 0);
        const int per = std::min(TL, 64);
        for (int s = 1; s < S; s++)
            for (int l = 0; l < 64; l++) {
                const int j = l % per, k = s * 64 + l;
                if (j >= d.st[s].nbl) continue;
                dig0[(size_t)k] = j % radix[0];
                int rem = j / radix[0];
                if (s + 1 < S) {
                    const int o = rem / d.st[s].lst;
                    rest[(size_t)k] = o * radix[(size_t)s] * d.st[s].lst + rem % d.st[s].lst;
                    continue;
                }
                for (int i = 1; i + 2 < S; i++) {
                    rest[(size_t)k] += (rem % radix[(size_t)i]) * d.st[i].lst;
                    rem /= radix[(size_t)i];
                }
                if (S >= 3) {
                    rest[(size_t)k] += rem * d.st[S - 2].lst;
                } else {
                    dig0[(size_t)k] = j;
                }
            }
        int best = 0;
        long best_cost = -1;
        for (int pad = 0; pad < 8; pad++) {
            const int a0 = A0 + pad;
            if (pad && radix[0] * a0 > lp_max) break;
            const int pitch = std::max(lp_min, radix[0] * a0) | 1;
            long cost = 0;
            for (int s = 1; s < S; s++) {
                for (int l0 = 0; l0 < 64; l0 += lanes) {
                    int bank[16] = {}, worst = 0;
                    for (int l = l0; l < l0 + lanes; l++) {
                        const int k = s * 64 + l;
                        if (dig0[(size_t)k] < 0) continue;
                        const int pos = dig0[(size_t)k] * a0 + rest[(size_t)k] + l / per * pitch;
                        worst = std::max(worst, ++bank[pos & (lanes - 1)]);
                    }
                    // a middle stage reads and writes, the last only reads
                    cost += (long)worst * radix[(size_t)s] * (s + 1 == S ? 1 : 2);
                }
            }
            if (best_cost < 0 || cost < best_cost) {
                best_cost = cost;
                best = pad;
            }
        }
        d.st[0].lst = A0 + best;
        LP = std::max(LP, radix[0] * d.st[0].lst);
    }
    d.LP = LP | 1;
    if (tw.empty()) tw.push_back({1.0, 0.0});
    return tb.add_complex(tw, prec);
}

// Two-level FP64 table for w_N^p, p < N: lo[q] = w_N^q (q < 2^b), hi[h] = w_N^(h 2^b).
static int64_t fourstep_twiddles(TableBuilder& tb, int64_t N, int* lobits)
{
    int b = 0;
    while (((int64_t)1 << (2 * b)) < N) b++;
    const int64_t lo_n = (int64_t)1 << b;
    const int64_t hi_n = (N + lo_n - 1) / lo_n;
    std::vector<d2> t((size_t)(lo_n + hi_n));
    for (int64_t q = 0; q < lo_n; q++) t[(size_t)q] = root_fwd(q, N);
    for (int64_t h = 0; h < hi_n; h++) t[(size_t)(lo_n + h)] = root_fwd(h * lo_n, N);
    *lobits = b;
    return tb.add(t.data(), t.size() * sizeof(d2));
}

// ---------------------------------------------------------------------------
// Pass construction
// ---------------------------------------------------------------------------
struct LineAxis {
    int64_t n, is, os;
    // coefficients of this axis's index in the sequence index g of the
    // input / output side (multi-pass Bluestein products; 0 for batch axes)
    int64_t gi = 0, go = 0;
};

struct PassReq {
    KernelKind kind = KernelKind::Pass;
    int L = 1;                 // transform length (M for Bluestein)
    int nvalid_in = -1, nvalid_out = -1;
    int64_t ies = 1, oes = 1;
    std::vector<LineAxis> lines;
    uint32_t flags = 0;
    bool want_in_col = false, want_out_col = false;
    Role in_role = Role::In, out_role = Role::Out;
    int64_t tw4_n = 0;
    int64_t chirp_off = -1, spec_off = -1, rtw_off = -1;
    int extra_lds_elems = 0;   // C2R needs L+1 slots
    int64_t in_base = 0, out_base = 0;  // byte offsets added to the role pointers
    int64_t gie = 0, goe = 0;  // element coefficients of the sequence index (kChirpFlags)
    int64_t nchirp = 0;
};

// Merge line axes that form one dense run for both input and output.
static std::vector<LineAxis> merge_axes(std::vector<LineAxis> ax)
{
    ax.erase(std::remove_if(ax.begin(), ax.end(), [](const LineAxis& a) { return a.n == 1; }), ax.end());
    bool changed = true;
    while (changed && ax.size() > 1) {
        changed = false;
        for (size_t i = 0; i < ax.size() && !changed; i++)
            for (size_t j = 0; j < ax.size() && !changed; j++) {
                if (i == j) continue;
                if (ax[j].is == ax[i].is * ax[i].n && ax[j].os == ax[i].os * ax[i].n &&
                    ax[j].gi == ax[i].gi * ax[i].n && ax[j].go == ax[i].go * ax[i].n) {
                    ax[i].n *= ax[j].n;
                    ax.erase(ax.begin() + (long)j);
                    changed = true;
                }
            }
    }
    return ax;
}

// Round x to `bits` significant bits, round-to-nearest-even, with a floor
// on the quantum exponent (subnormal spacing): bf16 = (8, -133), fp16 = (11, -24).
static double round_sig(double x, int bits, int qmin)
{
    if (x == 0.0) return 0.0;
    int e = 0;
    (void)std::frexp(x, &e);  // |x| in [2^(e-1), 2^e)
    const int q = std::max(e - bits, qmin);
    return std::ldexp(std::nearbyint(std::ldexp(x, -q)), q);
}

// Per-lane DFT-16 operand fragments for the matrix-core pass.  The real
// 32 x 32 operator is A = [[Fr, -Fi], [Fi, Fr]] with F[k][j] = w_16^(jk)
// (forward); rows 0-15 ("top") produce Re Y, rows 16-31 ("bottom") Im Y;
// column k < 16 multiplies Re x[k], column 16 + k multiplies Im x[k].
// The kernel permutes K so that lane group g = l / 16 supplies, as its
// element t < 8, part t & 1 (re / im) of input row rho = 4 (t >> 1) + g.
// Lane l (output row r = l % 16), 32 floats:
//   kMfmaF32:  [0..7] top[r][K(g, t)], [8..15] bottom[r][K(g, t)];
//   split:     [0..7] hi(top), [8..15] lo(top), [16..23] hi(bottom),
//              [24..31] lo(bottom); hi = round(a), lo = round(a - hi) in bf16
//              (kMfmaBf16x3) or fp16 (kMfmaF16x2), stored as the exactly
//              representable float values.
static int64_t mfma_fragments(TableBuilder& tb, int mode)
{
    std::vector<float> f(64 * 32, 0.0f);
    auto A = [](int half, int r, int k) -> double {
        const d2 w = root_fwd((int64_t)r * (k & 15), 16);  // (Fr, Fi)
        const bool im = k >= 16;
        if (half == 0) return im ? -w.y : w.x;
        return im ? w.x : w.y;
    };
    const int bits = mode == kMfmaBf16x3 ? 8 : 11;
    const int qmin = mode == kMfmaBf16x3 ? -133 : -24;
    for (int l = 0; l < 64; l++) {
        const int r = l & 15, g = l >> 4;
        float* o = &f[(size_t)l * 32];
        auto kidx = [g](int t) { return 16 * (t & 1) + 4 * (t >> 1) + g; };
        if (mode == kMfmaF32) {
            for (int t = 0; t < 8; t++) {
                o[t] = (float)A(0, r, kidx(t));
                o[8 + t] = (float)A(1, r, kidx(t));
            }
            continue;
        }
        for (int t = 0; t < 8; t++)
            for (int half = 0; half < 2; half++) {
                const double a = A(half, r, kidx(t));
                const double hi = round_sig(a, bits, qmin);
                const double lo = round_sig(a - hi, bits, qmin);
                o[16 * half + t] = (float)hi;
                o[16 * half + 8 + t] = (float)lo;
            }
    }
    return tb.add(f.data(), f.size() * sizeof(float));
}

// Stage twiddles of the matrix-core pass in the order its lanes read them:
// for stage s >= 1 (ls = 16^s) and c = j mod ls, 16 entries [g][q] =
// w_{16 ls}^((4 q + g) c) -- lane group g's four inputs i = 4 q + g of
// butterfly j, entry i = 0 being 1 -- stage after stage (FP64 roots rounded
// to FP32).  A lane reads its four twiddles of a block as 32 contiguous bytes.
// With scaled fp16 operands the entries carry an exact factor 1/16, which
// keeps each stage's inputs inside the fp16 range (the kernel undoes it at
// the last store).
static int64_t mfma_stage_twiddles(TableBuilder& tb, int L, int mode)
{
    std::vector<d2> t;
    const int S = L == 256 ? 2 : 3;
    const double f = mode == kMfmaF16x2 ? 1.0 / 16.0 : 1.0;
    for (int s = 1, ls = 16; s < S; s++, ls *= 16)
        for (int c = 0; c < ls; c++)
            for (int g = 0; g < 4; g++)
                for (int q = 0; q < 4; q++) {
                    const d2 w = root_fwd((int64_t)(4 * q + g) * c, 16 * ls);
                    t.push_back({w.x * f, w.y * f});
                }
    return tb.add_complex(t, 4);
}

static bool build_pass(Plan* plan, TableBuilder& tb, const PassReq& q, std::string& err)
{
    const int prec = plan->spec.prec_bytes;
    const int esize = 2 * prec;
    const DeviceInfo& dev = device_info();
    Launch ln;
    ln.kind = q.kind;
    PassDesc& d = ln.d;
    d.L = q.L;
    d.nvalid_in = q.nvalid_in < 0 ? q.L : q.nvalid_in;
    d.nvalid_out = q.nvalid_out < 0 ? q.L : q.nvalid_out;
    d.ies = q.ies;
    d.oes = q.oes;
    d.flags = q.flags;
    d.scale_f = 1.0f;
    d.scale_d = 1.0;

    std::vector<int> radix;
    if (!factor_radices(q.L, radix)) {
        err = "length " + std::to_string(q.L) + " has no radix plan";
        return false;
    }
    // a tuned radix order for this length (plain passes; the matrix-core
    // pass needs the all-16 plan)
    const bool r2c = (q.flags & kR2CPost) != 0, c2r = (q.flags & kC2RPre) != 0;
    if (r2c || c2r) radix = packed_radices(q.L, radix, c2r);
    if (const std::vector<int>* tr = plan->spec.tune.radices(q.L))
        if (q.kind == KernelKind::Pass && plan->spec.mfma_mode == kMfmaNone && radix_order_ok(q.L, *tr)) radix = *tr;
    d.nst = (int)radix.size();
    // The narrowest radix set that holds the line's radices: its kernel has the
    // fewest registers.  All radices -> set, when the sets were made (kernel time,
    // of one build): complex128 100 x 120 x 144 grid 91 -> 85 us (kRadLight), 2048 x
    // 675 real batch of 4 214 -> 155 us (kRadTo8), 2894 lines of 1372 47.7 -> 41 us;
    // complex64 3001 lines of 1200 forward 14.9 -> 14.1 us.  A complex64 set of
    // radices up to 8 would save no wavefront worth having over kRadLight (78
    // against 92 VGPRs).
    const bool real = q.kind == KernelKind::Pass && (q.flags & kRealFlags);
    for (int set : {kRadAll, kRadPow2, kRadLight, kRadTo8}) {
        if ((set == kRadLight && real) || (set == kRadTo8 && prec == 4)) continue;
        const int pair = radix.empty() ? 1 : r2c ? radix.back() : c2r ? radix.front() : 1;  // one point: no stage
        bool fits = rad_in_pairs(set, pair);
        for (int r : radix) fits = fits && rad_in_set(set, r);
        if (fits || set == kRadAll) ln.rad = set;
    }
    for (size_t s = 0; s < radix.size(); s++) d.radix[s] = radix[s];
    // a tuned number of values per thread
    const int tuned_e = plan->spec.tune.elems ? plan->spec.tune.elems : env_int("FFTZ_E", 0);
    const int need = q.L + q.extra_lds_elems;

    // fixed-length kernel: power-of-two L in [64, 4096], plain C2C pass
    const bool pow2L = q.L >= 64 && q.L <= 4096 && (q.L & (q.L - 1)) == 0;
    if ((q.flags & kChirpFlags) && (q.kind != KernelKind::Pass || (q.flags & kRealFlags))) {
        err = "internal: Bluestein products on a real pass";
        return false;
    }
    const bool fixed_ok = q.kind == KernelKind::Pass && pow2L && tuned_e != 8 && d.nvalid_in == q.L &&
                          d.nvalid_out == q.L &&
                          !(q.flags & (kRealFlags | kChirpFlags)) && env_int("FFTZ_FIXED", 1);
    bool plan_match = fixed_ok;
    if (fixed_ok) {
        // the fixed kernels hard-code 16, 16, ..., 2^rem (kernels_fixed.hip)
        const int lg = ilog2(q.L), S = (lg + 3) / 4, rem = lg - 4 * (S - 1);
        plan_match = (int)radix.size() == S;
        for (int s = 0; plan_match && s < S; s++)
            plan_match = radix[s] == (s < S - 1 ? 16 : (1 << rem));
    }
    // fixed kernels come in 256- and 512-thread variants (512 for wide column
    // tiles of L >= 256)
    const int tbig = (prec == 4 ? 1024 : 512) / ((q.flags & kRealFlags) && q.kind == KernelKind::Pass ? 2 : 1);
    int tmax = plan_match ? (q.L >= 256 ? 512 : 256) : tbig;
    int64_t nl_total = 1;
    for (auto& a : q.lines) nl_total *= a.n;
    // A complex128 workgroup of 512 threads is the only one on a CU but for
    // kRadTo8 (three wavefronts per SIMD or fewer): 256 threads for rows where the
    // LDS holds two tiles and the lines are more than the CUs (261 lines of 4004
    // 18.9 -> 14.5 us, 1024 of 4095 43.5 -> 35.9; 256 of 4095 the reverse, 13.2
    // and 14.4).  Columns have their own limit below.
    if (!plan_match && prec == 8 && ln.rad != kRadTo8 && nl_total > dev.cus && !q.want_in_col && !q.want_out_col &&
        tuned_e != 8 && tuned_e != 16 && 2 * (size_t)lds_pad(need) * esize <= dev.lds_per_block)
        tmax = std::min(tmax, 256);
    // threads per line, and the table and layout that go with the kernel
    int TL;
    bool few = false;  // few lines for column tiles
    if (plan_match) {
        TL = q.L / 16;
        ln.E = 16;
        ln.stw_off = stage_twiddles(tb, prec, radix, d.twoff);
        d.LP = (lds_pad(need - 1) + 1) | 1;
    } else {
        // column tiles: at most 64 threads per line (32 in complex128) while that
        // leaves 20 elements per thread, see the tile's limit below -- but not
        // where the lines are too few for one such tile's threads on every CU
        // (complex64, 64 or 128 threads against none of these limits: 8 lines of
        // 2800 12.7 -> 9.4 us, 514 of 1125 11.2 -> 9.5, 300 of 2800 15.0 -> 13.1)
        const bool cols = q.want_in_col || q.want_out_col;
        int most = cols ? 256 / prec : tmax;
        while (most < tmax && q.L > 20 * most) most *= 2;
        few = cols && nl_total * most < (int64_t)dev.cus * (2048 / prec);
        if (few) most = tmax;
        TL = line_threads(radix, q.L, cols ? 4 : 64 / esize, most,
                          r2c ? (int)radix.size() - 1 : c2r ? 0 : -1, nl_total, prec);
        if (tuned_e == 8 || tuned_e == 16) TL = std::min(next_pow2((q.L + tuned_e - 1) / tuned_e), tmax);
        ln.E = std::max(tuned_e == 8 || tuned_e == 16 ? tuned_e : 1, (q.L + TL - 1) / TL);
        ln.stw_off = digit_layout(tb, prec, radix, q.L, TL, lds_pad(need - 1) + 1,
                                 std::max(lds_pad(need - 1) + 1, q.L + 16), d);
    }
    const int LP = d.LP;
    d.TL = TL;
    d.tl_shift = ilog2(TL);
    // matrix-core pass: complex64, L = 16^2 or 16^3 with the plain 16-radix
    // plan, row mapping, no fused twiddle / real-packed step
    const int mm = plan->spec.mfma_mode;
    const bool use_mfma = mm != kMfmaNone && prec == 4 && plan_match && (q.L == 256 || q.L == 4096) &&
                          !q.want_in_col && !q.want_out_col &&
                          !(q.flags & (kTw4 | kRealFlags | kChirpFlags));

    // line axes: choose l0
    std::vector<LineAxis> ax = merge_axes(q.lines);
    if (ax.empty()) ax.push_back({1, 0, 0});
    size_t i0 = 0;
    bool in_col = false, out_col = false;
    if (q.want_in_col || q.want_out_col) {
        for (size_t i = 0; i < ax.size(); i++) {
            if ((q.want_in_col && ax[i].is == 1) || (!q.want_in_col && q.want_out_col && ax[i].os == 1)) {
                i0 = i;
                break;
            }
        }
    } else {
        for (size_t i = 1; i < ax.size(); i++)
            if (std::llabs(ax[i].is) < std::llabs(ax[i0].is)) i0 = i;
    }
    std::swap(ax[0], ax[i0]);
    // remaining axes sorted by input stride so l1 is the inner one
    std::sort(ax.begin() + 1, ax.end(), [](const LineAxis& a, const LineAxis& b) { return a.is < b.is; });
    int64_t n0 = ax[0].n;
    in_col = q.want_in_col && ax[0].is == 1 && q.ies != 1;
    out_col = q.want_out_col && ax[0].os == 1 && q.oes != 1;

    // lines per tile
    const size_t lds_cap = dev.lds_per_block;
    const size_t line_bytes = (size_t)LP * esize;
    if (line_bytes > lds_cap) {
        err = "pass length " + std::to_string(q.L) + " exceeds LDS";
        return false;
    }
    int C = 1;
    if (use_mfma) {
        in_col = out_col = false;
        C = q.L == 4096 ? 1 : 16;  // 16 column blocks of 16 butterflies per tile
        TL = 16;
        d.TL = TL;
        d.tl_shift = 4;
    } else if (in_col || out_col) {
        const int cmax = plan->spec.tune.col_c ? plan->spec.tune.col_c : env_int("FFTZ_COL_C", prec == 8 ? 16 : 32);
        const size_t budget = std::min(lds_cap, (size_t)env_int("FFTZ_COL_LDS", 96 * 1024));
        // Generic kernels: two workgroups per CU at their register counts, i.e.
        // 512 threads (256 in complex128), so that one loads while the other
        // computes: 1080-point columns of 961 x 13 images, 8 lines of 128
        // threads 78 us, of 64 threads 63 us; complex128 600-point columns, 8
        // lines of 64 threads 48 us, of 32 threads 38 us.
        // Not where the lines are few, nor where it would leave one line, read
        // at element stride (350 complex128 columns of 2800 33.6 -> 17.6 us), nor
        // two complex128 lines where the LDS holds one tile of four per CU and
        // fours leave few lines idle (1000 columns of 1300 24.7 -> 17.7 us, but 135
        // images of 10 columns of 1372 21.6 -> 28.1; complex64 loses: 984 columns
        // of 2800 25.8 -> 32.4).
        const int tcap = plan_match || few ? tmax : std::min(tmax, 2048 / prec);
        // a row of n0 lines that C does not divide is tiled raggedly (the
        // last tile of each row partly idle) rather than falling back to
        // element-strided row tiles
        const bool four = prec == 8 && 8 * line_bytes > lds_cap && (n0 + 3) / 4 * 4 <= n0 + n0 / 16;
        while (C * 2 <= cmax && (size_t)(C * 2) * line_bytes <= budget && C * 2 <= n0 &&
               C * 2 * TL <= (C == 1 || (C == 2 && four) ? tmax : tcap))
            C *= 2;
        // complex128 tiles of the fixed kernels take the whole LDS from 1024
        // points on: columns of 8 lines 35 us, of 4 lines 40 us (64 MiB each
        // way).  That is one tile per CU instead of two.  On rows that start on
        // cache lines it wins at any count (64 columns of 2048 points x 4: 10.9
        // us, 14.2 without); on others where it adds neither a round of tiles (20
        // images of 100 columns of 1024: 24 us, 15 without) nor idle lines (146 of 41:
        // 55 us, 45) and the narrower ones are more than the CUs (335 columns of
        // 2048: 13.6 us, 11.4).  4096 points have no narrower column tile.
        if (plan_match && prec == 8 && q.L >= 1024 && C * 2 <= cmax && (size_t)(C * 2) * line_bytes <= lds_cap &&
            C * 2 <= n0 && C * 2 * TL <= tmax) {
            const bool aligned = (!in_col || q.ies % 8 == 0) && (!out_col || q.oes % 8 == 0) && n0 % (C * 2) == 0;
            const int64_t rows = nl_total / n0, narrow = rows * ((n0 + C - 1) / C), wide = rows * ((n0 + C * 2 - 1) / (C * 2));
            const int64_t cus = dev.cus;
            if (C == 1 || aligned || plan->spec.tune.col_c || (narrow > cus && wide * 2 <= narrow + narrow / 32 &&
                                     (wide + cus - 1) / cus <= (narrow + 2 * cus - 1) / (2 * cus)))
                C *= 2;
        }
        // fewer than two tiles per CU: narrower ones, down to 16 lines (128- or
        // 256-byte segments); fewer than one for two CUs: down to four lines; long
        // lines, fewer than one for four: two (complex64: 40 lines of 2187 12.0 ->
        // 9.6 us, of 2000 10.9 -> 9.2; 130 complex128 lines of 144 5.6 -> 6.1).
        // Fixed kernels keep a whole wavefront (48 complex128 lines of 64 5.1 us as
        // 16 threads, 4.7 as 64).
        while (!plan->spec.tune.col_c && !(plan_match && C * TL <= 64) &&
               ((C > 16 && nl_total / C < 2 * dev.cus) || (C > 4 && nl_total / C < dev.cus / 2) ||
                (C > 2 && q.L >= 1024 && nl_total / C < dev.cus / 4)))
            C /= 2;
        if (C < 2) { in_col = false; out_col = false; C = 1; }
    }
    if (!(in_col || out_col) && !use_mfma) {
        const int tgt = plan->spec.tune.row_t ? plan->spec.tune.row_t : env_int("FFTZ_ROW_T", 256);
        const size_t budget = std::min(lds_cap, (size_t)env_int("FFTZ_ROW_LDS", plan_match ? 64 * 1024 : 40 * 1024));
        // lines per tile: up to tgt threads; beyond a wavefront only while
        // every CU keeps two tiles
        while (C * TL < tgt && (size_t)(C * 2) * line_bytes <= budget && C * 2 * TL <= tmax && C < nl_total &&
               (C * TL < 64 || nl_total / (C * 2) >= 2 * dev.cus || plan->spec.tune.row_t))
            C *= 2;
    }
    if (C * TL > 1024) {
        err = "tile too large";
        return false;
    }
    d.C = C;
    d.c_shift = ilog2(C);
    if (in_col) d.flags |= kInCol;
    if (out_col) d.flags |= kOutCol;

    // line levels: l0, l1, l2 (+ host-looped outer axes)
    std::vector<LineAxis> host_axes;
    while (ax.size() > 3) {
        host_axes.push_back(ax.back());
        ax.pop_back();
    }
    while (ax.size() < 3) ax.push_back({1, 0, 0});
    int64_t nl = ax[0].n * ax[1].n * ax[2].n;
    if (nl >= ((int64_t)1 << 31)) {
        err = "too many lines in one pass";
        return false;
    }
    d.nlines = nl;
    d.ln0 = make_fastdiv((uint32_t)ax[0].n);
    d.ln1 = make_fastdiv((uint32_t)ax[1].n);
    for (int k = 0; k < 3; k++) {
        d.ils[k] = ax[k].is;
        d.ols[k] = ax[k].os;
        d.gin[k] = ax[k].gi;
        d.gout[k] = ax[k].go;
    }
    d.gin[3] = q.gie;
    d.gout[3] = q.goe;
    d.nchirp = q.nchirp;
    if (q.flags & kTw4) {
        d.tw4_n = q.tw4_n;
        ln.tw4_off = fourstep_twiddles(tb, q.tw4_n, &d.tw4_lobits);
    }
    ln.chirp_off = q.chirp_off;
    ln.spec_off = q.spec_off;
    ln.rtw_off = q.rtw_off;
    ln.in_role = q.in_role;
    ln.out_role = q.out_role;
    ln.block = (uint32_t)(C * TL);
    ln.fixed = plan_match && ln.block <= 512 && !use_mfma;
    ln.maxt = ln.block <= 256 ? 256 : (ln.fixed ? 512 : 1024);
    if (use_mfma) {
        ln.mfma = mm;
        ln.mfma_nb = env_int("FFTZ_MFMA_NB", 4) == 2 ? 2 : 4;
        ln.block = (uint32_t)(1024 / ln.mfma_nb);
        ln.frag_off = mfma_fragments(tb, mm);
        ln.rtw_off = mfma_stage_twiddles(tb, q.L, mm);  // the pass's d.rtw: see kernels_mfma.hip
    }
    int64_t tiles = (nl + C - 1) / C;
    if ((in_col || out_col) && n0 % C != 0) {
        // ragged rows: ceil(n0 / C) tiles per row of n0 lines
        const int64_t tpr = (n0 + C - 1) / C;
        tiles = tpr * (nl / n0);
        if (tiles * C >= ((int64_t)1 << 31)) {
            err = "too many lines in one pass";
            return false;
        }
        d.vrow = make_fastdiv((uint32_t)(tpr * C));
    }
    ln.grid = (uint32_t)tiles;
    ln.lds_bytes = (uint32_t)((size_t)C * line_bytes);
    // Column exchanges in halves, where the LDS rather than the registers limits
    // the workgroups of a CU and more tiles wait than the two that the whole
    // exchange holds.  By what it measured (whole -> halves):
    //   * complex128, 256 points: 64 MiB 24.2 -> 22.5 us, ragged 32 MiB 16.2 ->
    //     14.1, 128 MiB 43.5 -> 40.0; 2^24 points in three passes 277 -> 271.  Not
    //     beyond the Infinity Cache, where more lines in flight than it holds
    //     cost: aligned rows from 512 MiB on 192 -> 204, others from 256 MiB 107 -> 120.
    //   * complex64, 512 points, the reverse: 64 MiB 28.4 -> 30.5, 256 MiB 119.4
    //     -> 116.8, 512 x 512 x 512 real in all 710 -> 694; short rows always lose
    //     (64 lines, 256 MiB 114 -> 120).
    //   * complex64, 256 and 1024 points: 64 MiB 23.3 -> 23.4 and 33.1 -> 35.5 us,
    //     no kernel; complex128, 512 points would gain from 64 to 128 MiB (52.9 -> 47.5).
    if (ln.fixed && (in_col || out_col) && tiles > 2 * dev.cus) {
        const int64_t mib = (nl * q.L * esize) >> 20;
        const bool aligned = n0 % C == 0 && (!in_col || (q.ies * esize) % 128 == 0) && (!out_col || (q.oes * esize) % 128 == 0);
        if (prec == 8)
            ln.split = q.L == 256 && ln.maxt == 256 && mib <= (aligned ? 256 : 128);
        else
            ln.split = q.L == 512 && ln.maxt == 512 && mib >= 256 && n0 > 4 * C;
    }
    if (use_mfma) ln.lds_bytes += 64;  // per-wavefront maxima of the fp16 line scale
    // XCD-contiguous tile order: measured to help passes that read rows and
    // store columns (the four-step's transposing last pass) and to cost ~5%
    // on passes that read columns
    // Also for column tiles whose segments straddle cache lines (an element
    // stride that is not a multiple of 128 bytes, e.g. the 257-wide
    // half-complex rows of a 3-D R2C): neighbouring tiles share those lines.
    const bool straddle = in_col && ((q.ies * esize) % 128) != 0;
    if (((out_col && !in_col) || straddle) && tiles >= 64 && env_int("FFTZ_XCD_REMAP", 1)) d.flags |= kXcdRemap;

    // Results in whole 128-byte lines may bypass the L2's write-back; those of
    // a pass whose output a later launch reads are put back by plan_create.
    // Lines of 4 KiB and more count as whole (one partial line in 32); one store
    // has to cover 128 bytes of a row (64-point complex64 lines, 32 bytes: 13 -> 19
    // us), 256 of a column tile (128: 512^3 R2C's last pass 231 -> 234 us) on
    // data beyond half of the Infinity Cache.
    // The next call may be another plan on this output, which it then finds in
    // the Infinity Cache less often.  Time with / without for rows of 256 to 6000
    // points: one plan alone; with a second plan reading its output; with that
    // one in place.
    //   output MiB                8      24      32      64      128     160     256
    //   fixed kernels alone     .97-1.0 .72-.80 .76-.84 .91-.94 .95-.97 .81-.90 .79-.87
    //     pair                  .95     .87-.96 .88-1.03 1.0-1.04 .95-.99 .84-.89 .94-.97
    //     pair, in place        1.0     .94-1.0 .95-1.07 1.0-1.02 1.0-1.04 1.0-1.07 1.0-1.06
    //   complex64 alone         .96-.99 .82-.92 .85-.93 .94-.97 .96-1.0 .70-.81 .69-.81
    //     pair                  .94-.98 .95-1.08 .97-1.12 1.0-1.13 .93-.98 .83-.90 .94-1.0
    //     pair, in place        .98-1.0 1.0-1.06 1.0-1.09 1.0-1.11 1.04-1.14 1.04-1.18 .96-1.0
    //   complex128 alone        .92-.98 .82-.97 .83-.93 .91-.95 .91-.97 .79-.89 .75-.87
    //     pair                  .93-.97 .88-.98 .94-1.03 .93-1.01 .91-.98 .84-.92 .89-.97
    //     pair, in place        .96-1.0 .94-1.0 .97-1.0 .95-1.02 .94-1.04 .94-1.06 .91-1.0
    // (generic kernels; Bluestein lines of either precision are as complex64.)
    // So complex64 generic and Bluestein rows keep to plain stores between 32
    // and 160 MiB, where a reader loses more than the plan gains.
    if (!(q.flags & kRealFlags) && q.out_role == Role::Out) {
        bool aligned = true;
        for (int k = out_col ? 1 : 0; k < 3; k++)
            if (ax[k].n > 1 && (ax[k].os * (int64_t)esize) % 128 != 0) aligned = false;
        const int64_t mib = (nl * d.nvalid_out * esize) >> 20;
        const bool reread = !plan_match && (prec == 4 || q.kind == KernelKind::Bluestein) && mib >= 32 && mib < 160;
        const bool rows = !out_col && q.oes == 1 && TL * esize >= 128 && !reread &&
                          (aligned || (int64_t)d.nvalid_out * esize >= 4096);
        const bool cols = out_col && aligned && (q.oes * esize) % 128 == 0 && C * esize >= 256 && n0 % C == 0 &&
                          nl * q.L * esize >= ((int64_t)128 << 20);
        if (rows || cols) d.flags |= kNtStore;
    }
    // expand host-looped axes
    std::vector<int64_t> ioffs{q.in_base}, ooffs{q.out_base}, gis{0}, gos{0};
    // real-side strides count real elements (packed R2C / C2R and the
    // full-length promoted / real-part forms alike)
    const int64_t in_scale = ((q.flags & (kRealIn | kRealPromote)) ? prec : esize);
    const int64_t out_scale = ((q.flags & (kRealOut | kRealPart)) ? prec : esize);
    for (auto& h : host_axes) {
        std::vector<int64_t> ni, no, ngi, ngo;
        for (size_t k = 0; k < ioffs.size(); k++)
            for (int64_t j = 0; j < h.n; j++) {
                ni.push_back(ioffs[k] + j * h.is * in_scale);
                no.push_back(ooffs[k] + j * h.os * out_scale);
                ngi.push_back(gis[k] + j * h.gi);
                ngo.push_back(gos[k] + j * h.go);
            }
        ioffs.swap(ni);
        ooffs.swap(no);
        gis.swap(ngi);
        gos.swap(ngo);
    }
    for (size_t k = 0; k < ioffs.size(); k++) {
        Launch l2 = ln;
        l2.in_off_bytes = ioffs[k];
        l2.out_off_bytes = ooffs[k];
        l2.d.gin_base = gis[k];
        l2.d.gout_base = gos[k];
        plan->launches.push_back(l2);
    }
    return true;
}

// ---------------------------------------------------------------------------
// Bluestein tables: chirp conj(B_k) (k < n) and spectrum conj(FFT_M(b)) / M.
// B_k = exp(+i pi (k^2 mod 2n) / n) (core/common/bluestein_utils.c:88-158).
// ---------------------------------------------------------------------------
static int64_t bluestein_length(int64_t n)
{
    for (int64_t m = 2 * n - 1;; m++)
        if (smooth13(m)) return m;
}

// Relative cost per element of one generic LDS stage of radix r: the in-register
// DFT-r (real operations per element of the codelet in codelets.h), the
// stage-twiddle product ((r - 1) / r complex products) and the addressing of one
// LDS read and write.  The last part was counted on self-sorting stages; the
// in-place ones take about a third less in all, much the same for every radix
// (74 instructions per element for 12 x 10 x 10 where this adds up to 77.5), so
// the order of the choices made by it stands.
static double radix_stage_cost(int r)
{
    switch (r) {
        case 2: return 17.5;
        case 3: return 19.5;
        case 4: return 19.5;
        case 5: return 22.0;
        case 6: return 22.5;
        case 7: return 25.0;
        case 8: return 22.0;
        case 9: return 26.0;
        case 10: return 25.5;
        case 11: return 29.0;
        case 12: return 26.5;
        case 13: return 31.0;
        default: return 25.0;  // 16
    }
}

// Extended length of a Bluestein transform that runs in one LDS tile.  Any
// 13-smooth M >= 2n - 1 gives the same transform; the reference takes the
// smallest (bluestein_length above, which the multi-pass form keeps).  In one
// tile the work is two M-point transforms through the LDS stages of M's
// fewest-stage radix plan, so this takes the M with the least
// M x sum(radix_stage_cost) among the 13-smooth lengths from the smallest up
// to the next power of two (the same thread count and tile class) and the
// tile limit.  E.g. n = 4099: 8232 = 12 7 7 7 2 becomes 8448 = 16 16 11 3.
// Lengths beyond the limit are returned as the smallest (the caller plans
// them multi-pass).
static double transform_stage_cost(int64_t m)
{
    std::vector<int> r;
    if (!smooth13(m) || !factor_radices((int)m, r)) return -1.0;
    double per = 0.0;
    for (int v : r) per += radix_stage_cost(v);
    return (double)m * per;
}

// transform_stage_cost of every length up to 16384 (-1 where there is no
// radix plan), built once per process
static const std::vector<double>& stage_cost_table()
{
    static std::vector<double> t;
    static std::once_flag once;
    std::call_once(once, [] {
        t.assign(16385, -1.0);
        for (int64_t m = 2; m <= 16384; m++) t[(size_t)m] = transform_stage_cost(m);
    });
    return t;
}

static int64_t bluestein_tile_length(int64_t n, int64_t limit)
{
    const int64_t m0 = bluestein_length(n);
    if (m0 > limit || !env_int("FFTZ_BLUESTEIN_COST", 1)) return m0;
    int64_t hi = 1;
    while (hi < m0) hi <<= 1;
    hi = std::min(hi, limit);
    const std::vector<double>& tab = stage_cost_table();
    int64_t best = m0;
    double best_cost = 0.0;
    for (int64_t m = m0; m <= hi; m++) {
        const double cost = m < (int64_t)tab.size() ? tab[(size_t)m] : transform_stage_cost(m);
        if (cost < 0.0) continue;
        if (m == m0 || cost < best_cost) {
            best = m;
            best_cost = cost;
        }
    }
    return best;
}

Plan* plan_create(const ProblemSpec& spec, std::string& err, bool dry_run);
hipError_t plan_enqueue(Plan* p, Slot* s, const void* in, void* out, hipStream_t stream);

// In-place FP64 forward FFT of v (13-smooth length) on the device, through a
// plan of this library: the spectrum table of a long Bluestein transform
// (M up to ~2^26), where the host recursion would take tens of seconds.
static bool device_fft_fp64(std::vector<d2>& v)
{
    ProblemSpec ss;
    ss.prec_bytes = 8;
    ss.type = FftType::C2C;
    ss.dir = 0;
    ss.inplace = true;
    ss.dims = {{(int64_t)v.size(), 1, 1}};
    std::string err;
    Plan* sub = plan_create(ss, err, false);
    if (!sub) return false;
    void* buf = nullptr;
    const size_t bytes = v.size() * sizeof(d2);
    bool ok = hipMalloc(&buf, bytes) == hipSuccess &&
              hipMemcpy(buf, v.data(), bytes, hipMemcpyHostToDevice) == hipSuccess;
    if (ok) {
        hipError_t e = hipSuccess;
        Slot* s = plan_acquire_slot(sub, &e);
        ok = s && plan_enqueue(sub, s, buf, buf, s->stream) == hipSuccess &&
             hipStreamSynchronize(s->stream) == hipSuccess;
        if (s) plan_release_slot(sub, s);
    }
    ok = ok && hipMemcpy(v.data(), buf, bytes, hipMemcpyDeviceToHost) == hipSuccess;
    if (buf) (void)hipFree(buf);
    plan_destroy(sub);
    return ok;
}

// dry_run: only the table sizes matter (no device, zero spectrum).
static void bluestein_tables(TableBuilder& tb, int prec, int64_t n, int64_t M, int64_t* chirp_off, int64_t* spec_off,
                             bool dry_run)
{
    // in one allocation with what follows (growing by doubling, the arena of a
    // long transform was copied and its pages touched twice: n = 500009 26 -> 12 ms)
    tb.buf.reserve(tb.buf.size() + (size_t)(n + M) * 2 * prec + (M > 32768 ? (size_t)1 << 20 : 4096));
    std::vector<d2> b((size_t)M, d2{0, 0});
    std::vector<d2> cb((size_t)n);
    for (int64_t k = 0; k < n; k++) {
        const int64_t sq = (int64_t)(((__int128)k * k) % (2 * n));
        d2 w = root_fwd(sq, 2 * n);  // exp(-i pi sq / n) = conj(B_k)
        cb[(size_t)k] = w;
        d2 bk = {w.x, -w.y};
        b[(size_t)k] = bk;
        if (k > 0) b[(size_t)(M - k)] = bk;
    }
    std::vector<d2> fb;
    if (dry_run) {
        fb.assign((size_t)M, d2{0, 0});
    } else if (M > (1 << 18) && device_fft_fp64(b)) {
        fb.swap(b);
    } else {
        fb.resize((size_t)M);
        host_fft(M, b.data(), fb.data());
    }
    const double inv = 1.0 / (double)M;
    for (auto& v : fb) v = {v.x * inv, -v.y * inv};
    *chirp_off = tb.add_complex(cb, prec);
    *spec_off = tb.add_complex(fb, prec);
}

// ---------------------------------------------------------------------------
// Plan construction
// ---------------------------------------------------------------------------
static int64_t single_pass_limit(int prec)
{
    return prec == 4 ? env_int("FFTZ_LMAX_F", 16384) : env_int("FFTZ_LMAX_D", 8192);
}

static int64_t extent(const std::vector<AxisSpec>& dims, const std::vector<AxisSpec>& vecs, bool use_in,
                      int64_t n0_override)
{
    int64_t e = 0;
    for (size_t i = 0; i < dims.size(); i++) {
        int64_t n = (i == 0 && n0_override > 0) ? n0_override : dims[i].n;
        e += (n - 1) * std::llabs(use_in ? dims[i].is : dims[i].os);
    }
    for (auto& v : vecs) e += (v.n - 1) * std::llabs(use_in ? v.is : v.os);
    return e + 1;
}

// Whether the output side is one gapless run: its axes, by stride, each continue
// where the one before ends (no zero, negative or overlapping strides).
static bool dense(const std::vector<AxisSpec>& dims, const std::vector<AxisSpec>& vecs, int64_t n0_override)
{
    std::vector<std::pair<int64_t, int64_t>> ax;  // stride, length
    for (size_t i = 0; i < dims.size(); i++)
        ax.push_back({dims[i].os, i == 0 && n0_override > 0 ? n0_override : dims[i].n});
    for (auto& v : vecs) ax.push_back({v.os, v.n});
    ax.erase(std::remove_if(ax.begin(), ax.end(), [](const auto& a) { return a.second == 1; }), ax.end());
    std::sort(ax.begin(), ax.end());
    int64_t next = 1;
    for (const auto& a : ax) {
        if (a.first != next) return false;
        next *= a.second;
    }
    return true;
}

// Balanced factorisation of a large 1-D length into p factors, each <= fmax
// and a product of radices.
static bool split_factors(int64_t N, int64_t fmax, std::vector<int64_t>& f)
{
    if (const char* forced = getenv("FFTZ_FACTORS")) {
        // explicit factor list (tuning experiments): "a,b[,c]" with product N
        std::vector<int64_t> g;
        int64_t prod = 1;
        for (const char* c = forced; *c;) {
            int64_t v = strtoll(c, (char**)&c, 10);
            if (v > 1) { g.push_back(v); prod *= v; }
            if (*c == ',') c++;
            else if (*c) break;
        }
        if (prod == N && g.size() >= 2 && g.size() <= 3) {
            f = g;
            return true;
        }
    }
    for (int p = 2; p <= 3; p++) {
        // candidate first factors near N^(1/p)
        const double target = std::pow((double)N, 1.0 / p);
        std::vector<int64_t> divs;
        for (int64_t d = 2; d <= fmax && d <= N; d++)
            if (N % d == 0 && smooth13(d)) divs.push_back(d);
        std::sort(divs.begin(), divs.end(),
                  [&](int64_t a, int64_t b) { return std::fabs(std::log((double)a / target)) < std::fabs(std::log((double)b / target)); });
        for (int64_t d0 : divs) {
            int64_t rest = N / d0;
            if (p == 2) {
                if (rest <= fmax && smooth13(rest)) {
                    f = {d0, rest};
                    return true;
                }
            } else {
                const double t2 = std::sqrt((double)rest);
                std::vector<int64_t> d2s;
                for (int64_t d = 2; d <= fmax && d <= rest; d++)
                    if (rest % d == 0 && smooth13(d) && rest / d <= fmax && smooth13(rest / d)) d2s.push_back(d);
                if (d2s.empty()) continue;
                std::sort(d2s.begin(), d2s.end(),
                          [&](int64_t a, int64_t b) { return std::fabs(std::log((double)a / t2)) < std::fabs(std::log((double)b / t2)); });
                f = {d0, d2s[0], rest / d2s[0]};
                return true;
            }
        }
    }
    return false;
}

// Time of a four-step pass over factor f, relative to a first pass of 256 in
// complex64 (fits to passes over 64 MiB, read and written: 30 us for 256).  A
// first or middle pass works on columns: its tile has as many lines as the LDS
// holds, so from 512 points on the segments of a row shrink below 256 bytes
// (complex128 tiles of 2^k take the whole LDS and hold out longer).  The last
// pass reads rows and is affected on its store only.  The generic kernel adds
// by its stages.  It does not know how many lines a generic tile gets: 4 lines of
// 1440 x 1440 complex128 points take 189 us as the two passes it prefers, 161 as
// three, but pricing such tiles up moved as many lengths the wrong way (5 lines
// of 632,736 61.8 -> 79.7 us).  Powers of two are priced as the fixed kernels also
// where the products of a Bluestein transform need the generic one; its two
// wide passes were the faster at every length tried (131071: 39.5 against 43.3
// us, 16 lines in complex128 132 against 165; 1048573: 88 against 91).
static double pass_cost(int64_t f, bool last, int prec)
{
    static const double col[2][6] = {{0.97, 1.0, 1.17, 1.4, 2.3, 4.0}, {0.95, 0.95, 1.12, 1.17, 1.45, 2.3}};  // 128 ..
    static const double row[2][7] = {{0.8, 0.83, 0.95, 1.03, 1.1, 1.17, 1.35},
                                     {0.8, 0.8, 0.82, 1.02, 1.02, 1.13, 1.27}};  // 64 .. 4096
    const double* t = last ? row[prec == 8] : col[prec == 8];
    const int n = last ? 7 : 6;
    const double x = std::min(std::max(std::log2((double)f) - (last ? 6.0 : 7.0), 0.0), n - 1.0);
    const int i = std::min((int)x, n - 2);
    double c = t[i] + (x - i) * (t[i + 1] - t[i]);
    std::vector<int> r;
    if ((f & (f - 1)) != 0 && factor_radices((int)f, r)) c *= r.size() <= 2 ? 1.1 : r.size() == 3 ? 1.12 : 1.3;
    return c;
}

// The cheapest two-pass split of N, each factor at most 2048; false when there is none.
static bool split_two(int64_t N, int prec, std::vector<int64_t>& f, double& cost)
{
    cost = 1e300;
    if (N > 2048 * 2048) return false;
    for (int64_t a = std::max<int64_t>(16, (N + 2047) / 2048); a <= 2048 && 16 * a <= N; a++) {
        if ((uint32_t)N % (uint32_t)a) continue;
        const int64_t b = N / a;
        if (!smooth13(a) || !smooth13(b)) continue;
        // wide generic passes leave one or two lines per tile
        const int64_t generic = prec == 4 ? 2048 : 1536;
        if (((a & (a - 1)) && a > generic) || ((b & (b - 1)) && b > generic)) continue;
        const double c = pass_cost(a, false, prec) + pass_cost(b, true, prec);
        if (c < cost) {
            cost = c;
            f = {a, b};
        }
    }
    return cost < 1e300;
}

static bool split_ok(int64_t N, const std::vector<int64_t>& f, int64_t fmax)
{
    if (f.size() < 2 || f.size() > 3) return false;
    int64_t prod = 1;
    for (int64_t v : f) {
        if (v < 2 || v > fmax || !smooth13(v)) return false;
        prod *= v;
    }
    return prod == N;
}

std::vector<std::vector<int64_t>> split_candidates(int64_t N, int prec, int maxn)
{
    // Ordered 2- and 3-factor splits within one LDS pass per factor, most
    // balanced first (sum of |log f - log N^(1/p)|), three factors before two.
    const int64_t fmax = single_pass_limit(prec);
    std::vector<std::pair<double, std::vector<int64_t>>> c;
    std::vector<int64_t> divs;
    for (int64_t d = 16; d <= fmax && d <= N; d++)
        if (N % d == 0 && smooth13(d)) divs.push_back(d);
    for (int p = 3; p >= 2; p--) {
        const double t = std::log((double)N) / p;
        for (int64_t a : divs)
            for (int64_t b : divs) {
                if (N % (a * b)) continue;
                const int64_t r = N / (a * b);
                std::vector<int64_t> f = p == 3 ? std::vector<int64_t>{a, b, r} : std::vector<int64_t>{a, N / a};
                if (p == 2 && b != divs[0]) continue;
                if (!split_ok(N, f, fmax) || f.back() < 16) continue;
                double score = (3 - p) * 100.0;
                for (int64_t v : f) score += std::fabs(std::log((double)v) - t);
                c.push_back({score, f});
            }
    }
    std::stable_sort(c.begin(), c.end(), [](const auto& x, const auto& y) { return x.first < y.first; });
    std::vector<std::vector<int64_t>> out;
    for (const auto& e : c)
        if ((int)out.size() < maxn && std::find(out.begin(), out.end(), e.second) == out.end()) out.push_back(e.second);
    return out;
}

// A length-N transform along one axis of a tensor, through the work buffer,
// as a four-step over p = 2 or 3 factors (the p = 2 form is
// core/solvers/complex/pow2_fourstep_solver_dft.c:700-763, with the twiddle
// and transpose of fused_twiddle_transpose_c.c:20-110 folded into the passes'
// stores): the first pass reads the source and writes the dense intermediate
// [batch][N] in the work buffer with the inter-pass twiddle applied, middle
// passes work in place on it, and the last pass writes the destination with
// the transpose folded into its store.  Any number of other axes ride along
// as batch lines (the reference loops them, batched_solver_dft.c:33-110).
struct LongAxis {
    int64_t N = 0;
    int64_t is = 1, os = 1;               // element strides in the source / destination
    std::vector<AxisSpec> batch;          // other axes: n, source stride, destination stride
    Role src = Role::In, dst = Role::Out;
    int64_t src_base = 0, dst_base = 0;   // bytes into the source / destination buffer
    int64_t work_base = 0;                // bytes into the work buffer of the intermediate
    bool conj_in = false, conj_out = false;
    uint32_t first_flags = 0, last_flags = 0;  // Bluestein products (kChirpFlags)
    int64_t nchirp = 0, chirp_off = -1, spec_off = -1;
};

static bool plan_long_axis(Plan* plan, TableBuilder& tb, const LongAxis& a, std::string& err)
{
    const int prec = plan->spec.prec_bytes;
    const int64_t N = a.N;
    // Largest pass length: 256 keeps column tiles 16 lines wide (256-byte
    // FP64 / 128-byte FP32 segments) with 256-thread workgroups; grow it only
    // when three passes of 256 cannot cover N.
    int64_t fmax = env_int(prec == 8 ? "FFTZ_FMAX_D" : "FFTZ_FMAX_F", 256);
    while (fmax < 4096 && fmax * fmax * fmax < N) fmax *= 2;
    std::vector<int64_t> f;
    const std::vector<int64_t>& tuned = plan->spec.tune.split;
    const bool use_tuned = split_ok(N, tuned, single_pass_limit(prec));
    if (use_tuned) {
        f = tuned;
    } else if (!split_factors(N, fmax, f)) {
        err = "no four-step factorisation for length " + std::to_string(N);
        return false;
    }
    // power-of-two factors last: the final (transposing) pass then runs on
    // the fixed-length kernel
    if (!use_tuned && !getenv("FFTZ_FACTORS")) {
        std::stable_sort(f.begin(), f.end(), [](int64_t x, int64_t y) {
            return ((x & (x - 1)) != 0) > ((y & (y - 1)) != 0);
        });
        // two wider passes where they cost clearly less than these (64 MiB in
        // all: 8 x 2^20 complex64 as 512 x 2048 65 us, as 128 x 128 x 64 75 us;
        // 9 x 1,000,000 as 1000 x 1000 81 us, as 100 x 100 x 100 98 us), but not
        // the widest powers of two on data beyond the Infinity Cache, where
        // segments below a cache line cost more than a third pass (16 x 2^20
        // there and back 327 against 288 us; complex128 8 x 2^21 583 against 562)
        double three = 0.0, two = 0.0;
        bool pow2 = true;
        for (size_t i = 0; i < f.size(); i++) {
            three += pass_cost(f[i], i + 1 == f.size(), prec);
            pow2 = pow2 && (f[i] & (f[i] - 1)) == 0;
        }
        int64_t total = N * 2 * prec;
        for (auto& b : a.batch) total *= b.n;
        const bool far = pow2 && total > ((int64_t)96 << 20) && N > (prec == 4 ? 1 << 19 : 1 << 20);
        std::vector<int64_t> g;
        if (!far && split_two(N, prec, g, two) && two < 0.93 * three) f = g;
    }
    // dense intermediate: batch axis i at stride N * prod_{j<i} n_j
    std::vector<int64_t> wst(a.batch.size());
    int64_t B = 1;
    for (size_t i = 0; i < a.batch.size(); i++) {
        wst[i] = N * B;
        B *= a.batch[i].n;
    }
    const size_t p = f.size();
    std::vector<int64_t> M(p);  // M[s] = N / (f0...fs)
    int64_t acc = N;
    for (size_t s = 0; s < p; s++) {
        acc /= f[s];
        M[s] = acc;
    }
    plan->work_bytes = std::max(plan->work_bytes, (size_t)(a.work_base + N * B * 2 * prec));
    // step 0: columns of the source (element g = l0 + e M0), twiddle on store
    {
        PassReq q;
        q.L = (int)f[0];
        q.ies = M[0] * a.is;
        q.oes = M[0];
        LineAxis l0{M[0], a.is, 1};
        l0.gi = 1;
        q.lines.push_back(l0);
        for (size_t i = 0; i < a.batch.size(); i++) q.lines.push_back({a.batch[i].n, a.batch[i].is, wst[i]});
        q.flags = kTw4 | (a.conj_in ? kConjIn : 0) | (a.first_flags & kChirpIn);
        q.tw4_n = N;
        q.want_in_col = (a.is == 1);
        q.want_out_col = true;
        q.in_role = a.src;
        q.out_role = Role::Work;
        q.in_base = a.src_base;
        q.out_base = a.work_base;
        q.gie = M[0];
        q.nchirp = a.nchirp;
        q.chirp_off = a.chirp_off;
        if (!build_pass(plan, tb, q, err)) return false;
    }
    // middle steps (p == 3)
    for (size_t s = 1; s + 1 < p; s++) {
        PassReq q;
        q.L = (int)f[s];
        q.ies = M[s];
        q.oes = M[s];
        q.lines.push_back({M[s], 1, 1});
        const int64_t rows = N / M[s - 1];
        q.lines.push_back({rows, M[s - 1], M[s - 1]});
        for (size_t i = 0; i < a.batch.size(); i++) q.lines.push_back({a.batch[i].n, wst[i], wst[i]});
        q.flags = kTw4;
        q.tw4_n = M[s - 1];
        q.want_in_col = q.want_out_col = true;
        q.in_role = q.out_role = Role::Work;
        q.in_base = q.out_base = a.work_base;
        if (!build_pass(plan, tb, q, err)) return false;
    }
    // last step: rows of length f[p-1]; row (k0, k1) element e is output
    // k = k0 + f0 k1 + e (N / f[p-1]), stored at k * os
    {
        PassReq q;
        q.L = (int)f[p - 1];
        q.ies = 1;
        const int64_t outer = N / f[p - 1];
        q.oes = a.os * outer;
        q.goe = outer;
        LineAxis k0{f[0], M[0], a.os};
        k0.go = 1;
        q.lines.push_back(k0);
        if (p == 3) {
            LineAxis k1{f[1], M[1], a.os * f[0]};
            k1.go = f[0];
            q.lines.push_back(k1);
        }
        for (size_t i = 0; i < a.batch.size(); i++) q.lines.push_back({a.batch[i].n, wst[i], a.batch[i].os});
        q.flags = (a.conj_out ? kConjOut : 0) | (a.last_flags & (kSpecOut | kChirpOut));
        q.want_in_col = false;
        q.want_out_col = (a.os == 1);
        q.in_role = Role::Work;
        q.out_role = a.dst;
        q.in_base = a.work_base;
        q.out_base = a.dst_base;
        q.nchirp = a.nchirp;
        q.chirp_off = a.chirp_off;
        q.spec_off = a.spec_off;
        if (!build_pass(plan, tb, q, err)) return false;
    }
    std::ostringstream os;
    os << "four-step";
    for (auto v : f) os << " " << v;
    plan->description += os.str() + "; ";
    return true;
}

// Bluestein for a length n whose extended length M exceeds one LDS tile
// (core/solvers/complex/bluestein_solver_dft.c:137-234): the chirp product
// x conj(B) rides on the first pass of a four-step FFT_M, the spectrum
// product conj(A) conj(FFT_M(b)) / M on its last store, a second four-step
// FFT_M reads that and its last store forms conj(B W) (forward) or B W
// (backward, whose input was conjugated on load) for the n outputs.  Work
// buffer: [intermediate of both transforms | product Z], M x batch each.
static bool plan_bluestein_long(Plan* plan, TableBuilder& tb, int64_t n, int64_t is, int64_t os,
                                const std::vector<AxisSpec>& batch, Role src, Role dst, bool bwd,
                                std::string& err)
{
    const int prec = plan->spec.prec_bytes;
    const int64_t M = bluestein_length(n);
    int64_t B = 1;
    for (auto& b : batch) B *= b.n;
    int64_t chirp_off = -1, spec_off = -1;
    bluestein_tables(tb, prec, n, M, &chirp_off, &spec_off, plan->dry_run);
    const int64_t zbase = M * B * 2 * prec;  // region of the product Z
    std::vector<AxisSpec> b1 = batch, b2 = batch;
    int64_t dense = M;
    for (size_t i = 0; i < batch.size(); i++) {
        b1[i].os = dense;
        b2[i].is = dense;
        dense *= batch[i].n;
    }
    LongAxis a1;
    a1.N = M;
    a1.is = is;
    a1.os = 1;
    a1.batch = b1;
    a1.src = src;
    a1.dst = Role::Work;
    a1.dst_base = zbase;
    a1.conj_in = bwd;
    a1.first_flags = kChirpIn;
    a1.last_flags = kSpecOut;
    a1.nchirp = n;
    a1.chirp_off = chirp_off;
    a1.spec_off = spec_off;
    if (!plan_long_axis(plan, tb, a1, err)) return false;
    LongAxis a2;
    a2.N = M;
    a2.is = 1;
    a2.os = os;
    a2.batch = b2;
    a2.src = Role::Work;
    a2.src_base = zbase;
    a2.dst = dst;
    a2.conj_out = !bwd;
    a2.last_flags = kChirpOut;
    a2.nchirp = n;
    a2.chirp_off = chirp_off;
    if (!plan_long_axis(plan, tb, a2, err)) return false;
    plan->work_bytes = std::max(plan->work_bytes, (size_t)(2 * zbase));
    plan->description += "Bluestein n=" + std::to_string(n) + " M=" + std::to_string(M) + " (multi-pass); ";
    return true;
}

// One complete 1-D transform along axis `ax` of a tensor as a list of passes:
// one LDS pass when the length fits a tile (a fused Bluestein pass for a
// length with a prime factor above 13), else the four-step or multi-pass
// Bluestein through the work buffer.  The input is read with the caller's
// input strides, or with the output strides when the axis runs in place on
// the output (use_out_strides_for_in).
static bool plan_axis_c2c(Plan* plan, TableBuilder& tb, const std::vector<AxisSpec>& dims,
                          const std::vector<AxisSpec>& vecs, size_t axis, bool conj_in, bool conj_out,
                          Role in_role, Role out_role, bool use_out_strides_for_in, std::string& err)
{
    const int prec = plan->spec.prec_bytes;
    const int64_t n = dims[axis].n;
    PassReq q;
    q.in_role = in_role;
    q.out_role = out_role;
    q.ies = use_out_strides_for_in ? dims[axis].os : dims[axis].is;
    q.oes = dims[axis].os;
    std::vector<AxisSpec> batch;
    for (size_t j = 0; j < dims.size(); j++)
        if (j != axis) batch.push_back({dims[j].n, use_out_strides_for_in ? dims[j].os : dims[j].is, dims[j].os});
    for (auto& v : vecs) batch.push_back({v.n, use_out_strides_for_in ? v.os : v.is, v.os});
    for (auto& b : batch) q.lines.push_back({b.n, b.is, b.os});
    if (conj_in) q.flags |= kConjIn;
    if (conj_out) q.flags |= kConjOut;
    q.want_in_col = q.ies != 1;
    q.want_out_col = q.oes != 1;
    if (smooth13(n)) {
        if (n > single_pass_limit(prec)) {
            LongAxis a;
            a.N = n;
            a.is = q.ies;
            a.os = q.oes;
            a.batch = batch;
            a.src = in_role;
            a.dst = out_role;
            a.conj_in = conj_in;
            a.conj_out = conj_out;
            return plan_long_axis(plan, tb, a, err);
        }
        q.L = (int)n;
        return build_pass(plan, tb, q, err);
    }
    // Bluestein
    const int64_t M = bluestein_tile_length(n, single_pass_limit(prec));
    if (M > single_pass_limit(prec))
        return plan_bluestein_long(plan, tb, n, q.ies, q.oes, batch, in_role, out_role, conj_in, err);
    q.kind = KernelKind::Bluestein;
    q.L = (int)M;
    q.nvalid_in = (int)n;
    q.nvalid_out = (int)n;
    bluestein_tables(tb, prec, n, M, &q.chirp_off, &q.spec_off, plan->dry_run);
    q.want_in_col = q.want_out_col = false;
    return build_pass(plan, tb, q, err);
}

static bool plan_c2c(Plan* plan, TableBuilder& tb, std::vector<AxisSpec> dims, const std::vector<AxisSpec>& vecs,
                     std::string& err)
{
    const bool bwd = plan->spec.dir == 1;
    for (size_t a = 0; a < dims.size(); a++) {
        const bool first = (a == 0);
        if (!plan_axis_c2c(plan, tb, dims, vecs, a, bwd, bwd, first ? Role::In : Role::Out, Role::Out, !first, err))
            return false;
    }
    plan->description += "row-column " + std::to_string(dims.size()) + "-D; ";
    return true;
}

// Full-length pass for a real axis of length n (odd n, or an even n whose half
// has no radix plan): the n-point complex transform of the real line promoted
// to complex (R2C), or of the Hermitian extension of the n/2+1 stored bins
// with only the real part stored (C2R).  Bluestein when n has a prime factor
// above 13.  Twice the arithmetic of the packed form; same HBM traffic.
static bool real_full_pass(Plan* plan, TableBuilder& tb, PassReq q, int64_t n, std::string& err)
{
    const int prec = plan->spec.prec_bytes;
    const bool r2c = (q.flags & kRealPromote) != 0;
    q.nvalid_in = (int)n;
    q.nvalid_out = r2c ? (int)(n / 2 + 1) : (int)n;
    q.want_in_col = q.want_out_col = false;
    if (smooth13(n)) {
        if (n > single_pass_limit(prec)) {
            err = "real length " + std::to_string(n) + " above the single-pass limit";
            return false;
        }
        q.L = (int)n;
        return build_pass(plan, tb, q, err);
    }
    const int64_t M = bluestein_tile_length(n, single_pass_limit(prec));
    if (M > single_pass_limit(prec)) {
        err = "Bluestein length " + std::to_string(M) + " for real length " + std::to_string(n) +
              " exceeds the fused single-pass limit";
        return false;
    }
    q.kind = KernelKind::Bluestein;
    q.L = (int)M;
    bluestein_tables(tb, prec, n, M, &q.chirp_off, &q.spec_off, plan->dry_run);
    return build_pass(plan, tb, q, err);
}

static bool plan_real(Plan* plan, TableBuilder& tb, std::vector<AxisSpec> dims, const std::vector<AxisSpec>& vecs,
                      std::string& err)
{
    const int prec = plan->spec.prec_bytes;
    const bool r2c = plan->spec.type == FftType::R2C;
    const int64_t n0 = dims[0].n;
    const int64_t L = n0 / 2;
    // real-packed (n0/2-point complex transform + recombine / separate) when
    // n0 is even and its half has a single-pass radix plan; otherwise the
    // full-length promoted / Hermitian pass
    const bool packed = n0 % 2 == 0 && smooth13(L) && L <= single_pass_limit(prec) && L >= 1;
    const int64_t nbins = n0 / 2 + 1;
    int64_t rtw_off = -1;
    if (packed) {
        std::vector<d2> rtw((size_t)L);
        const RootTable root(n0);
        for (int64_t k = 0; k < L; k++) rtw[(size_t)k] = root(k);
        rtw_off = tb.add_complex(rtw, prec);
    }
    // complex geometry of the half-spectrum side
    std::vector<AxisSpec> cd = dims;  // n of dim 0 becomes L+1 bins on the complex side
    if (r2c) {
        PassReq q;
        q.L = (int)L;
        q.ies = dims[0].is;  // real elements
        q.oes = dims[0].os;
        for (size_t j = 1; j < dims.size(); j++) q.lines.push_back({dims[j].n, dims[j].is, dims[j].os});
        for (auto& v : vecs) q.lines.push_back({v.n, v.is, v.os});
        q.in_role = Role::In;
        q.out_role = Role::Out;
        if (packed) {
            q.flags = kRealIn | kR2CPost;
            q.rtw_off = rtw_off;
            if (!build_pass(plan, tb, q, err)) return false;
        } else {
            q.flags = kRealPromote;
            if (!real_full_pass(plan, tb, q, n0, err)) return false;
        }
        // remaining axes: C2C forward in place on the output
        cd[0].n = nbins;
        for (size_t a = 1; a < dims.size(); a++) {
            std::vector<AxisSpec> od = cd;
            if (!plan_axis_c2c(plan, tb, od, vecs, a, false, false, Role::Out, Role::Out, true, err))
                return false;
        }
        plan->description += packed ? "real-packed R2C; " : "real R2C (full length); ";
        return true;
    }
    // C2R: outer axes backward into the work buffer, then separate + FFT.
    Role src = Role::In;
    std::vector<AxisSpec> wdims = dims;
    std::vector<AxisSpec> wvecs = vecs;
    if (dims.size() > 1) {
        // dense work layout: [vec][dims reversed], dim0 has L+1 bins
        int64_t stride = 1;
        std::vector<AxisSpec> dd = dims;
        dd[0].n = nbins;
        for (size_t j = 0; j < dd.size(); j++) {
            wdims[j] = {dd[j].n, dd[j].is, stride};
            stride *= dd[j].n;
        }
        int64_t per = stride;
        for (size_t v = 0; v < wvecs.size(); v++) {
            wvecs[v] = {vecs[v].n, vecs[v].is, stride};
            stride *= vecs[v].n;
        }
        plan->work_bytes = std::max(plan->work_bytes, (size_t)(stride * 2 * prec));
        (void)per;
        // copy-transform axis 1 from In to Work, then the rest in place on Work
        for (size_t a = 1; a < dims.size(); a++) {
            const bool first = (a == 1);
            std::vector<AxisSpec> od = wdims;
            if (!plan_axis_c2c(plan, tb, od, wvecs, a, true, true, first ? Role::In : Role::Work,
                               Role::Work, !first, err))
                return false;
        }
        src = Role::Work;
        for (size_t j = 0; j < wdims.size(); j++) wdims[j].is = wdims[j].os;
        for (size_t v = 0; v < wvecs.size(); v++) wvecs[v].is = wvecs[v].os;
    }
    PassReq q;
    q.L = (int)L;
    q.ies = wdims[0].is;
    q.oes = dims[0].os;  // real elements
    for (size_t j = 1; j < dims.size(); j++) q.lines.push_back({dims[j].n, wdims[j].is, dims[j].os});
    for (size_t v = 0; v < vecs.size(); v++) q.lines.push_back({vecs[v].n, wvecs[v].is, vecs[v].os});
    q.in_role = src;
    q.out_role = Role::Out;
    if (!packed) {
        // backward = conjugate in and out around the forward transform
        q.flags = kHermIn | kConjIn | kConjOut | kRealPart;
        if (!real_full_pass(plan, tb, q, n0, err)) return false;
        plan->description += "real C2R (full length); ";
        return true;
    }
    q.nvalid_in = (int)(L + 1);
    q.extra_lds_elems = 1;
    q.flags = kC2RPre | kConjOut | kRealOut;
    q.rtw_off = rtw_off;
    if (!build_pass(plan, tb, q, err)) return false;
    plan->description += "real-packed C2R; ";
    return true;
}

// ---------------------------------------------------------------------------
// Uneven batches (many lengths, one persistent launch per tile class).
// The reference runs such a list as independent plans, one setup/execute per
// (n, batch) item; here every distinct length becomes a pass descriptor in the
// plan arena and every item a run of tiles in a device work queue.
// ---------------------------------------------------------------------------
namespace {
struct SizeInfo {
    int64_t n = 0;
    bool bluestein = false;
    int L = 0;
    int cls = 0;
    int C = 1;
    PassDesc d{};
};
}  // namespace

static bool batch_size_desc(TableBuilder& tb, int prec, int64_t n, int maxt, size_t lds_budget,
                            SizeInfo& si, std::string& err)
{
    si.n = n;
    si.bluestein = !smooth13(n);
    const int64_t L = si.bluestein ? bluestein_tile_length(n, single_pass_limit(prec)) : n;
    si.L = (int)L;
    PassDesc& d = si.d;
    d = PassDesc{};
    std::vector<int> radix;
    if (!factor_radices((int)L, radix)) {
        err = "no radix plan for batch length " + std::to_string(L);
        return false;
    }
    d.L = (int)L;
    if (si.bluestein && radix.size() < 2) {
        err = "internal: Bluestein batch length " + std::to_string(L) + " with one stage";
        return false;
    }
    const int TL = line_threads(radix, (int)L, 32 / prec, maxt, -1, INT32_MAX, prec);
    const int most = (int)std::min<size_t>(L + L / 16 + 16, lds_budget / (2 * prec) - 1);
    const int64_t stw = digit_layout(tb, prec, radix, (int)L, TL, (int)L, most, d);
    d.TL = TL;
    d.tl_shift = ilog2(TL);
    const size_t line_bytes = (size_t)d.LP * 2 * prec;
    if (line_bytes > lds_budget) {
        err = "batch length " + std::to_string(L) + " exceeds LDS";
        return false;
    }
    int C = 1;
    const int cmax = env_int("FFTZ_BATCH_CMAX", 64);
    while (C * 2 * TL <= maxt && (size_t)(C * 2) * line_bytes <= lds_budget && C * 2 <= cmax) C *= 2;
    si.C = C;
    d.C = C;
    d.c_shift = ilog2(C);
    d.ies = 1;
    d.oes = 1;
    d.ln0 = make_fastdiv(1u << 30);  // l0 = line index (< 2^30)
    d.ln1 = make_fastdiv(1);
    d.ils[1] = d.ils[2] = d.ols[1] = d.ols[2] = 0;
    d.nvalid_in = si.bluestein ? (int)n : (int)L;
    d.nvalid_out = si.bluestein ? (int)n : (int)L;
    d.scale_f = 1.0f;
    d.scale_d = 1.0;
    // table pointers hold arena offsets until upload (resolved in place)
    d.stw = (const void*)(intptr_t)stw;
    if (si.bluestein) {
        int64_t co, so;
        bluestein_tables(tb, prec, n, L, &co, &so, false);
        d.chirp = (const void*)(intptr_t)co;
        d.spec = (const void*)(intptr_t)so;
    }
    return true;
}

Plan* batch_plan_create(const std::vector<BatchItem>& items, int prec, int dir, std::string& err, bool dry_run,
                        const TuneParams* tune)
{
    Plan* plan = new Plan();
    plan->dry_run = dry_run;
    plan->spec.prec_bytes = prec;
    plan->spec.dir = dir;
    plan->spec.type = FftType::C2C;
    plan->is_batch = true;
    if (!dry_run) {
        (void)hipGetDevice(&plan->device);
        (void)device_info();
    }
    const DeviceInfo& dev = device_info();
    const int esize = 2 * prec;
    TableBuilder tb{plan->host_tables};
    // size classes: small tiles (256 threads, <= 64 KiB LDS, several
    // workgroups per CU) and large tiles (whole LDS; 1024 threads, 512 in
    // complex128)
    const int big_threads = prec == 4 ? 1024 : 512;
    const size_t static_lds = kBatchHdrBytes;
    const size_t small_budget = (size_t)env_int("FFTZ_BATCH_SMALL_LDS", 64 * 1024);
    const size_t big_budget = dev.lds_per_block - static_lds;
    // medium tiles: 512 threads, at most half the LDS, two workgroups per CU
    // (lines up to 10175 complex64 points: 2000 items 2.12 -> 2.08 ms against 8192)
    const size_t medium_budget = dev.lds_per_block / 2 - static_lds;
    std::map<int64_t, int> size_index;
    std::vector<SizeInfo> sizes;
    int64_t in_ext = 0, out_ext = 0;
    double flops = 0.0;
    for (const BatchItem& it : items) {
        if (it.n <= 0 || it.batch < 0 || it.in_off < 0 || it.out_off < 0 || it.dist < 0) {
            err = "invalid batch item";
            delete plan;
            return nullptr;
        }
        if (it.batch == 0) continue;
        const int64_t dist = it.dist ? it.dist : it.n;
        in_ext = std::max(in_ext, it.in_off + (it.batch - 1) * dist + it.n);
        out_ext = std::max(out_ext, it.out_off + (it.batch - 1) * dist + it.n);
        flops += 5.0 * (double)it.n * std::log2(std::max<double>((double)it.n, 2.0)) * (double)it.batch;
        plan->n_transforms += it.batch;
        if (size_index.count(it.n)) continue;
        SizeInfo si;
        si.n = it.n;
        const int64_t L = smooth13(it.n) ? it.n : bluestein_tile_length(it.n, single_pass_limit(prec));
        const bool small = next_pow2((L + 7) / 8) <= 256 && (size_t)(lds_pad((int)L) + 2) * esize <= small_budget / 2;
        const bool medium = !small && (size_t)(L + 1) * esize <= medium_budget;
        si.cls = small ? 0 : (medium ? 1 : 2);
        size_index[it.n] = (int)sizes.size();
        sizes.push_back(si);
    }
    // Per-length descriptors and tables (stage twiddles, Bluestein chirp and
    // spectrum) are independent: build them on worker threads into separate
    // arenas, then append each arena to the plan's and rebase its offsets.
    {
        const int cT[3] = {256, 512, big_threads};
        const size_t cB[3] = {small_budget, medium_budget, big_budget};
        std::vector<std::vector<unsigned char>> arenas(sizes.size());
        std::vector<std::string> errs(sizes.size());
        std::vector<char> ok(sizes.size(), 0);
        std::atomic<size_t> next{0};
        auto work = [&]() {
            for (size_t i; (i = next.fetch_add(1)) < sizes.size();) {
                TableBuilder ltb{arenas[i]};
                SizeInfo& si = sizes[i];
                const int cls = si.cls;
                ok[i] = batch_size_desc(ltb, prec, si.n, cT[cls], cB[cls], si, errs[i]) ? 1 : 0;
                si.cls = cls;
            }
        };
        const unsigned hw = std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
        const size_t nthr = std::min<size_t>(hw, (sizes.size() + 7) / 8);
        std::vector<std::thread> pool;
        for (size_t t = 1; t < nthr; t++) pool.emplace_back(work);
        work();
        for (auto& t : pool) t.join();
        for (size_t i = 0; i < sizes.size(); i++) {
            if (!ok[i]) {
                err = errs[i];
                delete plan;
                return nullptr;
            }
            const int64_t base = tb.add(arenas[i].data(), arenas[i].size());
            PassDesc& d = sizes[i].d;
            auto rebase = [base](const void*& ptr) { ptr = (const void*)((intptr_t)ptr + (intptr_t)base); };
            rebase(d.stw);
            if (sizes[i].bluestein) {
                rebase(d.chirp);
                rebase(d.spec);
            }
        }
    }
    plan->in_extent_bytes = in_ext * esize;
    plan->out_extent_bytes = out_ext * esize;
    plan->flops = flops;
    // tiles per class, cost-sorted (largest first)
    // A queue entry covers up to `rounds` rounds of C lines, so that the per-entry
    // cost (queue atomic, descriptor loads, barriers) is amortised -- but its
    // rounds run one after the other, and a workgroup's last entry is the
    // launch's tail: an eighth of what a resident workgroup gets in all, between
    // 16 KiB and 128 / 256 KiB in the medium / large class.  Against 128 / 256 KiB
    // throughout: 2000 items 2.18 -> 2.05 ms, 400 items 0.65 -> 0.48 ms, 100 items
    // 0.43 -> 0.14 ms.  Entries of the small class are short, so that their number
    // counts: 4096 points, or the largest half of that which gives seven for
    // every four resident workgroups, down to 16 KiB (2000 items of 64 points each,
    // complex64: 32 KiB 61 us, 16 KiB 70 us; 500 items of 16 to 256 points the
    // reverse, 48 and 41 us; 128 KiB in a list with longer items 168 us, 135).
    const int64_t entry_env = env_int("FFTZ_BATCH_ENTRY_BYTES", 0);
    const int64_t resident[3] = {4, 2, 1};
    auto entry_rounds = [&](const SizeInfo& si, int64_t bytes) {
        return std::max<int64_t>(1, std::min<int64_t>(16, bytes / std::max<int64_t>(1, (int64_t)si.C * si.n * esize)));
    };
    int64_t entry_cls[3] = {4096 * esize, 128 * 1024, 256 * 1024}, bytes_cls[3] = {0, 0, 0}, short_cls[3] = {0, 0, 0};
    for (const BatchItem& it : items) {
        if (!it.batch) continue;
        const int c = sizes[(size_t)size_index[it.n]].cls;
        bytes_cls[c] += it.n * it.batch * esize;
        if (it.n * esize < 2048) short_cls[c] += it.n * it.batch * esize;
    }
    for (int c = 1; c < 3; c++)
        entry_cls[c] = std::max<int64_t>(16 * 1024, std::min(entry_cls[c], bytes_cls[c] / (8 * dev.cus * resident[c])));
    for (; entry_cls[0] > 16 * 1024; entry_cls[0] /= 2) {
        int64_t n = 0;
        for (const BatchItem& it : items) {
            const SizeInfo& si = sizes[(size_t)size_index[it.n]];
            const int64_t step = (int64_t)si.C * entry_rounds(si, entry_cls[0]);
            if (si.cls == 0) n += (it.batch + step - 1) / step;
        }
        if (4 * n >= 7 * dev.cus * resident[0]) break;
    }
    std::vector<std::vector<std::pair<double, BatchTile>>> tiles(3);
    for (const BatchItem& it : items) {
        if (it.batch == 0) continue;
        const SizeInfo& si = sizes[(size_t)size_index[it.n]];
        const int64_t dist = it.dist ? it.dist : it.n;
        const int64_t entry_bytes = entry_env > 0 ? entry_env : entry_cls[si.cls];
        const int64_t step = (int64_t)si.C * entry_rounds(si, entry_bytes);
        for (int64_t l0 = 0; l0 < it.batch; l0 += step) {
            BatchTile bt{};
            bt.desc = (uint32_t)size_index[it.n];
            bt.nlines = (uint32_t)std::min<int64_t>(step, it.batch - l0);
            bt.bluestein = si.bluestein ? 1u : 0u;
            bt.in_off = it.in_off + l0 * dist;
            bt.out_off = it.out_off + l0 * dist;
            bt.dist = dist;
            const double cost = (double)bt.nlines * si.L * (std::log2((double)si.L + 1.0) + 8.0) *
                                (si.bluestein ? 2.5 : 1.0);
            tiles[(size_t)si.cls].push_back({cost, bt});
        }
    }
    // direction: every tile is a complete transform; backward conjugates in
    // and out (the Bluestein body handles its own conjugation)
    for (SizeInfo& si : sizes)
        if (dir == 1) si.d.flags |= kConjIn | kConjOut;
    std::vector<PassDesc> descs;
    for (const SizeInfo& si : sizes) descs.push_back(si.d);
    plan->descs_off = tb.add(descs.data(), std::max<size_t>(1, descs.size()) * sizeof(PassDesc));
    for (int c = 0; c < 3; c++) {
        auto& tl = tiles[(size_t)c];
        std::stable_sort(tl.begin(), tl.end(), [](const auto& a, const auto& b) { return a.first > b.first; });
        BatchClass bc;
        bc.maxt = c == 0 ? 256 : (c == 1 ? 512 : big_threads);
        // Short lines anywhere in the buffers are not whole cache lines: plain
        // stores where most of the small class is below 2 KiB a line (3508 items of
        // 16 to 64 complex128 points 102 -> 96 us, then read in order 212 -> 192; 4000
        // of 16 to 256 points the reverse, 235 and 272).
        bc.nt = c > 0 || 2 * short_cls[0] <= bytes_cls[0];
        bc.ntiles = (int)tl.size();
        size_t lds = 0;
        for (const SizeInfo& si : sizes)
            if (si.cls == c) lds = std::max(lds, (size_t)si.C * si.d.LP * esize);
        bc.lds_bytes = (uint32_t)(lds + kBatchHdrBytes);
        bc.grid = 1;
        if (bc.ntiles) {
            std::vector<BatchTile> v;
            v.reserve(tl.size());
            for (auto& t : tl) v.push_back(t.second);
            bc.tiles_off = tb.add(v.data(), v.size() * sizeof(BatchTile));
        }
        plan->bclasses.push_back(bc);
    }
    std::ostringstream os;
    {
        plan->tune_key = batch_key(items, prec, dir);
        TuneParams t;
        if (tune) t = *tune;
        else (void)tune_lookup(plan->tune_key, t);
        batch_set_grids(plan, t.wg_small, t.wg_medium);
    }
    static const char* kClassName[3] = {"small", "medium", "large"};
    os << "uneven batch: " << plan->n_transforms << " transforms, " << sizes.size() << " lengths; tiles";
    for (int c = 0; c < 3; c++)
        os << " " << kClassName[c] << "=" << plan->bclasses[(size_t)c].ntiles << " (grid " << plan->bclasses[(size_t)c].grid
           << ", lds " << plan->bclasses[(size_t)c].lds_bytes << ")";
    os << "; ";
    plan->description = os.str();
    if (dry_run) return plan;
    if (hipMalloc(&plan->tables, plan->host_tables.size()) != hipSuccess) {
        err = "device allocation for batch tables failed";
        delete plan;
        return nullptr;
    }
    // resolve descriptor table offsets to device pointers, then upload
    char* base = (char*)plan->tables;
    PassDesc* hd = reinterpret_cast<PassDesc*>(plan->host_tables.data() + plan->descs_off);
    for (size_t i = 0; i < sizes.size(); i++) {
        hd[i].stw = base + (intptr_t)hd[i].stw;
        if (sizes[i].bluestein) {
            hd[i].chirp = base + (intptr_t)hd[i].chirp;
            hd[i].spec = base + (intptr_t)hd[i].spec;
        }
    }
    if (hipMemcpy(plan->tables, plan->host_tables.data(), plan->host_tables.size(), hipMemcpyHostToDevice) !=
        hipSuccess) {
        err = "upload of batch tables failed";
        (void)hipFree(plan->tables);
        delete plan;
        return nullptr;
    }
    for (size_t c = 0; c < plan->bclasses.size(); c++)
        (void)hipFuncSetAttribute(kernel_symbol_batch(prec, (int)c, plan->bclasses[c].nt),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)dev.lds_per_block);
    plan->host_tables.clear();
    plan->host_tables.shrink_to_fit();
    plan->use_graph = env_int("FFTZ_BATCH_GRAPH", 1) != 0;
    return plan;
}

void batch_set_grids(Plan* p, int wg_small, int wg_medium)
{
    const DeviceInfo& dev = device_info();
    for (size_t c = 0; c < p->bclasses.size(); c++) {
        BatchClass& bc = p->bclasses[c];
        const int per_cu = c == 0 ? (wg_small ? wg_small : env_int("FFTZ_BATCH_WG_SMALL", 8))
                           : c == 1 ? (wg_medium ? wg_medium : env_int("FFTZ_BATCH_WG_MEDIUM", 2))
                                    : env_int("FFTZ_BATCH_WG_BIG", 1);
        bc.grid = (uint32_t)std::max<int64_t>(1, std::min<int64_t>(bc.ntiles, (int64_t)dev.cus * per_cu));
    }
    // captured graphs hold the old grids
    for (Slot* s : p->slots) {
        if (s->graph) (void)hipGraphExecDestroy(s->graph);
        s->graph = nullptr;
        s->graph_in = nullptr;
        s->graph_out = nullptr;
    }
}

// ---------------------------------------------------------------------------
// Tuned-parameter cache
// ---------------------------------------------------------------------------
namespace {
std::mutex g_tune_mu;
std::map<std::string, TuneParams> g_tune;
}  // namespace

std::string problem_key(const ProblemSpec& s)
{
    std::ostringstream os;
    os << "p" << s.prec_bytes << ':' << (int)s.type << ':' << s.dir << ':' << s.inplace << ':' << s.mfma_mode << '|';
    for (const auto& a : s.dims) os << a.n << ',' << a.is << ',' << a.os << ';';
    os << '|';
    for (const auto& a : s.vecs) os << a.n << ',' << a.is << ',' << a.os << ';';
    return os.str();
}

std::string batch_key(const std::vector<BatchItem>& items, int prec, int dir)
{
    uint64_t h = 1469598103934665603ull;  // FNV-1a over the item list
    auto mix = [&](int64_t v) {
        for (int b = 0; b < 8; b++) {
            h ^= (uint64_t)((v >> (8 * b)) & 0xff);
            h *= 1099511628211ull;
        }
    };
    for (const BatchItem& it : items) {
        mix(it.n);
        mix(it.batch);
        mix(it.in_off);
        mix(it.out_off);
        mix(it.dist);
    }
    std::ostringstream os;
    os << "b" << prec << ':' << dir << ':' << items.size() << ':' << std::hex << h;
    return os.str();
}

bool tune_lookup(const std::string& key, TuneParams& out)
{
    std::lock_guard<std::mutex> g(g_tune_mu);
    auto it = g_tune.find(key);
    if (it == g_tune.end()) return false;
    out = it->second;
    return true;
}

void tune_store(const std::string& key, const TuneParams& t)
{
    std::lock_guard<std::mutex> g(g_tune_mu);
    g_tune[key] = t;
}

std::string tune_text(int* entries)
{
    std::lock_guard<std::mutex> g(g_tune_mu);
    std::ostringstream os;
    os << "# fftz tuned plans: key row_t col_c wg_small wg_medium [e=elems] [r=L:r.r.r/L:r.r] [f=f.f.f]\n";
    for (const auto& kv : g_tune) {
        const TuneParams& t = kv.second;
        os << kv.first << ' ' << t.row_t << ' ' << t.col_c << ' ' << t.wg_small << ' ' << t.wg_medium;
        if (t.elems) os << " e=" << t.elems;
        if (!t.radix_for.empty()) {
            os << " r=";
            for (size_t i = 0; i < t.radix_for.size(); i++) {
                os << (i ? "/" : "") << t.radix_for[i].first << ':';
                for (size_t j = 0; j < t.radix_for[i].second.size(); j++)
                    os << (j ? "." : "") << t.radix_for[i].second[j];
            }
        }
        if (!t.split.empty()) {
            os << " f=";
            for (size_t i = 0; i < t.split.size(); i++) os << (i ? "." : "") << t.split[i];
        }
        os << '\n';
    }
    if (entries) *entries = (int)g_tune.size();
    return os.str();
}

// "1.2.3" -> {1, 2, 3}; false on anything but positive integers and dots.
static bool parse_dotted(const std::string& v, std::vector<int64_t>& out)
{
    out.clear();
    size_t i = 0;
    while (i < v.size()) {
        size_t j = v.find('.', i);
        if (j == std::string::npos) j = v.size();
        const std::string tok = v.substr(i, j - i);
        if (tok.empty() || tok.size() > 12 || tok.find_first_not_of("0123456789") != std::string::npos) return false;
        out.push_back(std::stoll(tok));
        if (out.back() <= 0) return false;
        i = j + 1;
        if (j == v.size()) break;
        if (i == v.size()) return false;  // trailing dot
    }
    return !out.empty();
}

// Optional fields of a tuned-cache line: e=8, r=1024:16.8.8/256:16.16, f=256.256.256.
static bool parse_tune_token(const std::string& tok, TuneParams& t)
{
    if (tok.size() < 3 || tok[1] != '=') return false;
    const std::string v = tok.substr(2);
    std::vector<int64_t> nums;
    switch (tok[0]) {
        case 'e':
            if (v != "8" && v != "16") return false;
            t.elems = std::stoi(v);
            return true;
        case 'f':
            if (!parse_dotted(v, nums) || nums.size() < 2 || nums.size() > 3) return false;
            for (int64_t f : nums)
                if (f < 2) return false;
            t.split = nums;
            return true;
        case 'r': {
            size_t i = 0;
            while (i <= v.size()) {
                size_t j = v.find('/', i);
                if (j == std::string::npos) j = v.size();
                const std::string item = v.substr(i, j - i);
                const size_t c = item.find(':');
                if (c == std::string::npos || c == 0) return false;
                const std::string ls = item.substr(0, c);
                if (ls.size() > 9 || ls.find_first_not_of("0123456789") != std::string::npos) return false;
                const int L = std::stoi(ls);
                if (!parse_dotted(item.substr(c + 1), nums)) return false;
                std::vector<int> r(nums.begin(), nums.end());
                if (!radix_order_ok(L, r)) return false;
                t.radix_for.push_back({L, r});
                i = j + 1;
                if (j == v.size()) break;
            }
            return !t.radix_for.empty();
        }
        default:
            return false;
    }
}

int tune_parse(const std::string& text)
{
    // All or nothing: a malformed line leaves the cache untouched.
    std::vector<std::pair<std::string, TuneParams>> got;
    std::istringstream is(text);
    std::string line;
    while (std::getline(is, line)) {
        const size_t b = line.find_first_not_of(" \t\r");
        if (b == std::string::npos || line[b] == '#') continue;
        std::istringstream ls(line);
        std::string key, extra;
        TuneParams t;
        if (!(ls >> key >> t.row_t >> t.col_c >> t.wg_small >> t.wg_medium)) return -1;
        for (int v : {t.row_t, t.col_c, t.wg_small, t.wg_medium})
            if (v < 0 || v > 4096) return -1;
        while (ls >> extra)
            if (!parse_tune_token(extra, t)) return -1;
        got.emplace_back(key, t);
    }
    for (const auto& kv : got) tune_store(kv.first, kv.second);
    return (int)got.size();
}

void tune_clear()
{
    std::lock_guard<std::mutex> g(g_tune_mu);
    g_tune.clear();
}

int tune_export(const char* path)
{
    FILE* f = path ? fopen(path, "w") : nullptr;
    if (!f) return -1;
    int n = 0;
    const std::string text = tune_text(&n);
    const bool ok = fwrite(text.data(), 1, text.size(), f) == text.size();
    return (fclose(f) == 0 && ok) ? n : -1;
}

int tune_import(const char* path)
{
    FILE* f = path ? fopen(path, "r") : nullptr;
    if (!f) return -1;
    std::string text;
    char buf[4096];
    size_t got;
    while ((got = fread(buf, 1, sizeof(buf), f)) > 0) text.append(buf, got);
    fclose(f);
    return tune_parse(text);
}

Plan* plan_create(const ProblemSpec& spec_in, std::string& err, bool dry_run)
{
    Plan* plan = new Plan();
    plan->dry_run = dry_run;
    plan->spec = spec_in;
    ProblemSpec& spec = plan->spec;
    if (spec.tune.empty()) (void)tune_lookup(problem_key(spec), spec.tune);
    if (!dry_run) {
        (void)hipGetDevice(&plan->device);
        (void)device_info();
    }

    // Drop size-1 dims (SHRINK_DIM_RANK, selector/selector.h:194-214) and
    // size-1 batch axes; a zero-length batch axis is a no-op plan
    // (selector/selector.c:1375-1385).
    std::vector<AxisSpec> dims, vecs;
    for (size_t i = 0; i < spec.dims.size(); i++)
        if (spec.dims[i].n != 1 || (i == 0 && spec.type != FftType::C2C)) dims.push_back(spec.dims[i]);
    if (dims.empty()) dims.push_back({1, 1, 1});
    for (auto& v : spec.vecs) {
        if (v.n == 0) plan->noop = true;
        if (v.n > 1) vecs.push_back(v);
    }
    // extents for host staging
    if (spec.type == FftType::C2C) {
        plan->in_extent_bytes = extent(spec.dims, spec.vecs, true, -1) * 2 * spec.prec_bytes;
        plan->out_extent_bytes = extent(spec.dims, spec.vecs, false, -1) * 2 * spec.prec_bytes;
    } else if (spec.type == FftType::R2C) {
        plan->in_extent_bytes = extent(spec.dims, spec.vecs, true, -1) * spec.prec_bytes;
        plan->out_extent_bytes = extent(spec.dims, spec.vecs, false, spec.dims[0].n / 2 + 1) * 2 * spec.prec_bytes;
    } else {
        plan->in_extent_bytes = extent(spec.dims, spec.vecs, true, spec.dims[0].n / 2 + 1) * 2 * spec.prec_bytes;
        plan->out_extent_bytes = extent(spec.dims, spec.vecs, false, -1) * spec.prec_bytes;
    }
    plan->dense_out = dense(spec.dims, spec.vecs, spec.type == FftType::R2C ? spec.dims[0].n / 2 + 1 : -1);
    if (plan->noop) return plan;

    // algorithmic flop count (5 N log2 N for C2C, 2.5 N log2 N for real)
    double ntot = 1.0, nb = 1.0;
    for (auto& d : spec.dims) ntot *= (double)d.n;
    for (auto& v : spec.vecs) nb *= (double)v.n;
    plan->flops = (spec.type == FftType::C2C ? 5.0 : 2.5) * ntot * std::log2(std::max(ntot, 2.0)) * nb;

    TableBuilder tb{plan->host_tables};
    bool ok;
    if (spec.type == FftType::C2C)
        ok = plan_c2c(plan, tb, dims, vecs, err);
    else
        ok = plan_real(plan, tb, dims, vecs, err);
    if (!ok) {
        delete plan;
        return nullptr;
    }
    // results that a later launch reads (N-D passes in place on the output)
    // stay in the caches
    for (size_t i = 0; i < plan->launches.size(); i++)
        for (size_t j = i + 1; j < plan->launches.size(); j++)
            if (plan->launches[j].in_role == plan->launches[i].out_role) plan->launches[i].d.flags &= ~kNtStore;
    if (dry_run) return plan;
    // upload tables and resolve pointers
    if (!plan->host_tables.empty()) {
        if (hipMalloc(&plan->tables, plan->host_tables.size()) != hipSuccess ||
            hipMemcpy(plan->tables, plan->host_tables.data(), plan->host_tables.size(), hipMemcpyHostToDevice) !=
                hipSuccess) {
            err = "device allocation for plan tables failed";
            if (plan->tables) (void)hipFree(plan->tables);
            delete plan;
            return nullptr;
        }
    }
    char* base = (char*)plan->tables;
    for (auto& ln : plan->launches) {
        if (ln.stw_off >= 0) ln.d.stw = base + ln.stw_off;
        if (ln.tw4_off >= 0) ln.d.tw4 = base + ln.tw4_off;
        if (ln.chirp_off >= 0) ln.d.chirp = base + ln.chirp_off;
        if (ln.spec_off >= 0) ln.d.spec = base + ln.spec_off;
        if (ln.rtw_off >= 0) ln.d.rtw = base + ln.rtw_off;
        if (ln.frag_off >= 0) ln.frag = reinterpret_cast<const float*>(base + ln.frag_off);
    }
    plan->host_tables.clear();
    plan->host_tables.shrink_to_fit();
    plan->use_graph = env_int("FFTZ_GRAPH", 0) != 0;
    return plan;
}

static std::string batch_json(const Plan* p)
{
    std::ostringstream os;
    os << "{\"batch\":1,\"prec\":" << p->spec.prec_bytes << ",\"in_extent_bytes\":" << p->in_extent_bytes
       << ",\"out_extent_bytes\":" << p->out_extent_bytes << ",\"sizes\":[";
    const PassDesc* hd = p->host_tables.empty()
                             ? nullptr
                             : reinterpret_cast<const PassDesc*>(p->host_tables.data() + p->descs_off);
    size_t nsz = 0;
    for (const BatchClass& bc : p->bclasses) {
        const BatchTile* t = hd ? reinterpret_cast<const BatchTile*>(p->host_tables.data() + bc.tiles_off) : nullptr;
        for (int i = 0; hd && i < bc.ntiles; i++) nsz = std::max(nsz, (size_t)t[i].desc + 1);
    }
    for (size_t i = 0; hd && i < nsz; i++) {
        const PassDesc& d = hd[i];
        os << (i ? "," : "") << "{\"L\":" << d.L << ",\"nvalid\":" << d.nvalid_in << ",\"C\":" << d.C
           << ",\"TL\":" << d.TL << ",\"LP\":" << d.LP << ",\"flags\":" << d.flags << ",\"radix\":[";
        for (int s = 0; s < d.nst; s++) os << (s ? "," : "") << d.radix[s];
        os << "]}";
    }
    os << "],\"classes\":[";
    for (size_t c = 0; c < p->bclasses.size(); c++) {
        const BatchClass& bc = p->bclasses[c];
        // complex values of a line per thread: the most in this class
        const BatchTile* q = hd ? reinterpret_cast<const BatchTile*>(p->host_tables.data() + bc.tiles_off) : nullptr;
        int E = 0;
        for (int i = 0; q && i < bc.ntiles; i++) {
            const PassDesc& d = hd[q[i].desc];
            E = std::max(E, (d.L + d.TL - 1) / d.TL);
        }
        os << (c ? "," : "") << "{\"E\":" << E << ",\"nt\":" << (bc.nt ? 1 : 0) << ",\"maxt\":" << bc.maxt << ",\"lds\":" << bc.lds_bytes
           << ",\"grid\":" << bc.grid << ",\"tiles\":[";
        for (int i = 0; q && i < bc.ntiles; i++)
            os << (i ? "," : "") << "[" << q[i].desc << "," << q[i].nlines << "," << q[i].bluestein << ","
               << q[i].in_off << "," << q[i].out_off << "," << q[i].dist << "]";
        os << "]}";
    }
    os << "]}";
    return os.str();
}

static KernelKind pass_kind(const Launch& ln);

// Kernel form of a launch: the fixed-length and matrix-core kernels, or the generic
// kernel's (KernelKind).
static const char* form_name(const Launch& ln)
{
    if (ln.mfma) return "mfma";
    if (ln.fixed) return "fixed";
    switch (pass_kind(ln)) {
        case KernelKind::Bluestein: return "bluestein";
        case KernelKind::Real: return "real";
        case KernelKind::RealWide: return "real_wide";
        default: return "pass";
    }
}

std::string plan_json(const Plan* p)
{
    if (p->is_batch) return batch_json(p);
    std::ostringstream os;
    os << "{\"noop\":" << (p->noop ? 1 : 0) << ",\"work_bytes\":" << p->work_bytes
       << ",\"in_extent_bytes\":" << p->in_extent_bytes << ",\"out_extent_bytes\":" << p->out_extent_bytes
       << ",\"prec\":" << p->spec.prec_bytes << ",\"launches\":[";
    bool first = true;
    for (const Launch& ln : p->launches) {
        const PassDesc& d = ln.d;
        os << (first ? "" : ",") << "{\"kind\":\"" << (ln.kind == KernelKind::Bluestein ? "bluestein" : "pass")
           << "\",\"L\":" << d.L << ",\"nvalid_in\":" << d.nvalid_in << ",\"nvalid_out\":" << d.nvalid_out
           << ",\"ies\":" << d.ies << ",\"oes\":" << d.oes << ",\"ils\":[" << d.ils[0] << "," << d.ils[1]
           << "," << d.ils[2] << "],\"ols\":[" << d.ols[0] << "," << d.ols[1] << "," << d.ols[2]
           << "],\"nlines\":" << d.nlines << ",\"ln0\":" << d.ln0.d << ",\"ln1\":" << d.ln1.d
           << ",\"flags\":" << d.flags << ",\"C\":" << d.C << ",\"TL\":" << d.TL << ",\"LP\":" << d.LP
           << ",\"vrow\":" << d.vrow.d << ",\"maxt\":" << ln.maxt
           << ",\"E\":" << ln.E << ",\"fixed\":" << (ln.fixed ? 1 : 0) << ",\"mfma\":" << ln.mfma << ",\"grid\":" << ln.grid << ",\"block\":" << ln.block
           << ",\"rad\":" << ln.rad << ",\"form\":\"" << form_name(ln) << "\",\"split\":" << (ln.split ? 1 : 0)
           << ",\"nt\":" << ((d.flags & kNtStore) ? 1 : 0) << ",\"lds\":" << ln.lds_bytes
           << ",\"lds_launched\":" << ln.launched_lds() << ",\"in_role\":" << (int)ln.in_role
           << ",\"out_role\":" << (int)ln.out_role << ",\"in_off\":" << ln.in_off_bytes
           << ",\"out_off\":" << ln.out_off_bytes << ",\"tw4_n\":" << d.tw4_n << ",\"nchirp\":" << d.nchirp
           << ",\"gin\":[" << d.gin[0] << "," << d.gin[1] << "," << d.gin[2] << "," << d.gin[3] << "],\"gout\":["
           << d.gout[0] << "," << d.gout[1] << "," << d.gout[2] << "," << d.gout[3] << "],\"gin_base\":" << d.gin_base
           << ",\"gout_base\":" << d.gout_base << ",\"radix\":[";
        for (int s = 0; s < d.nst; s++) os << (s ? "," : "") << d.radix[s];
        os << "],\"ls\":[";
        for (int s = 0, ls = 1; s < d.nst; ls *= d.radix[s++]) os << (s ? "," : "") << ls;
        os << "]}";
        first = false;
    }
    os << "]}";
    return os.str();
}

static void slot_free(Slot* s)
{
    if (s->graph) (void)hipGraphExecDestroy(s->graph);
    if (s->work) (void)hipFree(s->work);
    if (s->stage_in) (void)hipFree(s->stage_in);
    if (s->stage_out) (void)hipFree(s->stage_out);
    if (s->counters) (void)hipFree(s->counters);
    if (s->stream) (void)hipStreamDestroy(s->stream);
    delete s;
}

void plan_destroy(Plan* p)
{
    if (!p) return;
    for (Slot* s : p->slots) {
        if (s->stream) (void)hipStreamSynchronize(s->stream);
        slot_free(s);
    }
    if (p->tables) (void)hipFree(p->tables);
    for (hipEvent_t e : p->prof_events) (void)hipEventDestroy(e);
    for (hipEvent_t e : p->prof_pool) (void)hipEventDestroy(e);
    delete p;
}

Slot* plan_acquire_slot(Plan* p, hipError_t* err)
{
    std::lock_guard<std::mutex> g(p->mu);
    *err = hipSuccess;
    for (Slot* s : p->slots)
        if (!s->busy) {
            s->busy = true;
            return s;
        }
    Slot* s = new Slot();
    // a blocking stream: a synchronous execute is ordered after work still
    // pending on the null stream (where most callers produced their buffers)
    hipError_t e = hipStreamCreateWithFlags(&s->stream, hipStreamDefault);
    if (e == hipSuccess && p->work_bytes) {
        e = hipMalloc(&s->work, p->work_bytes);
        s->work_bytes = p->work_bytes;
    }
    if (e == hipSuccess && p->is_batch) e = hipMalloc((void**)&s->counters, 64);
    if (e != hipSuccess) {
        *err = e;
        slot_free(s);
        return nullptr;
    }
    s->busy = true;
    p->slots.push_back(s);
    return s;
}

void plan_release_slot(Plan* p, Slot* s)
{
    std::lock_guard<std::mutex> g(p->mu);
    s->busy = false;
}

static hipError_t record_prof(Plan* p, hipStream_t stream)
{
    hipEvent_t ev;
    {
        std::lock_guard<std::mutex> g(p->mu);
        if (p->prof_pool.empty()) {
            hipError_t e = hipEventCreate(&ev);
            if (e != hipSuccess) return e;
        } else {
            ev = p->prof_pool.back();
            p->prof_pool.pop_back();
        }
        p->prof_events.push_back(ev);
    }
    return hipEventRecord(ev, stream);
}

// Launches of one execute.  work: the work buffer (four-step and multi-axis
// C2R intermediates), counters: the uneven batch's queue counters; prof:
// record timing events (which allocates them on first use).
static hipError_t launch_batch(Plan* p, unsigned* counters, const void* in, void* out, hipStream_t stream,
                               bool prof)
{
    // counters are cleared by a kernel (not a memset node) so the sequence
    // can be captured in a graph and replayed
    int nc = (int)p->bclasses.size();
    void* rargs[] = {&counters, &nc};
    hipError_t e = hipLaunchKernel(kernel_symbol_reset(), dim3(1), dim3(64), rargs, 0, stream);
    if (e != hipSuccess) return e;
    if (prof && (e = record_prof(p, stream)) != hipSuccess) return e;
    const char* base = (const char*)p->tables;
    for (size_t c = 0; c < p->bclasses.size(); c++) {
        const BatchClass& bc = p->bclasses[c];
        if (bc.ntiles > 0) {
            BatchArgs a;
            a.descs = reinterpret_cast<const PassDesc*>(base + p->descs_off);
            a.tiles = reinterpret_cast<const BatchTile*>(base + bc.tiles_off);
            a.ntiles = bc.ntiles;
            a.counter = counters + c;
            a.in = in;
            a.out = out;
            void* args[] = {&a};
            e = hipLaunchKernel(kernel_symbol_batch(p->spec.prec_bytes, (int)c, bc.nt), dim3(bc.grid),
                                dim3(bc.maxt), args, bc.lds_bytes, stream);
            if (e != hipSuccess) return e;
        }
        if (prof && (e = record_prof(p, stream)) != hipSuccess) return e;
    }
    return hipGetLastError();
}

static KernelKind pass_kind(const Launch& ln)
{
    const PassDesc& d = ln.d;
    if (ln.kind != KernelKind::Pass || !(d.flags & kRealFlags)) return ln.kind;
    const int pair = (d.flags & kR2CPost) && d.nst ? d.radix[d.nst - 1] : (d.flags & kC2RPre) && d.nst ? d.radix[0] : 1;
    return pair > 10 ? KernelKind::RealWide : KernelKind::Real;
}

static hipError_t launch_all(Plan* p, void* work, unsigned* counters, const void* in, void* out, hipStream_t stream,
                             bool prof)
{
    if (p->is_batch) return launch_batch(p, counters, in, out, stream, prof);
    if (prof) {
        hipError_t e = record_prof(p, stream);
        if (e != hipSuccess) return e;
    }
    for (const Launch& ln : p->launches) {
        PassDesc d = ln.d;
        auto role_ptr = [&](Role r) -> char* {
            switch (r) {
                case Role::In: return (char*)in;
                case Role::Out: return (char*)out;
                default: return (char*)work;
            }
        };
        d.in = role_ptr(ln.in_role) + ln.in_off_bytes;
        d.out = role_ptr(ln.out_role) + ln.out_off_bytes;
        const float* frag = ln.frag;
        void* args[] = {&d, &frag};
        const void* fn = ln.mfma ? kernel_symbol_mfma(ln.mfma, ln.d.L, ln.mfma_nb)
                         : ln.fixed ? kernel_symbol_fixed(p->spec.prec_bytes, ln.d.L, ln.maxt, ln.split,
                                                          (d.flags & kNtStore) != 0)
                                    : kernel_symbol(pass_kind(ln), p->spec.prec_bytes, ln.rad,
                                                    (d.flags & kNtStore) != 0, ln.maxt);
        hipError_t e = hipLaunchKernel(fn, dim3(ln.grid), dim3(ln.block), args,
                                       ln.launched_lds(), stream);
        if (e != hipSuccess) return e;
        if (prof) {
            e = record_prof(p, stream);
            if (e != hipSuccess) return e;
        }
    }
    return hipGetLastError();
}

hipError_t plan_enqueue_scratch(Plan* p, void* work, unsigned* counters, const void* in, void* out,
                                hipStream_t stream)
{
    if (p->noop) return hipSuccess;
    return launch_all(p, work, counters, in, out, stream, false);
}

int plan_profile_read(Plan* p, float* ms, int cap)
{
    std::vector<hipEvent_t> evs;
    {
        std::lock_guard<std::mutex> g(p->mu);
        evs.swap(p->prof_events);
    }
    const size_t per = (p->is_batch ? p->bclasses.size() : p->launches.size()) + 1;  // events per execute
    int n = 0;
    for (size_t base = 0; base + per <= evs.size(); base += per) {
        for (size_t i = 0; i + 1 < per; i++) {
            float t = 0.f;
            if (hipEventSynchronize(evs[base + i + 1]) != hipSuccess ||
                hipEventElapsedTime(&t, evs[base + i], evs[base + i + 1]) != hipSuccess)
                t = -1.f;
            if (ms && n < cap) ms[n] = t;
            n++;
        }
    }
    std::lock_guard<std::mutex> g(p->mu);
    for (hipEvent_t e : evs) p->prof_pool.push_back(e);
    return n;
}

hipError_t plan_enqueue(Plan* p, Slot* s, const void* in, void* out, hipStream_t stream)
{
    if (p->noop) return hipSuccess;
    if (!p->use_graph || p->profile) return launch_all(p, s->work, s->counters, in, out, stream, p->profile);
    // One hipGraph per (slot, in, out): captured once, replayed afterwards.
    if (!s->graph || s->graph_in != in || s->graph_out != out) {
        if (s->graph) {
            (void)hipGraphExecDestroy(s->graph);
            s->graph = nullptr;
        }
        hipGraph_t g;
        hipError_t e = hipStreamBeginCapture(s->stream, hipStreamCaptureModeThreadLocal);
        if (e != hipSuccess) return e;
        e = launch_all(p, s->work, s->counters, in, out, s->stream, false);
        hipError_t e2 = hipStreamEndCapture(s->stream, &g);
        if (e != hipSuccess) return e;
        if (e2 != hipSuccess) return e2;
        e = hipGraphInstantiate(&s->graph, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e != hipSuccess) return e;
        s->graph_in = in;
        s->graph_out = out;
    }
    return hipGraphLaunch(s->graph, stream);
}

}  // namespace fftz

namespace fftz {

double plan_time(Plan* p, const void* in, void* out, int reps)
{
    hipError_t e = hipSuccess;
    Slot* s = plan_acquire_slot(p, &e);
    if (!s) return -1.0;
    hipEvent_t a = nullptr, b = nullptr;
    double ms = -1.0;
    if (hipEventCreate(&a) == hipSuccess && hipEventCreate(&b) == hipSuccess) {
        e = plan_enqueue(p, s, in, out, s->stream);  // warm (and graph capture)
        if (e == hipSuccess) e = hipEventRecord(a, s->stream);
        for (int r = 0; r < reps && e == hipSuccess; r++) e = plan_enqueue(p, s, in, out, s->stream);
        if (e == hipSuccess) e = hipEventRecord(b, s->stream);
        if (e == hipSuccess) e = hipEventSynchronize(b);
        float t = 0.f;
        if (e == hipSuccess && hipEventElapsedTime(&t, a, b) == hipSuccess) ms = (double)t / reps;
    }
    if (a) (void)hipEventDestroy(a);
    if (b) (void)hipEventDestroy(b);
    if (e != hipSuccess) (void)hipGetLastError();
    plan_release_slot(p, s);
    return ms;
}

}  // namespace fftz
