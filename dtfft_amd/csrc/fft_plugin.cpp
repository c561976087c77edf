// FFT executor plugin: batched 1D / 2D C2C (and R2C / C2R) stages on gfx950.
//
// Drop-in for the cuFFT / VkFFT executors behind abstract_executor
// (src/dtfft_abstract_executor.F90:47-112; cuFFT: src/interfaces/fft/cufft/
// dtfft_executor_cufft_m.F90:52-125).  create receives exactly what
// abstract_executor%create computes from the pencils (:115-216): fft_rank, the sizes
// in FFTW row-major order, inembed/onembed, idist/odist and how_many, unit stride.
//
// Each 1D stage is one launch of the Stockham kernel in device/fft.hip, compiled by
// hipRTC for its length.  Radix schedule, threads per line, lines per block and LDS
// padding come from a heuristic or, at effort >= MEASURE, from timing the candidates
// on the device (the project's replacement for dtfft_nvrtc_block_optimizer).
#include <algorithm>
#include <numeric>
#include <array>
#include <cmath>
#include <functional>

#include "internal.h"

namespace dtfft_hip {

// Primes above 13 that the kernels have as radices of their own (bfly in device/fft.hip).
static const int kLargePrimes[] = {17, 19, 23, 29, 31, 37, 41, 43, 47, 53, 59, 61};
static bool large_prime(int r) {
    return std::find(std::begin(kLargePrimes), std::end(kLargePrimes), r) != std::end(kLargePrimes);
}

// ---- schedules ----------------------------------------------------------------------
bool prime_schedule(int n, std::vector<int>& radices) {
    radices.clear();
    if (n < 1) return false;
    if (n == 1) { radices.push_back(1); return true; }
    int a = 0, m = n;
    while (m % 2 == 0) { m /= 2; a++; }
    // power-of-two part: fewest passes with radices 16/8/4/2
    if (a > 0) {
        int passes = (a + 3) / 4;
        std::vector<int> e(passes, a / passes);
        for (int i = 0; i < a % passes; i++) e[i]++;
        for (int x : e) radices.push_back(1 << x);
    }
    const int primes[] = {3, 5, 7, 11, 13};
    for (int p : primes)
        while (m % p == 0) { radices.push_back(p); m /= p; }
    if (m != 1) return false;
    if (radices.size() > 10) return false;  // dtfft::sched holds up to 10 passes
    return true;
}

// Share of thread-rounds that do work when a line's passes run on tpl threads, inverted: 1 when
// every pass fills its rounds of butterflies, 2 when half of the threads wait.
static double idle_factor(const std::vector<int>& radices, int n, int tpl) {
    double sum = 0;
    for (int r : radices) sum += (double)((n / r + tpl - 1) / tpl) * tpl * r;
    return sum / ((double)n * (double)radices.size());
}

// Threads per line with the least idle rounds: the butterflies of one of the passes.
static int best_tpl(const std::vector<int>& radices, int n) {
    int best = 1;
    double bf = 1e30;
    for (int r : radices) {
        const int t = n / r;
        const double f = idle_factor(radices, n, t);
        if (f < bf - 1e-9 || (f < bf + 1e-9 && t > best)) { bf = f; best = t; }
    }
    return best;
}

// The radix schedule of n: fewest passes of radices up to 16 -- but two for 6 to 16, where one
// thread would hold a whole line (16 = 4 4 on four threads 78 us per 256 MB of FP32 rows, 135 us
// as one radix 16) -- then the least idle rounds and the smallest radix.
bool factorize(int n, std::vector<int>& radices) {
    if (!prime_schedule(n, radices)) return false;  // a prime above 13
    if (n == 1) return true;
    static std::mutex mu;
    static std::map<int, std::vector<int>> known;  // plans ask for a few lengths many times
    {
        std::lock_guard<std::mutex> lk(mu);
        auto it = known.find(n);
        if (it != known.end()) { radices = it->second; return true; }
    }
    std::vector<int> cur, best;
    double cost = 1e30;
    std::function<void(int, int)> rec = [&](int m, int hi) {
        if (m == 1) {
            double f = 100.0 * (double)cur.size() + 16.0 * idle_factor(cur, n, best_tpl(cur, n)) + cur[0];
            for (int r : cur) f += 0.01 * r;
            if (n >= 6 && cur.size() == 1) f += 200.0;
            if (f < cost) { cost = f; best = cur; }
            return;
        }
        if (cur.size() >= 10 || (!best.empty() && cur.size() >= std::max<size_t>(2, best.size()))) return;
        for (int r = std::min(hi, 16); r >= 2; r--)
            if (m % r == 0) {
                cur.push_back(r);
                rec(m / r, r);
                cur.pop_back();
            }
    };
    rec(n, 16);
    if (!best.empty()) radices = best;
    std::lock_guard<std::mutex> lk(mu);
    known[n] = radices;
    return true;
}

// Schedules of lengths with prime factors above 13 that have radices of their own, those first:
// the first pass needs no twiddles, 36 of them per butterfly of 37.  Only lengths that the
// Bluestein form would take (its work line fits the LDS) and only up to max_prime.
bool large_schedule(int n, bool dbl, int max_prime, std::vector<int>& radices) {
    radices.clear();
    if (2 * (int64_t)n - 1 > (int64_t)(160 * 1024 / (dbl ? 16 : 8))) return false;
    int m = n;
    std::vector<int> rest;
    for (int p : kLargePrimes)
        while (p <= max_prime && m % p == 0) { radices.insert(radices.begin(), p); m /= p; }
    if (radices.empty() || !factorize(m, rest)) return false;
    if (m <= 16) rest = {m};
    if (m > 1) radices.insert(radices.end(), rest.begin(), rest.end());
    return radices.size() <= 10;
}

std::string fft_config::expr() const {
    if (any) {
        // the schedule, and its radices in reverse for the second transform of Bluestein's form
        std::string s = std::string("fft_any_kernel<") + (dbl ? "double" : "float");
        const std::vector<int> rev(radices.rbegin(), radices.rend());
        for (const auto* r : {&radices, &rev}) {
            s += ", dtfft::sched<" + std::to_string(n);
            for (int x : *r) s += ", " + std::to_string(x);
            s += ">";
        }
        s += ", " + std::to_string(tpl) + ", " + std::to_string(lpb) + ", " + std::to_string(pad) + ", " +
             std::to_string(kind);
        for (bool b : {chirp, in_cols, out_cols}) s += b ? ", true" : ", false";
        return s + ">";
    }
    if (dma && kind == 2) {
        std::string s = std::string(dma == 1 ? "fft_c2r_dma2_kernel<" : "fft_c2r_dma_kernel<") +
                        (dbl ? "double" : "float") + ", dtfft::sched<" + std::to_string(n);
        for (int r : radices) s += ", " + std::to_string(r);
        s += ">, " + std::to_string(tpl) + ", " + std::to_string(lpb) + ", " + std::to_string(pad);
        if (dma == 1) return s + ">";
        return s + (twl ? ", true>" : ", false>");
    }
    if (dma) {
        std::string s = std::string(dma == 2 ? "fft_cols_dma1_kernel<" : "fft_cols_dma_kernel<") +
                        (dbl ? "double" : "float") + ", dtfft::sched<" + std::to_string(n);
        for (int r : radices) s += ", " + std::to_string(r);
        return s + ">, " + std::to_string(tpl) + ", " + std::to_string(lpb) + ", " + std::to_string(pad) +
               (out_cols ? ", true>" : ">");
    }
    std::string s = kind == 0 ? "fft_c2c_kernel<" : (kind == 1 ? "fft_r2c_kernel<" : "fft_c2r_kernel<");
    s += dbl ? "double" : "float";
    s += ", dtfft::sched<" + std::to_string(n);
    for (int r : radices) s += ", " + std::to_string(r);
    s += ">, " + std::to_string(tpl) + ", " + std::to_string(lpb) + ", ";
    if (kind == 0) s += std::string(in_cols ? "true" : "false") + ", " + (out_cols ? "true" : "false") + ", ";
    s += std::to_string(pad);
    if (kind == 0 && (seg > 0 || twl || oseg > 0 || staged)) s += ", " + std::to_string(seg);
    if (kind == 0 && (twl || oseg > 0 || staged)) s += twl ? ", true" : ", false";
    if (kind == 0 && (oseg > 0 || staged)) s += ", " + std::to_string(oseg);
    if (kind == 0 && staged) s += ", true";
    if (kind == 1 && oseg > 0) s += ", " + std::to_string(oseg);
    if (kind == 2 && (in_cols || twl)) s += in_cols ? ", true" : ", false";
    if (kind == 2 && twl) s += ", true";
    s += ">";
    return s;
}

static int elem_bytes(bool dbl) { return dbl ? 16 : 8; }
static const size_t kMaxLds = 160 * 1024;

// LDS bytes of fft_cols_dma_kernel: two tile buffers (load layout of 1152-byte groups of 8
// rows, or the line-major staging layout, whichever is larger) and the twiddle table.
static size_t lds_dma(const fft_config& c) {
    const size_t es = (size_t)elem_bytes(c.dbl);
    if (c.kind == 2) {
        // fft_c2r_dma(2)_kernel: buffers of the n + 1 input rows (the last group unpadded) or the
        // staging layout; dma 1 (double buffer): both twiddle tables in LDS (the FFT table and
        // the untangling half of n / 2 + 1 entries); dma 2: the FFT table when twl is set
        const size_t groups = (size_t)((c.n + 1 + 7) / 8);
        const size_t load = (groups - 1) * 1152 + ((size_t)(c.n + 1) - 8 * (groups - 1)) * 128;
        const size_t stage = (size_t)c.lpb * (size_t)((c.n + c.pad) | 1) * es;
        size_t tw = 0, L = 1;
        for (int r : c.radices) { tw += L * (size_t)(r - 1); L *= (size_t)r; }
        const size_t twb = std::max<size_t>(1, tw) * 16 + 16;
        if (c.dma == 1) return 2 * std::max(load, stage) + twb + (size_t)(c.n / 2 + 1) * 16 + 16;
        return std::max(load, stage) + (c.twl ? twb : 0);
    }
    const size_t groups = (size_t)((c.n + 7) / 8);
    const size_t load = (groups - 1) * 1152 + ((size_t)c.n - 8 * (groups - 1)) * 128;
    const size_t stage = (size_t)c.lpb * (size_t)((c.n + c.pad) | 1) * es;
    size_t tw = 0, L = 1;
    for (int r : c.radices) { tw += L * (size_t)(r - 1); L *= (size_t)r; }
    return (c.dma == 2 ? 1 : 2) * std::max(load, stage) + std::max<size_t>(1, tw) * 16;
}

// The LDS-DMA kernels hold radices up to 16: a large prime's butterfly needs bfly_large.
static bool dma_radices(const fft_config& c) {
    return std::all_of(c.radices.begin(), c.radices.end(), [](int r) { return r <= 16; });
}

// Whether a fused column-in C2R stage can use fft_c2r_dma_kernel.
static bool c2r_dma_ok(const fft_config& c, const lines_desc& d) {
    const int64_t es = elem_bytes(c.dbl);
    return dma_radices(c) && c.kind == 2 && (c.dma == 1 || c.dma == 2) && c.n > 1 && c.n % 8 == 0 && c.lpb * es == 128 && (c.tpl * c.lpb) % 64 == 0 &&
           c.tpl * c.lpb <= 1024 && d.in_ls == 1 && d.out_ns == 1 && d.nl % c.lpb == 0 && (d.in_ns * es) % 16 == 0 &&
           (d.in_bs * es) % 16 == 0 && lds_dma(c) <= kMaxLds;
}

bool dma_ok(const fft_config& c, const lines_desc& d) {
    if (c.kind == 2) return c2r_dma_ok(c, d);
    const int64_t es = elem_bytes(c.dbl);
    const bool out_ok = c.out_cols ? (d.out_ls == 1 && (d.out_ns * es) % 16 == 0 && (d.out_bs * es) % 16 == 0)
                                   : d.out_ns == 1;
    return dma_radices(c) && c.kind == 0 && c.in_cols && c.seg == 0 && c.n > 1 && c.lpb * es == 128 &&
           (c.tpl * c.lpb) % 64 == 0 && c.tpl * c.lpb <= 1024 && d.in_ls == 1 && out_ok && (d.nl * es) % 16 == 0 &&
           (d.in_ns * es) % 16 == 0 && (d.in_bs * es) % 16 == 0 && lds_dma(c) <= kMaxLds;
}

// LDS line stride of fft_tile (device/fft.hip): n + pad, or with pad 2 / 3 one spare slot per
// 16 elements plus (pad & 1), made odd.
static size_t lds_line(int n, int pad) {
    return pad >= 2 ? (size_t)((n + (n >> 4) + (pad & 1)) | 1) : (size_t)(n + pad);
}

// Entries of the schedule's twiddle table: sum over passes of L_p * (R_p - 1).
static size_t tw_entries(const fft_config& c) {
    size_t tw = 0, L = 1;
    for (int r : c.radices) { tw += L * (size_t)(r - 1); L *= (size_t)r; }
    return tw;
}

size_t fft_lds_bytes(const fft_config& c) {
    if (c.dma) return lds_dma(c);
    if (c.any) return (size_t)c.lpb * lds_line(c.n, c.pad) * elem_bytes(c.dbl);
    size_t b = (size_t)c.lpb * lds_line(c.n, c.pad) * elem_bytes(c.dbl);
    if (c.twl) {
        // the tables are separate __shared__ arrays of 16-byte entries (FP32 hi+lo pairs or
        // FP64 complex); 16 bytes of slack each for their alignment
        b += std::max<size_t>(1, tw_entries(c)) * 16 + 16;
        if (c.kind == 2) b += (size_t)(c.n + 1) * 16 + 16;  // C2R untangling table, M + 1 entries
    }
    return b;
}

static bool valid(const fft_config& c) {
    const int threads = c.tpl * c.lpb;
    if (threads < 1 || threads > 1024) return false;
    if (fft_lds_bytes(c) > kMaxLds) return false;
    return true;
}

// Whether two blocks of the kernel fit the LDS of a CU.
static bool two_blocks(const fft_config& c) { return 2 * fft_lds_bytes(c) <= kMaxLds; }

void apply_twl(fft_config& c, const lines_desc& d, int mode) {
    c.twl = 0;
    // the LDS-DMA column kernels keep their twiddles in LDS anyway; R2C rows have no such form
    if (mode == 0 || c.dma || c.any || c.kind == 1 || c.n < 2) return;
    const int64_t ntiles = ((d.nl + c.lpb - 1) / c.lpb) * d.nb;
    bool want = mode >= 2;
    if (mode == 1) {
        // Default rule, measured on MI355X.  Long FP32 rows (n > 1024, plain or fused
        // unpack+FFT): the table (n - 1 entries of 16 bytes) otherwise shares the L1 cache with
        // the tile (us per 2 GiB, global / LDS table: 1280 points 508 / 441, 2048 points 468 / 406,
        // 3200 points 567 / 490).  At n = 512 and 1024 the one-tile-per-block launch stays faster
        // (384 against 412 us, 398 against 528), and where tile and table leave room for one block
        // per CU only (3600 points 573 / 745, 4096 points 522 / 722).  FP32
        // column-in passes without LDS-DMA (e.g. 513 lines per row, the complex X pencil of an
        // R2C plan) run one 1024-thread block per CU anyway, so persistence costs no occupancy:
        // 1024 x 512 x 256 R2C's X->Y pass went from 325 to 276 us.  FP64 measured no gain.
        const bool rows = c.kind == 0 && !c.in_cols && !c.out_cols;
        const bool cols = c.kind == 0 && c.in_cols && c.seg == 0;
        fft_config t = c;
        t.twl = 1;
        want = !c.dbl && ntiles >= 2048 && ((rows && c.n > 1024 && two_blocks(t)) || cols);
    }
    if (!want) return;
    c.twl = 1;
    if (!valid(c)) c.twl = 0;  // tile + tables over the LDS budget: global twiddles
}

// Schedule and threads per line of n for `points` elements per thread.  Up to two passes: the
// largest radix first and n / rmin threads, one butterfly each in the second pass (84 = 12 7 on
// 12 threads 216 us per GiB of FP32 rows, on 7 threads 483; column tiles 192 against 238).  More
// passes: of the schedules of fewest passes, the one with the least idle rounds on the smallest
// power of two (16 at least) of threads that leaves at most `points` elements to each, radices
// descending: whole waves then hold whole lines (384 FP32 columns: 12 8 4 on 16 threads 226 us,
// 8 8 6 on 48 285 us).
void pick_schedule(int n, int points, std::vector<int>& radices, int& tpl) {
    if (!factorize(n, radices)) return;
    tpl = 1;
    if (radices.size() == 1) return;
    if (radices.size() == 2) { tpl = n / radices[1]; return; }
    tpl = 16;
    while (n > tpl * points) tpl *= 2;
    static std::mutex mu;
    static std::map<std::pair<int, int>, std::vector<int>> known;  // (n, tpl)
    {
        std::lock_guard<std::mutex> lk(mu);
        auto it = known.find({n, tpl});
        if (it != known.end()) { radices = it->second; return; }
    }
    const size_t np = radices.size();
    std::vector<int> cur;
    double best = 1e30;
    std::function<void(int, int)> rec = [&](int m, int hi) {
        if (m == 1) {
            double f = idle_factor(cur, n, tpl);
            for (int r : cur) f += 1e-4 * r;  // equal otherwise: the smaller radices
            if (cur.size() == np && f < best) { best = f; radices = cur; }
            return;
        }
        if (cur.size() >= np) return;
        for (int r = std::min(hi, 16); r >= 2; r--)
            if (m % r == 0) {
                cur.push_back(r);
                rec(m / r, r);
                cur.pop_back();
            }
    };
    rec(n, 16);
    std::lock_guard<std::mutex> lk(mu);
    known[{n, tpl}] = radices;
}

// n as four radices up to 10, as equal as they come: the passes of long rows whose three passes of up
// to 16 hold more registers per thread than leave enough waves (rows, us per 2 GiB, three / four passes:
// 1280 points FP32 513 / 441, FP64 452 / 396; 1536 points FP32 469 / 447, FP64 424 / 378; 2560 points
// FP32 534 / 467; 4096 points FP32 588 / 522, FP64 416 / 399).
static bool four_passes(int n, std::vector<int>& radices) {
    int sum = 1 << 30;
    for (int a = 10; a >= 2; a--)
        for (int b = a; b >= 2; b--)
            for (int e = b; e >= 2; e--) {
                if (n % (a * b * e) != 0) continue;
                const int f = n / (a * b * e);
                if (f < 2 || f > e || a + b + e + f >= sum) continue;
                sum = a + b + e + f;
                radices = {a, b, e, f};
            }
    return sum < 1 << 30;
}

fft_config default_fft_config(int n, bool dbl, bool in_cols, bool out_cols, int64_t lines, int64_t nl) {
    fft_config c;
    c.n = n; c.dbl = dbl; c.in_cols = in_cols; c.out_cols = out_cols;
    const bool cols = in_cols || out_cols;
    const int es = elem_bytes(dbl);
    // Launches that would not give every CU two tiles are bound by latency, not by HBM: one
    // butterfly per thread (8 elements) and the smallest tiles.  A 512-point FP32 row pass of
    // 0.7 MB takes 4.0 us with one line per block, 4.7 us with four; column passes 5.6 us with 8
    // lines, 7.5 us with 16.
    const int wide = cols ? (dbl ? 8 : 16) : 4;
    const bool few = lines > 0 && lines < (int64_t)wide * 512;
    if (large_schedule(n, dbl, kMaxPrime(dbl), c.radices)) {
        // One butterfly of the prime per thread and at most 24 points in the other passes (444 =
        // 37 12 on 12 threads: four butterflies of 12, 332 VGPRs); rows prefer one butterfly of
        // the last pass while those are few (136 = 17 8 FP32: 17 threads 86 us per 256 MB, 8
        // threads 289; 333 = 37 9: 37 threads 219, 14 threads 209).
        const int last = n / c.radices.back();
        c.tpl = std::max(n / c.radices[0], (n + 23) / 24);
        if (!cols && c.radices.size() == 2 && last <= 31) c.tpl = last;
        c.staged = !cols && c.radices.size() == 2 && c.radices[1] <= 4;
    } else {
        // FP32 takes 24 elements per thread at most and FP64 16: the bytes in flight that hide
        // the latency of HBM come from many loads per thread.
        pick_schedule(n, few ? 8 : dbl ? 16 : 24, c.radices, c.tpl);
    }
    if (cols) {
        // FP32 16 lines per tile (128-byte pieces of rows), FP64 8; fewer where the tile leaves
        // no room for three blocks per CU (512 points FP32: 8 lines 224 us, 16 lines 248 us; FP64
        // at 384 points: 8 lines 195 us, 16 lines 237 us); more where a line has few threads
        // (12 points FP32 on 4 threads: 64 lines 102 us, 32 lines 111 us per 256 MB).
        c.pad = 1;
        c.lpb = wide;
        while (!dbl && c.lpb > 8 && (size_t)c.lpb * (size_t)n * (size_t)es > 52 * 1024) c.lpb /= 2;
        while (c.lpb * 2 * c.tpl <= 128 && c.lpb < 64 && (nl == 0 || c.lpb < nl)) c.lpb *= 2;
        // half of that for a few lines, where rows of nl lines start on whole 128-byte pieces: else two
        // XCDs share every piece (75 x 128 x 36 FP64, 128 points in place: 4 lines 11.5 us, 8 lines
        // 6.2 us)
        if (few && nl > 0 && nl % (128 / es) == 0) while (c.lpb * es > 64 && lines / c.lpb < 512) c.lpb /= 2;
    } else {
        // two waves per block (84 points FP32 on 12 threads: 10 lines 90 us, 5 lines 92 us per
        // 256 MB; FP64 79 and 84 us)
        c.pad = 0;
        c.lpb = std::max(1, (c.tpl >= 128 ? 256 : 128) / c.tpl);
        std::vector<int> four;
        if (!few && n >= 1024 && n <= 4096 && four_passes(n, four)) {
            const int tpl = n <= 2048 ? 128 : 256;
            // FP32: where the schedule above holds up to 16 points a thread it is the faster one (us per
            // 2 GiB, that / four radices up to 10: 1792 points 420 / 552, 1920 points 419 / 540, 2048
            // points 406 / 465, 3200 points 490 / 549, 3360 points 432 / 522), unless the twiddles are not
            // in LDS and the four leave no more threads idle (4096 points 588 / 522, 3600 points 573 / 705)
            fft_config t = c;
            t.twl = 1;
            const bool few_points = !dbl && n <= 16 * c.tpl;
            if (!few_points || (!two_blocks(t) && idle_factor(four, n, tpl) <= idle_factor(c.radices, n, c.tpl))) {
                c.radices = four;
                c.tpl = tpl;
                c.lpb = !dbl && n > 2048 && n <= 2560 ? 2 : 1;
            }
        }
        if (few) while (c.lpb > 1 && c.tpl * c.lpb >= 128 && lines / c.lpb < 512) c.lpb /= 2;
    }
    while (c.tpl * c.lpb > 1024 && c.lpb > 1) c.lpb /= 2;
    while (c.tpl > 1024) c.tpl = (c.tpl + 1) / 2;
    while (!valid(c) && c.lpb > 1) c.lpb /= 2;
    return c;
}

// Radix schedules of n for the autotuner, the default (factorize) first: the power-of-two
// part split into the fewest passes of radix <= 16 or one more, in descending and ascending
// order, with the odd primes after (default) or before it.  At most `max_count`.
std::vector<std::vector<int>> radix_schedules(int n, int max_count) {
    std::vector<std::vector<int>> out;
    std::vector<int> def;
    if (!factorize(n, def)) return out;
    out.push_back(def);
    int a = 0, m = n;
    while (m % 2 == 0) { m /= 2; a++; }
    std::vector<int> odd;
    std::vector<int> primes;
    prime_schedule(n, primes);
    for (int r : primes)
        if (r % 2 != 0 && r != 1) odd.push_back(r);
    std::vector<std::vector<int>> pow2;  // exponent lists, each in [1, 4]
    if (a == 0) pow2.push_back({});
    const int kmin = (a + 3) / 4;
    for (int k = kmin; a > 0 && k <= std::min(a, kmin + 1); k++) {
        // multisets of k exponents in [1, 4] summing to a, descending
        std::vector<int> e(k, 1);
        std::function<void(int, int, int)> rec = [&](int i, int left, int hi) {
            if (i == k) { if (left == 0) pow2.push_back(e); return; }
            for (int x = std::min(hi, 4); x >= 1; x--) {
                if (x > left - (k - i - 1)) continue;
                e[i] = x;
                rec(i + 1, left - x, x);
            }
        };
        rec(0, a, 4);
    }
    auto push = [&](const std::vector<int>& r) {
        if ((int)out.size() >= max_count || r.empty() || r.size() > 10) return;
        for (auto& o : out) if (o == r) return;
        out.push_back(r);
    };
    for (auto& ex : pow2) {
        std::vector<int> p2;
        for (int x : ex) p2.push_back(1 << x);
        std::vector<int> asc(p2.rbegin(), p2.rend());
        for (const auto* seq : {&p2, &asc}) {
            std::vector<int> r = *seq;
            r.insert(r.end(), odd.begin(), odd.end());
            push(r);
            std::vector<int> f = odd;
            f.insert(f.end(), seq->begin(), seq->end());
            push(f);
        }
    }
    return out;
}

std::vector<fft_config> fft_candidates(int n, bool dbl, bool in_cols, bool out_cols, int64_t lines, int64_t nl) {
    std::vector<fft_config> out;
    fft_config base = default_fft_config(n, dbl, in_cols, out_cols, lines, nl);
    out.push_back(base);
    std::vector<int> lpbs;
    if (in_cols || out_cols) lpbs = {4, 8, 16, 32};
    else lpbs = {1, 2, 4, 8, 16, 32, 64};
    auto add = [&](const fft_config& c) {
        if (!valid(c) || c.tpl * c.lpb < 64) return;
        for (auto& o : out)
            if (o.tpl == c.tpl && o.lpb == c.lpb && o.pad == c.pad && o.radices == c.radices) return;
        out.push_back(c);
    };
    // other radix schedules first (MEASURE times the first 12 candidates), each with the
    // threads per line of its own largest radix (one and two butterflies per thread and pass)
    // and the default's lines per block and padding
    const auto scheds = radix_schedules(n, 4);
    for (size_t i = 0; i < scheds.size(); i++) {
        const int rmax = *std::max_element(scheds[i].begin(), scheds[i].end());
        for (int t : {n / rmax, n / rmax / 2}) {
            if (t < 1) continue;
            fft_config c = base;
            c.radices = scheds[i];
            c.tpl = t;
            while (c.tpl * c.lpb > 1024 && c.lpb > 1) c.lpb /= 2;
            add(c);
        }
    }
    // launch shapes of the default schedule
    std::vector<int> tpls;
    for (int t = base.tpl; t >= 1 && (int)tpls.size() < 3; t /= 2) tpls.push_back(t);
    for (int t : tpls)
        for (int l : lpbs)
            for (int p : {0, 1, 2, 3}) {
                fft_config c = base;
                c.tpl = t; c.lpb = l; c.pad = p;
                add(c);
            }
    return out;
}

// Any-length kernel: the work line of m points sits whole in LDS.  Bluestein takes an
// m >= 2n - 1, up to an eighth above it, that costs least: points times the passes (12 for the
// trip through LDS, and the butterfly), and half of the threads that wait.  The largest radix goes to
// the middle: the first and last pass hold chirps and global addresses, the turning pass (the last
// radix) two tables.  One butterfly per thread in the first pass, blocks of about 160 threads.
// Lines of 313 points, 128 MB in FP32: 640 = 10 8 8 or 8 10 8 on 80 threads 173-178 us, on 64
// threads 196 us, 672 = 12 8 7 on 56 threads 202 us, the slowest of 90 shapes 399 us; 619 points:
// 1280 = 10 16 8 on 128 threads 204 us, 8 16 10 on 160 threads 231 us, the slowest 712 us.
bool any_config(int kind, int n, bool dbl, bool direct, bool cols, fft_config& c) {
    c = fft_config{};
    c.any = 1;
    c.kind = kind;
    c.nlog = n;
    c.dbl = dbl;
    c.chirp = !direct;
    const int64_t es = elem_bytes(dbl);
    const int64_t mmax = (int64_t)(kMaxLds / (size_t)es);
    const int64_t lo = direct ? n : 2 * (int64_t)n - 1;
    double best = 0;
    for (int64_t m = lo; m <= mmax && (m == lo || !direct) && (best == 0 || m <= lo + lo / 8); m++) {
        std::vector<int> r;
        if (!factorize((int)m, r)) continue;
        if (!direct) {
            std::sort(r.begin(), r.end());
            if (r.size() > 2) {  // smallest last, second largest first
                std::rotate(r.begin(), r.begin() + 1, r.end());
                std::swap(r.front(), r[r.size() - 3]);
            }
        }
        int tpl = direct ? best_tpl(r, (int)m) : (int)m / r[0];
        while (tpl > 1024) tpl = (tpl + 1) / 2;
        double cost = 0;
        for (int x : r) cost += 12.0 + 0.3 * x + (x == 11 || x == 13 ? 8.0 : 0.0);
        cost *= (double)m * std::sqrt(idle_factor(r, (int)m, tpl));
        if (best != 0 && cost >= best) continue;
        best = cost;
        c.n = (int)m;
        c.radices = r;
        c.tpl = tpl;
    }
    if (best == 0) return false;
    auto fits = [&](int l) {
        return l * c.tpl <= 1024 && (size_t)l * lds_line(c.n, 1) * (size_t)es <= 64 * 1024;
    };
    c.lpb = std::max(1, (c.tpl <= 16 ? 256 : 160) / c.tpl);
    while (c.lpb > 1 && !fits(c.lpb)) c.lpb /= 2;
    // lines adjacent in memory: 64-byte pieces of them where the tile allows it
    if (cols) while (c.lpb * es < 64 && fits(c.lpb * 2)) c.lpb *= 2;
    c.pad = c.lpb > 1 ? 1 : 0;
    return valid(c);
}

// ---- twiddles -------------------------------------------------------------------------
twiddles::~twiddles() {
    // Tables live in a process-wide cache and are released at exit; freeing device memory
    // from a static destructor after the runtime shut down is not safe, so leave it.
}

static std::mutex g_tw_mu;
static std::map<std::string, std::shared_ptr<twiddles>> g_tw;

int32_t get_twiddles(int n, const std::vector<int>& radices, bool dbl, std::shared_ptr<twiddles>* out) {
    std::string key = std::to_string(n) + (dbl ? "d" : "f");
    for (int r : radices) key += "," + std::to_string(r);
    std::lock_guard<std::mutex> lk(g_tw_mu);
    auto it = g_tw.find(key);
    if (it != g_tw.end()) { *out = it->second; return DTFFT_HIP_SUCCESS; }
    auto t = std::make_shared<twiddles>();
    int64_t total = 0, L = 1;
    std::vector<std::array<int64_t, 3>> passes;  // (off, L, R)
    for (int r : radices) {
        passes.push_back({total, L, r});
        total += L * (r - 1);
        L *= r;
    }
    const rtc_kernel* k = nullptr;
    TRY(rtc_get("fft", dbl ? "gen_twiddles_f64" : "gen_twiddles_f32", &k));
    t->bytes = std::max<int64_t>(total, 1) * 16;
    if (!compile_only()) {
        HIP_TRY(hipMalloc(&t->ptr, (size_t)t->bytes));
        for (auto& p : passes) {
            int off = (int)p[0], Lp = (int)p[1], R = (int)p[2];
            int cnt = Lp * (R - 1);
            if (cnt <= 0) continue;
            void* ptr = t->ptr;
            void* args[] = {&ptr, &off, &Lp, &R};
            TRY(launch(k, (unsigned)((cnt + 255) / 256), 256, nullptr, args));
        }
        HIP_TRY(hipDeviceSynchronize());
    }
    g_tw[key] = t;
    *out = t;
    return DTFFT_HIP_SUCCESS;
}

int32_t get_rtwiddles(int n, bool dbl, std::shared_ptr<twiddles>* out) {
    std::string key = "r" + std::to_string(n) + (dbl ? "d" : "f");
    std::lock_guard<std::mutex> lk(g_tw_mu);
    auto it = g_tw.find(key);
    if (it != g_tw.end()) { *out = it->second; return DTFFT_HIP_SUCCESS; }
    auto t = std::make_shared<twiddles>();
    int cnt = n / 2 + 1;
    const rtc_kernel* k = nullptr;
    TRY(rtc_get("fft", dbl ? "gen_rtwiddles_f64" : "gen_rtwiddles_f32", &k));
    t->bytes = (int64_t)cnt * 16;
    if (!compile_only()) {
        HIP_TRY(hipMalloc(&t->ptr, (size_t)t->bytes));
        void* ptr = t->ptr;
        int off = 0, nn = n;
        void* args[] = {&ptr, &off, &nn, &cnt};
        TRY(launch(k, (unsigned)((cnt + 255) / 256), 256, nullptr, args));
        HIP_TRY(hipDeviceSynchronize());
    }
    g_tw[key] = t;
    *out = t;
    return DTFFT_HIP_SUCCESS;
}

int32_t get_bluestein(int n, int m, bool dbl, std::shared_ptr<twiddles>* chirp, std::shared_ptr<twiddles>* bh) {
    const std::string kc = "c" + std::to_string(n) + (dbl ? "d" : "f");
    const std::string kb = "b" + std::to_string(n) + "," + std::to_string(m) + (dbl ? "d" : "f");
    std::lock_guard<std::mutex> lk(g_tw_mu);
    auto ic = g_tw.find(kc), ib = g_tw.find(kb);
    if (ic != g_tw.end() && ib != g_tw.end()) { *chirp = ic->second; *bh = ib->second; return DTFFT_HIP_SUCCESS; }
    const std::string t = dbl ? "double" : "float";
    const rtc_kernel *kch = nullptr, *kbh = nullptr;
    TRY(rtc_get("anylen", "gen_chirp<" + t + ">", &kch));
    TRY(rtc_get("anylen", "gen_bluestein_bh<" + t + ">", &kbh));
    auto c = std::make_shared<twiddles>(), b = std::make_shared<twiddles>();
    c->bytes = (int64_t)n * 16;
    b->bytes = (int64_t)m * 16;
    if (!compile_only()) {
        HIP_TRY(hipMalloc(&c->ptr, (size_t)c->bytes));
        HIP_TRY(hipMalloc(&b->ptr, (size_t)b->bytes));
        int nn = n, mm = m;
        void* ac[] = {&c->ptr, &nn};
        TRY(launch(kch, (unsigned)((n + 255) / 256), 256, nullptr, ac));
        void* ab[] = {&b->ptr, &nn, &mm};
        TRY(launch(kbh, (unsigned)m, 256, nullptr, ab));
        HIP_TRY(hipDeviceSynchronize());
    }
    g_tw[kc] = c;
    g_tw[kb] = b;
    *chirp = c;
    *bh = b;
    return DTFFT_HIP_SUCCESS;
}

// ---- stages ---------------------------------------------------------------------------
lines_desc make_lines(int64_t nl, int64_t nb, int64_t in_ls, int64_t in_bs, int64_t in_ns, int64_t out_ls,
                      int64_t out_bs, int64_t out_ns, int lpb) {
    lines_desc d{};
    d.nl = nl; d.nb = nb;
    d.in_ls = in_ls; d.in_bs = in_bs; d.in_ns = in_ns;
    d.out_ls = out_ls; d.out_bs = out_bs; d.out_ns = out_ns;
    d.ntl = (nl + lpb - 1) / lpb;
    d.ntiles = d.ntl * nb;
    return d;
}

int32_t fft_stage::init(const fft_config& c, const lines_desc& desc) {
    cfg = c;
    d = desc;
    d.ntl = (d.nl + c.lpb - 1) / c.lpb;
    d.ntiles = d.ntl * d.nb;
    if (c.any) {
        // threads run across lines where the lines are adjacent in memory, else along them
        cfg.in_cols = d.in_ls == 1 && d.in_ns != 1;
        cfg.out_cols = d.out_ls == 1 && d.out_ns != 1;
        TRY(rtc_get("anylen", cfg.expr(), &k));
        TRY(get_twiddles(c.n, c.radices, c.dbl, &tw));
        if (c.chirp) {
            TRY(get_twiddles(c.n, {c.radices.rbegin(), c.radices.rend()}, c.dbl, &twr));
            TRY(get_bluestein(c.nlog, c.n, c.dbl, &chirp, &bh));
        }
        block = (unsigned)(c.tpl * c.lpb);
        grid = (unsigned)std::min<int64_t>(d.ntiles, 1 << 22);
        return DTFFT_HIP_SUCCESS;
    }
    if (c.n > 1 || c.kind != 0) {
        TRY(rtc_get("fft", c.expr(), &k));
        TRY(get_twiddles(c.n, c.radices, c.dbl, &tw));
    }
    if (c.kind != 0) TRY(get_rtwiddles(2 * c.n, c.dbl, &rtw));
    block = (unsigned)(c.tpl * c.lpb);
    grid = (unsigned)std::min<int64_t>(d.ntiles, 1 << 22);
    if (c.twl && (c.kind == 0 || c.kind == 2) && !c.dma) {
        // persistent: as many blocks as are resident, each copying the twiddles to LDS once
        int per_cu = 1;
        if (!compile_only() && k && k->fn &&
            hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k->fn, (int)block, 0) != hipSuccess)
            per_cu = 1;
        per_cu = std::max(1, per_cu);
        grid = (unsigned)std::max<int64_t>(
            1, std::min<int64_t>(d.ntiles, (int64_t)per_cu * std::max(1, device().num_cus)));
    }
    if (c.dma) {
        if (!dma_ok(c, d)) {
            set_last_error("LDS-DMA column kernel requested for an unsuitable stage");
            return DTFFT_HIP_ERROR_INVALID_ARGUMENT;
        }
        fft_config alt = c;
        alt.dma = 0;
        if (c.kind == 2) {
            // the fallback for misaligned buffers: the plain fused C2R of the same block shape
            alt.twl = 0;
            apply_twl(alt, d, global_config().twl);
        }
        TRY(rtc_get("fft", alt.expr(), &k_alt));
        grid_alt = grid;
        if (c.dma == 1) {
            // persistent: as many blocks as are resident (one per CU with two tile buffers)
            int per_cu = 1;
            if (!compile_only() && k && k->fn &&
                hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k->fn, (int)block, 0) != hipSuccess)
                per_cu = 1;
            per_cu = std::max(1, per_cu);
            grid = (unsigned)std::max<int64_t>(
                1, std::min<int64_t>(d.ntiles, (int64_t)per_cu * std::max(1, device().num_cus)));
        }
        // dma == 2: one tile per block (the kernel strides by the grid beyond 2^22 tiles).
        // Blocks start in tile order, so the blocks resident together gather neighbouring
        // 128-byte pieces of the same rows; on MI355X this ran the 512^3 column-in / row-out
        // pass in 430 us against 446 us for the persistent double buffer, whose blocks drift
        // apart over their 64 tiles each.
    }
    return DTFFT_HIP_SUCCESS;
}

int32_t fft_stage::run(const void* in, void* out, int sign, hipStream_t s) const {
    if (d.ntiles == 0) return DTFFT_HIP_SUCCESS;
    if (cfg.any) {
        void* twp = tw ? tw->ptr : nullptr;
        void* twrp = twr ? twr->ptr : nullptr;
        void* cp = chirp ? chirp->ptr : nullptr;
        void* bp = bh ? bh->ptr : nullptr;
        lines_desc dd = d;
        int inv = sign > 0 ? 1 : 0, nl = cfg.nlog;
        void* args[] = {(void*)&in, &out, &twp, &twrp, &cp, &bp, &dd, &inv, &nl};
        return launch(k, grid, block, s, args);
    }
    if (cfg.kind != 0) {
        void* twp = tw ? tw->ptr : nullptr;
        void* rtwp = rtw ? rtw->ptr : nullptr;
        lines_desc dd = d;
        void* args[] = {(void*)&in, &out, &twp, &rtwp, &dd};
        if (cfg.dma && ((uintptr_t)in % 16) != 0) return launch(k_alt, grid_alt, block, s, args);
        return launch(k, grid, block, s, args);
    }
    if (cfg.n == 1) {
        // length-1 transform is the identity (copy the lines)
        if (in == out) return DTFFT_HIP_SUCCESS;
        if (d.in_ls == d.out_ls && d.in_bs == d.out_bs && (d.nb == 1 || d.in_bs == d.nl * d.in_ls) && d.in_ls == 1) {
            HIP_TRY(hipMemcpyAsync(out, in, (size_t)(d.nl * d.nb) * elem_bytes(cfg.dbl), hipMemcpyDeviceToDevice, s));
            return DTFFT_HIP_SUCCESS;
        }
        set_last_error("length-1 FFT stage with a strided layout");
        return DTFFT_HIP_ERROR_UNSUPPORTED_SIZE;
    }
    int inv = sign > 0 ? 1 : 0;
    void* twp = tw ? tw->ptr : nullptr;
    lines_desc dd = d;
    void* args[] = {(void*)&in, &out, &twp, &dd, &inv};
    if (cfg.dma && (((uintptr_t)in % 16) != 0 || ((uintptr_t)out % 16) != 0))
        return launch(k_alt, grid_alt, block, s, args);
    return launch(k, grid, block, s, args);
}

// "r0,r1,..." -> radices whose product is n, each a radix the kernels have
bool parse_radices(const char* text, int n, std::vector<int>& out) {
    out.clear();
    long prod = 1;
    const char* p = text;
    while (*p) {
        char* end = nullptr;
        const long r = std::strtol(p, &end, 10);
        if (end == p) return false;
        if (r < 2 || (r > 16 && !large_prime((int)r))) return false;
        out.push_back((int)r);
        prod *= r;
        p = end;
        if (*p == ',') p++;
        else if (*p) return false;
    }
    return !out.empty() && out.size() <= 10 && prod == n;
}

static int64_t span(const lines_desc& d, bool in, int n) {
    int64_t ls = in ? d.in_ls : d.out_ls, bs = in ? d.in_bs : d.out_bs, ns = in ? d.in_ns : d.out_ns;
    return (d.nl - 1) * ls + (d.nb - 1) * bs + (int64_t)(n - 1) * ns + 1;
}

// The shape of an LDS-DMA column stage for the lines of cfg: the radices as equal as they come.
// Single buffer (dma 2): several blocks share a CU, 16 threads per line up to 255 points, 32 up to
// 512 (us per 2 GiB: 160 points 360 on 16, 394 on 20; 96 points 348 on 16, 389 on 12; 320 points 362
// on 32, 389 on 16; 512 points 384 on 32, 392 on 64), but half of that where a pass would hold more
// than 16 points in a thread: over 128 VGPRs only one block of 512 threads fits a CU (480 = 10 8 6:
// 539 on 32, 420 on 16; 900 = 10 10 9: 829 on 64, 536 on 32).  Double buffer (dma 1, one block per CU):
// one butterfly per thread for powers of two from 256 on, else 32 threads.
fft_config dma_config(const fft_config& cfg, int dma) {
    fft_config c = cfg;
    c.dma = dma;
    c.staged = false;
    c.lpb = 128 / elem_bytes(c.dbl);  // a tile row is one 128-byte piece
    std::vector<int> rad;
    if (factorize(c.n, rad)) {
        c.radices = rad;
        if (dma == 2) {
            c.tpl = c.n <= 32 ? 8 : c.n < 256 ? 16 : c.n <= 512 ? 32 : 64;
            int points = 0;  // of one thread in the pass that holds most
            for (int r : rad) points = std::max(points, (c.n / r + c.tpl - 1) / c.tpl * r);
            if (c.tpl > 16 && points > 16) c.tpl /= 2;
        } else {
            c.tpl = c.n <= 512 ? 32 : 64;
            if (c.n >= 256 && (c.n & (c.n - 1)) == 0) c.tpl = c.n / rad[0];
        }
    }
    return c;
}

// Takes a column-in stage from its plain configuration to the LDS-DMA one where it is forced (lds_dma 2
// or 3) or the default rule has it so, or to the wide plain form; false: cfg stays.
static bool cols_config(fft_config& cfg, const lines_desc& d, bool inplace, int lds_dma) {
    if (lds_dma == 0 || (lds_dma == 1 && cfg.dbl)) return false;
    // Default for FP32 column-in passes, us per 2 GiB, LDS-DMA (one tile per block) against the
    // plain column kernel: 16 points 354 / 404, 36 points 384 / 550, 64 points 346 / 395, 210
    // points 380 / 490, 320 points 374 / 500, 512 points 384 / 442, 900 points 536 / 662; rows
    // of 210 lines, whose pieces straddle 128-byte lines: 64 points 357 / 441, 320 points 419 /
    // 514, 512 points 461 / 536.  In place from 48 points on (60 points 394 / 453, 36 points 467 /
    // 408, 512 points 395 / 453).  Launches of few tiles are bound by latency, where the plain
    // kernel's loads go straight to the first pass (256 points, 4 MB: 5.9 / 5.2).  FP64 keeps
    // the plain kernel, which the autotuner preferred there.
    const fft_config c = dma_config(cfg, lds_dma == 2 ? 1 : 2);
    const bool use = lds_dma >= 2 || (d.nl * d.nb >= 8192 && cfg.n >= (c.out_cols ? 48 : 16));
    if (lds_dma == 1 && inplace && cfg.out_cols && cfg.n >= 512) {
        // In-place FP32 column passes of n >= 512 where a 32-line tile (256-byte pieces of
        // every row) fits with the LDS twiddle table: the plain kernel, persistent, four
        // butterflies per thread and pass.  EXHAUSTIVE picked it at 512^3 in three runs,
        // 416 us against 427 us for the LDS-DMA double buffer (the 32-line tile fits only
        // up to n = 512; at 256^3 and 384^3 the tuner picked other kernels, which keep the
        // rule below).
        fft_config w = cfg;
        const int rmax = *std::max_element(w.radices.begin(), w.radices.end());
        w.dma = 0;
        w.lpb = 32;
        w.pad = 1;
        w.tpl = std::max(1, cfg.n / rmax / 4);
        apply_twl(w, d, 1);  // the measured form: persistent with LDS twiddles (>= 2048 tiles)
        if (w.twl && valid(w)) { cfg = w; return true; }
    }
    if (!use || !dma_ok(c, d)) return false;
    cfg = c;
    return true;
}

int32_t plan_fft_stage(int n, bool dbl, int64_t nl, int64_t nb, int64_t in_ls, int64_t in_bs, int64_t in_ns,
                       int64_t out_ls, int64_t out_bs, int64_t out_ns, bool inplace, int effort,
                       hipStream_t stream, fft_stage* st, int lds_dma) {
    std::vector<int> rad;
    if (!factorize(n, rad) && !large_schedule(n, dbl, kMaxPrime(dbl), rad)) {
        // a prime factor without a radix of its own, or more passes than a schedule holds:
        // Bluestein
        fft_config c;
        if (!any_config(0, n, dbl, false, (in_ns != 1 && in_ls == 1) || (out_ns != 1 && out_ls == 1), c)) {
            set_last_error("FFT length " + std::to_string(n) + ": the Bluestein work line does not fit in LDS");
            return DTFFT_HIP_ERROR_UNSUPPORTED_SIZE;
        }
        return st->init(c, make_lines(nl, nb, in_ls, in_bs, in_ns, out_ls, out_bs, out_ns, c.lpb));
    }
    const bool in_cols = (in_ns != 1 && in_ls == 1);
    const bool out_cols = (out_ns != 1 && out_ls == 1);
    fft_config cfg = default_fft_config(n, dbl, in_cols, out_cols, nl * nb, nl);
    lines_desc d = make_lines(nl, nb, in_ls, in_bs, in_ns, out_ls, out_bs, out_ns, cfg.lpb);
    char kb[256];
    std::snprintf(kb, sizeof kb, "fft|%d|%c|%d%d%d|%lld|%lld|%lld,%lld,%lld|%lld,%lld,%lld", n, dbl ? 'd' : 'f',
                  (int)in_cols, (int)out_cols, (int)inplace, (long long)nl, (long long)nb, (long long)in_ls,
                  (long long)in_bs, (long long)in_ns, (long long)out_ls, (long long)out_bs, (long long)out_ns);
    const std::string key(kb);
    const int twl_mode = global_config().twl;
    std::string rec;
    bool tuned = false;
    int rec_twl = -1;  // twl of a tuning record (-1: the record predates the field)
    if (n > 1 && tune_lookup(key, rec)) {
        tuned = true;
        int t, l, p, dm = 0, tw = -1, used = 0;
        char rads[128] = {0};
        const int got = std::sscanf(rec.c_str(), "%d %d %d %d %d %n%127s", &t, &l, &p, &dm, &tw, &used, rads);
        if (got >= 3) {
            fft_config c = cfg;
            c.tpl = t; c.lpb = l; c.pad = p;
            c.dma = dm;
            // the radix schedule, "r0,r1,..." (records without one keep the default)
            std::vector<int> r;
            if (got >= 6 && parse_radices(rads, n, r)) c.radices = r;
            if (valid(c) && (!c.dma || dma_ok(c, d))) { cfg = c; rec_twl = tw; }
        }
    } else if (n > 1 && effort >= DTFFT_HIP_MEASURE && !compile_only()) {
        const int64_t si = span(d, true, n), so = span(d, false, n);
        void *bi = nullptr, *bo = nullptr;
        const size_t es = (size_t)elem_bytes(dbl);
        HIP_TRY(hipMalloc(&bi, (size_t)si * es));
        if (!inplace && hipMalloc(&bo, (size_t)so * es) != hipSuccess) { hipFree(bi); return DTFFT_HIP_ERROR_ALLOC_FAILED; }
        if (inplace) bo = bi;
        TRY(fill_tuning_scratch(bi, (size_t)si * es, dbl, stream));
        double best = 1e30;
        auto cands = fft_candidates(n, dbl, in_cols, out_cols, nl * nb, nl);
        if (effort < DTFFT_HIP_EXHAUSTIVE && cands.size() > 12) cands.resize(12);
        for (size_t i = 0, nc = cands.size(); lds_dma != 0 && i < nc; i++) {  // LDS-DMA twins
            for (int v : {1, 2}) {
                fft_config c = cands[i];
                c.dma = v;
                if (dma_ok(c, d)) cands.push_back(c);
            }
        }
        // what an untuned stage runs, and both LDS-DMA kernels in their own shape
        if (lds_dma != 0) {
            fft_config untuned = cfg;
            cols_config(untuned, d, inplace, 1);
            for (const fft_config& c : {untuned, dma_config(cfg, 1), dma_config(cfg, 2)}) {
                bool known = c.dma && !dma_ok(c, d);
                for (auto& o : cands)
                    known |= o.dma == c.dma && o.tpl == c.tpl && o.lpb == c.lpb && o.pad == c.pad && o.radices == c.radices;
                if (!known) cands.push_back(c);
            }
        }
        // each candidate is timed in the form it would run: with the LDS twiddle table where
        // the rule of this configuration gives it one, and at EXHAUSTIVE also in the other form
        for (size_t i = 0, nc = cands.size(); i < nc; i++) {
            apply_twl(cands[i], d, twl_mode);
            if (effort >= DTFFT_HIP_EXHAUSTIVE && twl_mode != 0 && !cands[i].dma) {
                fft_config c = cands[i];
                apply_twl(c, d, c.twl ? 0 : 2);
                if (c.twl != cands[i].twl) cands.push_back(c);
            }
        }
        std::vector<fft_stage> built;
        std::vector<fft_config> kept;
        for (auto& c : cands) {
            fft_stage cand;
            if (cand.init(c, d)) continue;
            built.push_back(cand);
            kept.push_back(c);
        }
        std::vector<std::function<int32_t()>> runs;
        for (auto& st : built) runs.push_back([&st, bi, bo, stream]() { return st.run(bi, bo, -1, stream); });
        const std::vector<double> ms = time_candidates(runs, stream);
        for (size_t i = 0; i < kept.size(); i++)
            if (ms[i] < best) { best = ms[i]; cfg = kept[i]; }
        hipStreamSynchronize(stream);
        hipFree(bi);
        if (!inplace) hipFree(bo);
        std::string r;
        for (size_t i = 0; i < cfg.radices.size(); i++) r += (i ? "," : "") + std::to_string(cfg.radices[i]);
        char buf[160];
        std::snprintf(buf, sizeof buf, "%d %d %d %d %d %s", cfg.tpl, cfg.lpb, cfg.pad, cfg.dma, cfg.twl, r.c_str());
        tune_store(key, buf);
        tuned = true;
        rec_twl = cfg.twl;
    }
    if (lds_dma == 0) {
        cfg.dma = 0;
    } else if (!cfg.dma && (lds_dma >= 2 || !tuned) && cols_config(cfg, d, inplace, lds_dma)) {
        rec_twl = -1;
    }
    // persistent blocks with the twiddle table in LDS: as the tuning record says (the form it
    // was timed in), else by the rule of the configuration
    if (rec_twl >= 0 && twl_mode == 1) {
        apply_twl(cfg, d, rec_twl ? 2 : 0);
    } else {
        apply_twl(cfg, d, twl_mode);
    }
    return st->init(cfg, d);
}

// Schedule and threads per line of the half-length transform (m points) of a real line, R2C order.
// The last pass runs on mirror pairs, two butterflies a thread, so its radix sets the threads: 4
// gives 8 points to each, where 16 points leave too few waves (registers) and 4 too many passes
// (rows, us per GiB, FP32 / FP64: 512 points 8 4 4 4 on 64 threads 200 / 176, 8 8 8 on 32 threads
// 222 / 183, on 64 threads 281 / 218; 128 points 8 4 4 203 / 179, 16 8 247 / 202).  Lines under 64
// points take 2 or 3 (32 points: 4 4 2 222 / 178, 8 4 261 / 205).  The other passes: the fewest of
// radices up to 10, as equal as they come.  False: m in one pass.
static bool real_schedule(int m, bool dbl, std::vector<int>& radices, int& tpl) {
    if (!factorize(m, radices) || radices.size() < 2) return false;
    int last = 0;
    for (int r : m < 64 ? std::vector<int>{3, 2, 5, 7, 11, 13} : std::vector<int>{4, 3, 5, 2, 7, 11, 13})
        if (!last && m % r == 0) last = r;
    std::vector<int> cur, best;
    std::function<void(int, int)> rec = [&](int k, int hi) {
        if (k == 1) {
            const int a = std::accumulate(cur.begin(), cur.end(), 0), b = std::accumulate(best.begin(), best.end(), 0);
            if (best.empty() || cur.size() < best.size() || (cur.size() == best.size() && a < b)) best = cur;
            return;
        }
        if (cur.size() >= 8 || (!best.empty() && cur.size() >= best.size())) return;
        for (int r = std::min(hi, 13); r >= 2; r--)
            if (k % r == 0 && (r <= 10 || r == 11 || r == 13)) {
                cur.push_back(r);
                rec(k / r, r);
                cur.pop_back();
            }
    };
    rec(m / last, 13);
    if (best.empty()) return false;
    radices = best;
    radices.push_back(last);
    tpl = (m / last + 1) / 2;
    if (tpl > (dbl ? 128 : 64)) tpl = (tpl + 1) / 2;
    while (tpl > 1024) tpl = (tpl + 1) / 2;  // a block's most threads
    return true;
}

int32_t plan_real_stage(int kind, int n, bool dbl, int64_t how_many, int64_t idist, int64_t odist, int effort,
                        hipStream_t stream, fft_stage* st) {
    (void)effort; (void)stream;
    if (n < 1) {
        set_last_error("R2C/C2R length must be positive, got " + std::to_string(n));
        return DTFFT_HIP_ERROR_INVALID_DIMENSION_SIZE;
    }
    const int m = n / 2;
    fft_config c;
    // halves with a prime that is a radix of its own: only where the Bluestein form of n would fit
    std::vector<int> rad;
    const bool prime_ok = large_schedule(n, dbl, kMaxPrime(dbl), rad);
    if (n % 2 != 0 || !(factorize(m, c.radices) || prime_ok)) {
        // odd lengths (directly when n factorizes) and halves with a prime factor without a radix
        // of its own (Bluestein) take the any-length kernel: real side in real units
        const bool direct = n % 2 != 0 && factorize(n, rad);
        if (!any_config(kind, n, dbl, direct, false, c)) {
            set_last_error("R2C/C2R length " + std::to_string(n) + ": the work line does not fit in LDS");
            return DTFFT_HIP_ERROR_UNSUPPORTED_SIZE;
        }
        return st->init(c, make_lines(how_many, 1, idist, 0, 1, odist, 0, 1, c.lpb));
    }
    c = default_fft_config(m, dbl, false, false, how_many, how_many);
    c.staged = false;
    c.kind = kind;
    if (m == 1) {
        c.radices = {1}; c.tpl = 1; c.lpb = 64;
    } else if (real_schedule(m, dbl, rad, c.tpl)) {
        c.radices = rad;
        if (kind == 2) std::reverse(c.radices.begin(), c.radices.end());
        // about two waves per block, as full as they come
        auto full = [&](int l) { return (double)(l * c.tpl) / (double)((l * c.tpl + 63) / 64 * 64); };
        c.lpb = std::max(1, 128 / c.tpl);
        for (int l = c.lpb + 1; l * c.tpl <= 256; l++)
            if (full(l) > full(c.lpb) + 0.04) c.lpb = l;
    } else if (factorize(m, rad)) {
        pick_schedule(m, 8, c.radices, c.tpl);
        c.lpb = std::max(1, (c.tpl >= 64 ? 256 : 128) / c.tpl);
    }
    lines_desc d;
    if (kind == 1) {  // real lines (idist reals) viewed as complex; complex out (odist)
        if (idist % 2) { set_last_error("R2C idist must be even"); return DTFFT_HIP_ERROR_INVALID_ARGUMENT; }
        d = make_lines(how_many, 1, idist / 2, 0, 1, odist, 0, 1, c.lpb);
    } else {          // complex in (idist), real out viewed as complex (odist / 2)
        if (odist % 2) { set_last_error("C2R odist must be even"); return DTFFT_HIP_ERROR_INVALID_ARGUMENT; }
        d = make_lines(how_many, 1, idist, 0, 1, odist / 2, 0, 1, c.lpb);
    }
    apply_twl(c, d, global_config().twl);  // C2R rows: only when forced (no gain measured)
    return st->init(c, d);
}

int32_t plan_c2r_cols_stage(int n, bool dbl, int64_t nl, int64_t nb, int64_t in_bs, int64_t in_ns, int64_t out_ls,
                            int64_t out_bs, fft_stage* st, int lds_dma) {
    if (n < 2 || n % 2 != 0) {
        set_last_error("C2R stages need an even length, got " + std::to_string(n));
        return DTFFT_HIP_ERROR_UNSUPPORTED_SIZE;
    }
    const int m = n / 2;
    fft_config c;
    std::vector<int> rad;
    if (!(factorize(m, c.radices) || large_schedule(n, dbl, kMaxPrime(dbl), rad)) || m < 2) {
        // Bluestein (or the direct form for n = 2) on the any-length kernel, which writes
        // real units: the strides of the complex view double
        if (!any_config(2, n, dbl, factorize(n, rad) && m < 2, true, c)) {
            set_last_error("fused C2R length " + std::to_string(n) + ": the work line does not fit in LDS");
            return DTFFT_HIP_ERROR_UNSUPPORTED_SIZE;
        }
        return st->init(c, make_lines(nl, nb, 1, in_bs, in_ns, 2 * out_ls, 2 * out_bs, 1, c.lpb));
    }
    c = default_fft_config(m, dbl, true, false, nl * nb, nl);
    c.kind = 2;
    const fft_config whole = c;  // the schedule of the LDS-DMA kernels
    if (real_schedule(m, dbl, rad, c.tpl)) {
        c.radices.assign(rad.rbegin(), rad.rend());
        while (c.tpl * c.lpb > 1024 && c.lpb > 1) c.lpb /= 2;
    }
    lines_desc d = make_lines(nl, nb, 1, in_bs, in_ns, out_ls, out_bs, 1, c.lpb);
    apply_twl(c, d, global_config().twl);  // the tables in LDS only when forced (no gain measured)
    if (lds_dma != 0) {
        // LDS-DMA kernels: 128-byte input row pieces loaded straight into LDS, each read once;
        // two butterflies per thread and pass.  lds_dma 2: the persistent double buffer
        // (fft_c2r_dma2_kernel, one block per CU); 3: one tile per block (fft_c2r_dma_kernel,
        // two blocks per CU, the FFT twiddles in LDS only when forced with twl = 2, which leaves
        // room for one block per CU); 1: the double buffer where it fits, else one tile per block
        fft_config x = whole;
        x.lpb = 128 / elem_bytes(dbl);
        x.pad = 1;
        const int rmax = *std::max_element(x.radices.begin(), x.radices.end());
        x.tpl = std::max(1, (m / rmax) / 2);
        const lines_desc dx = make_lines(nl, nb, 1, in_bs, in_ns, out_ls, out_bs, 1, x.lpb);
        for (int v : {1, 2}) {
            if ((lds_dma == 2 && v != 1) || (lds_dma == 3 && v != 2)) continue;
            x.dma = v;
            x.twl = v == 2 && global_config().twl == 2 ? 1 : 0;
            if (dma_ok(x, dx)) return st->init(x, dx);
        }
    }
    return st->init(c, d);
}

// ---- executor handle -------------------------------------------------------------------
struct fft_plan {
    int rank = 1, type = DTFFT_HIP_FFT_C2C;
    bool dbl = false;
    hipStream_t stream = nullptr;
    // C2C: rank 1 one stage; rank 2 fast axis (in -> out) then slow axis (in place on out).
    std::vector<fft_stage> stages;
    // R2C: forward R2C along the fast axis then C2C along the slow one (in place on out);
    // backward C2C along the slow axis in place on the input (FFTW_DESTROY_INPUT, as the
    // reference's FFTW flags allow) then C2R along the fast axis.
    std::vector<fft_stage> bwd;
    // R2R: forward kinds along the fast axis (in -> out) then the slow one (in place on
    // out); backward the same order with the inverse kinds.  One work buffer serves all.
    std::vector<r2r_stage> rf, rb;
    void* work = nullptr;
    fft_plan() = default;
    fft_plan(const fft_plan&) = delete;
    ~fft_plan() { if (work) hipFree(work); }
};

}  // namespace dtfft_hip

using namespace dtfft_hip;

extern "C" {

int32_t dtfft_hip_fft_create(int8_t fft_rank, int8_t fft_type, int32_t precision, int32_t idist, int32_t odist,
                             int32_t how_many, const int32_t* fft_sizes, const int32_t* inembed,
                             const int32_t* onembed, const int32_t* r2r_kinds, int32_t effort, void* stream,
                             void** plan) {
    (void)inembed;
    if (!plan || !fft_sizes) return DTFFT_HIP_ERROR_INVALID_ARGUMENT;
    *plan = nullptr;
    if (fft_rank != 1 && fft_rank != 2) return DTFFT_HIP_ERROR_INVALID_N_DIMENSIONS;
    if (precision != DTFFT_HIP_SINGLE && precision != DTFFT_HIP_DOUBLE) return DTFFT_HIP_ERROR_INVALID_PRECISION;
    if (fft_type != DTFFT_HIP_FFT_C2C && fft_type != DTFFT_HIP_FFT_R2C && fft_type != DTFFT_HIP_FFT_R2R)
        return DTFFT_HIP_ERROR_INVALID_ARGUMENT;
    if (fft_type == DTFFT_HIP_FFT_R2R) {
        if (!r2r_kinds) return DTFFT_HIP_ERROR_MISSING_R2R_KINDS;
        for (int i = 0; i < fft_rank; i++)
            if (!r2r_kind_valid(r2r_kinds[i])) return DTFFT_HIP_ERROR_INVALID_R2R_KINDS;
    }
    if (how_many < 0) return DTFFT_HIP_ERROR_INVALID_ARGUMENT;
    if (effort < DTFFT_HIP_ESTIMATE || effort > DTFFT_HIP_EXHAUSTIVE) return DTFFT_HIP_ERROR_INVALID_EFFORT_FLAG;
    for (int i = 0; i < fft_rank; i++) if (fft_sizes[i] <= 0) return DTFFT_HIP_ERROR_INVALID_DIMENSION_SIZE;
    auto p = std::make_unique<fft_plan>();
    p->rank = fft_rank;
    p->type = fft_type;
    p->dbl = precision == DTFFT_HIP_DOUBLE;
    p->stream = (hipStream_t)stream;
    if (fft_type == DTFFT_HIP_FFT_R2R) {
        for (int dir = 0; dir < 2; dir++) {
            auto& v = dir == 0 ? p->rf : p->rb;
            auto kind_of = [&](int i) { return dir == 0 ? r2r_kinds[i] : r2r_inverse_kind(r2r_kinds[i]); };
            r2r_stage a;
            if (fft_rank == 1) {
                TRY(a.init(kind_of(0), fft_sizes[0], p->dbl, how_many, 1, dir == 0 ? idist : odist, 0, 1,
                           dir == 0 ? odist : idist, 0, 1, effort, p->stream));
                v.push_back(a);
            } else {
                const int64_t n0 = fft_sizes[0], n1 = fft_sizes[1];  // n0 slow, n1 fast (FFTW order)
                const int64_t id = dir == 0 ? idist : odist, od = dir == 0 ? odist : idist;
                r2r_stage b;
                TRY(a.init(kind_of(1), n1, p->dbl, n0, how_many, n1, id, 1, n1, od, 1, effort, p->stream));
                TRY(b.init(kind_of(0), n0, p->dbl, n1, how_many, 1, od, n1, 1, od, n1, effort, p->stream));
                v.push_back(a);
                v.push_back(b);
            }
        }
        size_t wb = 0;
        for (auto* v : {&p->rf, &p->rb})
            for (auto& st : *v) wb = std::max(wb, st.work_bytes());
        if (!compile_only()) HIP_TRY(hipMalloc(&p->work, std::max<size_t>(wb, 16)));
    } else if (fft_type == DTFFT_HIP_FFT_C2C) {
        if (fft_rank == 1) {
            fft_stage st;
            TRY(plan_fft_stage(fft_sizes[0], p->dbl, how_many, 1, idist, 0, 1, odist, 0, 1, false, effort,
                               p->stream, &st));
            p->stages.push_back(st);
        } else {
            const int n0 = fft_sizes[0], n1 = fft_sizes[1];  // n0 slow, n1 fast (FFTW order)
            fft_stage a, b;
            TRY(plan_fft_stage(n1, p->dbl, (int64_t)n0 * how_many, 1, n1, 0, 1, n1, 0, 1, false, effort,
                               p->stream, &a));
            TRY(plan_fft_stage(n0, p->dbl, n1, how_many, 1, odist, n1, 1, odist, n1, true, effort, p->stream, &b));
            p->stages.push_back(a);
            p->stages.push_back(b);
        }
    } else {
        if (fft_rank == 1) {
            fft_stage f, b;
            TRY(plan_real_stage(1, fft_sizes[0], p->dbl, how_many, idist, odist, effort, p->stream, &f));
            TRY(plan_real_stage(2, fft_sizes[0], p->dbl, how_many, odist, idist, effort, p->stream, &b));
            p->stages.push_back(f);
            p->bwd.push_back(b);
        } else {
            const int n0 = fft_sizes[0], n1 = fft_sizes[1];
            const int c1 = onembed ? onembed[1] : n1 / 2 + 1;  // complex fast extent
            fft_stage f, fs, bs, b;
            TRY(plan_real_stage(1, n1, p->dbl, (int64_t)n0 * how_many, n1, c1, effort, p->stream, &f));
            TRY(plan_fft_stage(n0, p->dbl, c1, how_many, 1, odist, c1, 1, odist, c1, true, effort, p->stream, &fs));
            TRY(plan_fft_stage(n0, p->dbl, c1, how_many, 1, odist, c1, 1, odist, c1, true, effort, p->stream, &bs));
            TRY(plan_real_stage(2, n1, p->dbl, (int64_t)n0 * how_many, c1, n1, effort, p->stream, &b));
            p->stages.push_back(f);
            p->stages.push_back(fs);
            p->bwd.push_back(bs);
            p->bwd.push_back(b);
        }
    }
    *plan = p.release();
    return DTFFT_HIP_SUCCESS;
}

int32_t dtfft_hip_fft_execute(void* plan, const void* in, void* out, int8_t sign) {
    auto* p = (fft_plan*)plan;
    if (!p) return DTFFT_HIP_ERROR_PLAN_NOT_CREATED;
    if (sign != DTFFT_HIP_FFT_FORWARD && sign != DTFFT_HIP_FFT_BACKWARD) return DTFFT_HIP_ERROR_INVALID_ARGUMENT;
    if (p->type == DTFFT_HIP_FFT_R2R) {
        const auto& v = sign == DTFFT_HIP_FFT_FORWARD ? p->rf : p->rb;
        TRY(v[0].run(in, out, p->work, p->stream));
        for (size_t i = 1; i < v.size(); i++) TRY(v[i].run(out, out, p->work, p->stream));
        return DTFFT_HIP_SUCCESS;
    }
    if (p->type == DTFFT_HIP_FFT_R2C) {
        if (in == out) return DTFFT_HIP_ERROR_INVALID_USAGE;  // src/dtfft_abstract_executor.F90:226-228
        if (sign == DTFFT_HIP_FFT_FORWARD) {
            TRY(p->stages[0].run(in, out, sign, p->stream));
            for (size_t i = 1; i < p->stages.size(); i++) TRY(p->stages[i].run(out, out, sign, p->stream));
        } else {
            if (p->bwd.size() == 2) {
                TRY(p->bwd[0].run(in, (void*)in, sign, p->stream));
                TRY(p->bwd[1].run(in, out, sign, p->stream));
            } else {
                TRY(p->bwd[0].run(in, out, sign, p->stream));
            }
        }
        return DTFFT_HIP_SUCCESS;
    }
    TRY(p->stages[0].run(in, out, sign, p->stream));
    for (size_t i = 1; i < p->stages.size(); i++) TRY(p->stages[i].run(out, out, sign, p->stream));
    return DTFFT_HIP_SUCCESS;
}

int32_t dtfft_hip_fft_destroy(void* plan) {
    delete (fft_plan*)plan;
    return DTFFT_HIP_SUCCESS;
}

}  // extern "C"
