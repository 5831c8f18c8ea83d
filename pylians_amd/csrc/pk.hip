// Power spectrum on gfx950: bin geometry, the x-pass FFT fused with window deconvolution
// and k-shell binning, and the normalisation of the outputs.
//
// Semantics follow Pk_library.pyx:266-425:
//  * independent modes: kz in [0, N/2]; on the kz = 0 and kz = N/2 planes skip kx < 0, and where
//    kx is 0 or N/2 also skip ky < 0 (Pk_library.pyx:322-330);
//  * 3-D bin = floor(|k|) (integer k^2, exact isqrt), 1-D bin = |k_par| for |k| <= N/2,
//    2-D bin = (kmax_par+1) * floor(sqrt(k_perp^2)) + |k_par| (Pk_library.pyx:334-373);
//  * window factor prod_i (x_i/sin x_i)^p, x_i = pi k_i/N (Pk_library.pyx:75-87, 354-355);
//  * multipole weights L2 = (3mu^2-1)/2, L4 = (35mu^4-30mu^2+3)/8, mu = k_par/|k| (:346-348, :376-380);
//  * phase = atan2(Re, |delta|) (:361).
// Per-mode arithmetic is in the working precision R; every shell sum is float64.
#include <math.h>

#include <algorithm>
#include <functional>
#include <map>
#include <mutex>
#include <thread>
#include <type_traits>

#include "fft.hpp"
#include "fft_engine.hpp"
#include "pk.hpp"
#include "util.hpp"

namespace pyl {

static int isqrt_host(long long v) {
    long long r = (long long)sqrt((double)v);
    while (r * r > v) --r;
    while ((r + 1) * (r + 1) <= v) ++r;
    return (int)r;
}

PkDims pk_dims(int N, int64_t P) {
    PkDims d;
    d.N = N;
    d.middle = N / 2;
    d.kmax_par = d.middle;
    d.kmax_per = isqrt_host(2LL * d.middle * d.middle);
    d.kmax = isqrt_host(3LL * d.middle * d.middle);
    d.P = P;
    return d;
}

size_t pk_out_len(const PkDims& d) { return (size_t)6 * d.kmax + 3 * (size_t)d.kmax_par + 4 * (size_t)d.n2(); }

__device__ __forceinline__ bool indep_mode(int kx, int ky, int kz, int middle, bool even) {
    if (kz == 0 || (kz == middle && even)) {
        if (kx < 0) return false;
        if ((kx == 0 || (kx == middle && even)) && ky < 0) return false;
    }
    return true;
}

// ------------------------------------------------------------------ geometry
// Counts and |k| sums of the independent modes, computed once per (N, axis) on the host with
// exact integer arithmetic; threads own slabs of kx and their histograms are summed in a fixed
// order, so the float64 |k| sums are reproducible.
static void geom_slab(int N, int axis, const PkDims& d, int x0, int x1, std::vector<unsigned long long>& n1,
                      std::vector<unsigned long long>& n2, std::vector<unsigned long long>& n3,
                      std::vector<double>& k3) {
    const int middle = N / 2;
    const bool even = (N % 2) == 0;
    for (int kxx = x0; kxx < x1; ++kxx) {
        const int kx = kxx > middle ? kxx - N : kxx;
        for (int kyy = 0; kyy < N; ++kyy) {
            const int ky = kyy > middle ? kyy - N : kyy;
            for (int kz = 0; kz <= middle; ++kz) {
                if (kz == 0 || (kz == middle && even)) {
                    if (kx < 0) continue;
                    if ((kx == 0 || (kx == middle && even)) && ky < 0) continue;
                }
                const long long k2 = (long long)kx * kx + (long long)ky * ky + (long long)kz * kz;
                const int bin = isqrt_host(k2);
                n3[bin] += 1;
                k3[bin] += sqrt((double)k2);
                int kpar, kper;
                if (axis == 0) {
                    kpar = kx;
                    kper = isqrt_host((long long)ky * ky + (long long)kz * kz);
                } else if (axis == 1) {
                    kpar = ky;
                    kper = isqrt_host((long long)kx * kx + (long long)kz * kz);
                } else {
                    kpar = kz;
                    kper = isqrt_host((long long)kx * kx + (long long)ky * ky);
                }
                kpar = kpar < 0 ? -kpar : kpar;
                if (k2 <= (long long)middle * middle) n1[kpar] += 1;
                n2[(size_t)(d.kmax_par + 1) * kper + kpar] += 1;
            }
        }
    }
}

// host half of the geometry (device pointers null), cached per (N, axis)
static const PkGeometry* host_geometry(int N, int axis) {
    static std::mutex mu;
    static std::map<std::pair<int, int>, PkGeometry*> cache;
    std::lock_guard<std::mutex> lk(mu);
    auto key = std::make_pair(N, axis);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    PkGeometry* g = new PkGeometry();
    g->d = pk_dims(N, half_len(N));
    g->axis = axis;
    g->n1 = g->n2 = g->n3 = nullptr;
    g->k3sum = nullptr;
    const PkDims& d = g->d;
    g->h_n1.assign(d.n1(), 0);
    g->h_n2.assign(d.n2(), 0);
    g->h_n3.assign(d.n3(), 0);
    g->h_k3sum.assign(d.n3(), 0.0);
    unsigned nth = std::thread::hardware_concurrency();
    nth = nth < 1 ? 1 : (nth > 16 ? 16 : nth);
    if ((int)nth > N) nth = N;
    std::vector<std::vector<unsigned long long>> a1(nth, std::vector<unsigned long long>(d.n1(), 0)),
        a2(nth, std::vector<unsigned long long>(d.n2(), 0)), a3(nth, std::vector<unsigned long long>(d.n3(), 0));
    std::vector<std::vector<double>> ak(nth, std::vector<double>(d.n3(), 0.0));
    std::vector<std::thread> pool;
    for (unsigned t = 0; t < nth; ++t) {
        const int x0 = (int)((long long)N * t / nth), x1 = (int)((long long)N * (t + 1) / nth);
        pool.emplace_back(geom_slab, N, axis, std::cref(d), x0, x1, std::ref(a1[t]), std::ref(a2[t]),
                          std::ref(a3[t]), std::ref(ak[t]));
    }
    for (auto& th : pool) th.join();
    for (unsigned t = 0; t < nth; ++t) {
        for (int i = 0; i < d.n1(); ++i) g->h_n1[i] += a1[t][i];
        for (int i = 0; i < d.n2(); ++i) g->h_n2[i] += a2[t][i];
        for (int i = 0; i < d.n3(); ++i) {
            g->h_n3[i] += a3[t][i];
            g->h_k3sum[i] += ak[t][i];
        }
    }
    cache[key] = g;
    return g;
}

// Device geometry: cached per (device, N, axis); inside a fixed arena, a per-thread copy whose
// device arrays are fresh uploads into the arena.
const PkGeometry* pk_geometry(int N, int axis, int* rc) {
    *rc = OK;
    const PkGeometry* hg = host_geometry(N, axis);
    const PkDims& d = hg->d;
    const size_t b1 = sizeof(unsigned long long) * d.n1(), b2 = sizeof(unsigned long long) * d.n2(),
                 b3 = sizeof(unsigned long long) * d.n3(), bk = sizeof(double) * d.n3();
    if (arena_fixed()) {
        static thread_local PkGeometry tg;
        tg = *hg;
        tg.n1 = (unsigned long long*)arena_upload(hg->h_n1.data(), b1, rc);
        if (*rc) return nullptr;
        tg.n2 = (unsigned long long*)arena_upload(hg->h_n2.data(), b2, rc);
        if (*rc) return nullptr;
        tg.n3 = (unsigned long long*)arena_upload(hg->h_n3.data(), b3, rc);
        if (*rc) return nullptr;
        tg.k3sum = (double*)arena_upload(hg->h_k3sum.data(), bk, rc);
        if (*rc) return nullptr;
        return &tg;
    }
    static std::mutex mu;
    static std::map<std::tuple<int, int, int>, PkGeometry*> cache;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        set_error("hipGetDevice failed");
        *rc = E_LAUNCH;
        return nullptr;
    }
    std::lock_guard<std::mutex> lk(mu);
    auto key = std::make_tuple(dev, N, axis);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    PkGeometry* g = new PkGeometry(*hg);
    char* base = nullptr;
    if (hipMalloc((void**)&base, b1 + b2 + b3 + bk) != hipSuccess) {
        set_error("geometry allocation failed");
        *rc = E_ALLOC;
        delete g;
        return nullptr;
    }
    g->k3sum = (double*)base;
    g->n1 = (unsigned long long*)(base + bk);
    g->n2 = (unsigned long long*)(base + bk + b1);
    g->n3 = (unsigned long long*)(base + bk + b1 + b2);
    hipError_t e = hipSuccess;
    if (e == hipSuccess) e = hipMemcpy(g->n1, g->h_n1.data(), b1, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(g->n2, g->h_n2.data(), b2, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(g->n3, g->h_n3.data(), b3, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(g->k3sum, g->h_k3sum.data(), bk, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        set_error("geometry upload failed: %s", hipGetErrorString(e));
        *rc = E_LAUNCH;
        (void)hipFree(base);
        delete g;
        return nullptr;
    }
    cache[key] = g;
    return g;
}

// ------------------------------------------------------------------ window tables
// win[i] = (x/sin x)^p with x = pi kfreq(i)/N (1 at x = 0): Pk_library.pyx:86-87, 316-324
static const std::vector<double>& host_window(int N, int p) {
    static std::mutex mu;
    static std::map<std::pair<int, int>, std::vector<double>> cache;
    std::lock_guard<std::mutex> lk(mu);
    auto key = std::make_pair(N, p);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    std::vector<double>& h = cache[key];
    h.resize(N);
    for (int i = 0; i < N; ++i) {
        int k = i > N / 2 ? i - N : i;
        double x = M_PI / N * k;
        h[i] = (x == 0.0) ? 1.0 : pow(x / sin(x), p);
    }
    return h;
}

// device copy cached per (device, N, p); inside a fixed arena a fresh copy in the arena
static const double* window_table(int N, int p) {
    const std::vector<double>& h = host_window(N, p);
    if (arena_fixed()) {
        int rc = OK;
        return (const double*)arena_upload(h.data(), sizeof(double) * N, &rc);
    }
    static std::mutex mu;
    static std::map<std::tuple<int, int, int>, double*> cache;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    std::lock_guard<std::mutex> lk(mu);
    auto key = std::make_tuple(dev, N, p);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    double* dptr = nullptr;
    if (hipMalloc((void**)&dptr, sizeof(double) * N) != hipSuccess) return nullptr;
    if (hipMemcpy(dptr, h.data(), sizeof(double) * N, hipMemcpyHostToDevice) != hipSuccess) return nullptr;
    cache[key] = dptr;
    return dptr;
}
const double* pk_window_table(int N, int p) { return window_table(N, p); }

// ------------------------------------------------------------------ last pass + binning
constexpr int isqrt_c(long long v) {
    long long r = 0;
    while ((r + 1) * (r + 1) <= v) ++r;
    return (int)r;
}
// LDS bytes of the histograms: 3-D (4 float64 sums + a mode count), 1-D and the 2-D window (one
// k_par row; NL rows when blocks own a kz block, fixk = 1), each a float64 sum and a 32-bit count
constexpr int hist_bytes(int N, int NL, bool fixk) {
    return (isqrt_c(3LL * (N / 2) * (N / 2)) + 1) * (4 * 8 + 4) + (N / 2 + 1) * 12 +
           (fixk ? NL : 1) * (isqrt_c(2LL * (N / 2) * (N / 2)) + 1) * 12;
}
// Threads of the binning kernel: N/16 per column line, doubled (measured faster) for lines with a
// radix-3 factor from 192 points up and where bin_wide says so: blocks that own a kz block (line of
// sight z) hold a 2-D histogram row per line, which leaves room for few blocks per CU, and from 256
// points up twice the waves per block paid (0.73 -> 0.55 ms at 512); with the line of sight along x
// or y, 256 points gained (0.094 -> 0.085 ms) and 512 lost (0.397 -> 0.410 ms).
constexpr bool bin_wide(int N, bool fixk) { return fixk ? N >= 256 : (N >= 64 && N <= 256); }
constexpr int threads_bin_c(int N, int NL, bool fixk) {
    return clamp_i(N * NL / 16 * ((N % 3 == 0 && N >= 192) || bin_wide(N, fixk) ? 2 : 1), 64, 512);
}
// LDS rows of the binning kernel's transform (RowMap::ROWS for its EU), at least N + T / NL
// (rows of NL + 1 values in the mapped layout)
constexpr int bin_rows(int N, int T, int NL) {
    const int eu = (N / 2 + 1) / (T / NL) > 0 ? (N / 2 + 1) / (T / NL) : 1;
    const int rows = eu % 2 == 0 ? N + 2 * ((N / 2) / eu) + 2 : N;
    return rows > N + T / NL ? rows : N + T / NL;
}
// LDS bytes of one binning block: the mapped rows, the twiddle and window tables, the histograms
template <typename R> constexpr int lds_bin(int N, int T, int NL, bool fixk) {
    return bin_rows(N, T, NL) * (NL + 1) * (int)sizeof(cplx<R>) + N * (int)(sizeof(cplx<R>) + sizeof(R)) +
           hist_bytes(N, NL, fixk);
}
// lines per block when two blocks share a CU (160 KB of LDS) beside their histograms: at most 8
template <typename R, int N, bool FIXK> constexpr int nl_pair() {
    int nl = 8;
    while (nl > 2 && lds_bin<R>(N, threads_bin_c(N, nl, FIXK), nl, FIXK) > 80 * 1024) nl /= 2;
    return nl;
}
// Where two blocks per CU leave only 2 lines per block (float64 lines from 512 points, float32 from
// 640: 32- or 16-byte column segments and 1-2 waves per block), one block per CU with 8 lines, or 4
// where 8 do not fit, and N * lines / 8 threads (at most 512) (float64 at 512: line of sight x
// 1.42 -> 0.69 ms with 8 lines, z 1.27 -> 0.99 ms with 4)
constexpr int SOLO_LDS = 150 * 1024;
constexpr int solo_threads(int N, int nl) { return clamp_i(N * nl / 8, 64, 512); }
template <typename R, int N, bool FIXK> constexpr int solo_nl() {
    if (nl_pair<R, N, FIXK>() != 2) return 0;
    if (lds_bin<R>(N, solo_threads(N, 8), 8, FIXK) <= SOLO_LDS) return 8;
    if (lds_bin<R>(N, solo_threads(N, 4), 4, FIXK) <= SOLO_LDS) return 4;
    return 0;
}
template <typename R, int N, bool FIXK> constexpr int nl_bin() {
    return solo_nl<R, N, FIXK>() ? solo_nl<R, N, FIXK>() : nl_pair<R, N, FIXK>();
}
template <typename R, int N, bool FIXK> constexpr int threads_bin() {
    return solo_nl<R, N, FIXK>() ? solo_threads(N, solo_nl<R, N, FIXK>())
                                 : threads_bin_c(N, nl_bin<R, N, FIXK>(), FIXK);
}


// Squared phase atan2(re, |v|)^2 of a mode (Pk_library.pyx:374), r2 = |v|^2 >= re^2.  float32:
// t = |re|/|v| in [0, 1] and atan(t) = t P(t^2) with a degree-7 polynomial fitted (Lawson-weighted
// least squares) to atan(t)/t on the whole of [0, 1], so there is no range reduction and no branch:
// 2.1e-7 relative error in float32.  r2 = 0 (then re = 0) gives 0.  float64: the library atan2.
__device__ __forceinline__ float phase_sq(float re, float r2) {
    // t may exceed 1 by the rounding of rsq; the polynomial holds there too
    const float t = fabsf(re) * __builtin_amdgcn_rsqf(r2 + 1.17549435e-38f);
    const float s = t * t;
    float p = -0.004693399649f;
    p = p * s + 0.024252869189f;
    p = p * s - 0.059487096965f;
    p = p * s + 0.099143467844f;
    p = p * s - 0.140195026994f;
    p = p * s + 0.199697285891f;
    p = p * s - 0.333319902420f;
    p = p * s + 0.999999880791f;
    const float a = t * p;
    return a * a;
}
__device__ __forceinline__ double phase_sq(double re, double r2) {
    const double ph = atan2(re, sqrt(r2));
    return ph * ph;
}

// LDS row of FFT output k in the binning kernel.  The epilogue pairs rows k and N-k (same |k|);
// thread jre of a column owns the EU pairs from u = jre*EU (the last few threads one more, each
// shifted by one per thread before it that took one more).  Rows hold MP = NL + 1 values (8-byte
// units), so the rows that consecutive threads read at one step are an odd number of units apart
// (EU rows, plus one spare row per group of EU rows when EU is even) and fall on distinct LDS banks.
template <int N, int EU> struct RowMap {
    static constexpr int PADR = (EU % 2 == 0) ? 1 : 0;
    static constexpr int GL = (N / 2) / EU + 1;   // groups of the lower half k <= N/2
    static constexpr int GU = (N / 2) / EU;
    static constexpr int ROWS = N + PADR * (GL + GU + 1);
    static __device__ __forceinline__ int row(int k) {
        if (PADR == 0) return k;
        if (k <= N / 2) return k + k / EU;
        return k + GL + GU - (N - k) / EU;
    }
};

// Last radix stage of the forward transform, written back to LDS in the RowMap order with MP
// values per row.
template <typename R, int N, int NL, int T, class RM, int MP>
__device__ __forceinline__ void last_stage_mapped(cplx<R>* s, const cplx<R>* tw, int tid) {
    constexpr Radices PL = make_radices(N);
    constexpr int RAD = PL.r[PL.n - 1];
    constexpr int NS = N / RAD;
    constexpr int NBF = NS * NL;
    constexpr int B = (NBF + T - 1) / T;
    cplx<R> v[B][RAD];
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int g = tid + b * T;
        if (NBF % T == 0 || g < NBF) {
            const int l = g % NL, j = g / NL;
#pragma unroll
            for (int m = 0; m < RAD; ++m) v[b][m] = s[(j + m * NS) * NL + l];
            if (NS > 1) {
#pragma unroll
                for (int m = 1; m < RAD; ++m) v[b][m] = cmul(v[b][m], tw[m * j]);
            }
            Dft<R, RAD>::run(v[b]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int g = tid + b * T;
        if (NBF % T == 0 || g < NBF) {
            const int l = g % NL, j = g / NL;
#pragma unroll
            for (int m = 0; m < RAD; ++m) s[RM::row(j + m * NS) * MP + l] = v[b][m];
        }
    }
    __syncthreads();
}

// The last FFT pass of the forward transform, fused with the window deconvolution and the
// binning.  The pass runs along x (last = 0; column (u = y, kz)) or y (last = 1; column
// (u = x, kz)), chosen so that k_par is constant along each column (line of sight x or y: k_par =
// k_u; z: k_par = kz).  Blocks own either one u and a range of kz blocks ("fixk = 0") or one kz
// block and a range of u ("fixk = 1"), so their 2-D histogram window stays in LDS.  A block walks
// its column blocks in order; the first-stage inputs of the next one are loaded into registers
// while the current one is transformed and binned.  The spectrum has row pitch P (kz < W valid);
// the optional window-corrected copy `keep` has pitch W.
// Every histogram entry also counts the modes it received (Nmodes, Pk_library.pyx:376-381): a
// block's row of `part` is [3-D sums (4 n3) | 1-D sums (n1) | 3-D counts (n3) | 1-D counts (n1) |
// 2-D sums (n2w) | 2-D counts (n2w)], counts held as float64.

template <typename R, int N, int NL, int T>
__device__ __forceinline__ void last_bin_body(const LastBinArgs<R>& A, Blk B) {
    const cplx<R>* __restrict__ src = A.src;
    cplx<R>* __restrict__ keep = A.keep;
    const long long P = A.P;
    const int W = A.W, last = A.last, axis = A.axis, fixk = A.fixk, nchunk = A.nchunk, flags = A.flags;
    const int kmax_par = A.kmax_par, kmax_per = A.kmax_per, n1 = A.n1, n3 = A.n3;
    const double* __restrict__ wing = A.win;
    const cplx<R>* __restrict__ twg = A.tw;
    double* __restrict__ part = A.part;
    const int RS = A.RS;
    constexpr int TPC = T / NL;              // threads per column
    constexpr int U = N / 2 + 1;             // row pairs (k, N-k), k = 0 .. N/2 (k = 0, N/2 alone)
    constexpr int EU = U / TPC;              // consecutive pairs per thread; the last UR threads of a
    constexpr int UR = U % TPC;              // column take one more
    static_assert(T % NL == 0, "bad binning geometry");
    using F = First<N, NL, T>;
    using RM = RowMap<N, (EU > 0 ? EU : 1)>;
    constexpr int MP = NL + 1;               // values per row of the mapped layout
    constexpr bool ONE = F::NST == 1;
    __shared__ cplx<R> s[(RM::ROWS * MP > N * NL ? RM::ROWS * MP : N * NL)];
    __shared__ cplx<R> tw[N];
    __shared__ R win[N];
    extern __shared__ double hs[];
    const int nper = kmax_per + 1;
    const int n2w = (fixk ? NL : 1) * nper;
    const int nsum = 4 * n3 + n1 + n2w;
    double* h3 = hs;             // n3 * 4
    double* h1 = hs + 4 * n3;    // n1
    double* h2 = h1 + n1;        // NL * nper (fixk = 1) or nper (fixk = 0)
    unsigned* c3 = (unsigned*)(hs + nsum);   // mode counts: n3 | n1 | n2w
    unsigned* c1 = c3 + n3;
    unsigned* c2 = c1 + n1;
    const int tid = threadIdx.x;
    for (int i = tid; i < N; i += T) {
        tw[i] = twg[i];
        win[i] = (R)wing[i];
    }
    for (int i = tid; i < nsum; i += T) hs[i] = 0.0;
    for (int i = tid; i < n3 + n1 + n2w; i += T) c3[i] = 0u;
    if (B.x == 0 && tid == 0) *A.status = 0u;   // counted by k_pk_reduce
    const bool drop0 = flags & PK_DROP_KZ0;

    const int middle = N / 2;
    const bool even = (N % 2) == 0;
    const int nkzb = (W + NL - 1) / NL;
    const long long EST = last == 0 ? (long long)N * P : P;   // element stride along the pass axis
    const long long UST = last == 0 ? P : (long long)N * P;   // stride of the outer coordinate u
    const long long KEST = last == 0 ? (long long)N * W : W;  // the same in `keep`
    const long long KUST = last == 0 ? W : (long long)N * W;
    const int l = tid % NL;
    const bool do1 = flags & PK_1D, do2 = flags & PK_2D, doph = flags & PK_PHASE;
    // column blocks of this block: items it = 0 .. nit-1
    int u0, kzb0, nit;
    if (fixk) {
        const int kzb = B.x / nchunk, ch = B.x % nchunk;
        const int UC = (N + nchunk - 1) / nchunk;
        u0 = ch * UC;
        nit = max(0, min(N, u0 + UC) - u0);
        kzb0 = kzb;
    } else {
        const int KB = (nkzb + nchunk - 1) / nchunk;
        u0 = B.x / nchunk;
        kzb0 = (B.x % nchunk) * KB;
        nit = max(0, min(nkzb, kzb0 + KB) - kzb0);
    }
    auto item = [&](int it, int& u, int& kzz) {
        u = fixk ? u0 + it : u0;
        kzz = (fixk ? kzb0 : kzb0 + it) * NL + l;
    };
    auto fetch = [&](int it, cplx<R> (&v)[F::B][F::RAD]) {
        int u, kzz;
        item(it, u, kzz);
        // unconditional, so that the loads stay in flight: columns past kz = N/2 read column 0 and are not binned
        const cplx<R>* p = src + (kzz < W ? (long long)u * UST + kzz : 0);
        first_load<R, N, NL, T>(v, [&](int j, int) { return p[j * EST]; }, tid);
    };
    cplx<R> nxt[F::B][F::RAD];
    if (nit > 0) fetch(0, nxt);
    for (int it = 0; it < nit; ++it) {
        {
            cplx<R> cur[F::B][F::RAD];
#pragma unroll
            for (int b = 0; b < F::B; ++b)
#pragma unroll
                for (int m = 0; m < F::RAD; ++m) cur[b][m] = nxt[b][m];
            if (it + 1 < nit) fetch(it + 1, nxt);
            __syncthreads();   // the previous epilogue has read s
            if constexpr (ONE) {
                // a single radix stage: straight from registers to the padded rows
#pragma unroll
                for (int b = 0; b < F::B; ++b) {
                    const int g = tid + b * T;
                    if (F::NBF % T == 0 || g < F::NBF) {
                        const int jj = g / NL;
                        Dft<R, F::RAD>::run(cur[b]);
#pragma unroll
                        for (int m = 0; m < F::RAD; ++m) s[RM::row(jj * F::RAD + m) * MP + l] = cur[b][m];
                    }
                }
                __syncthreads();
            } else {
                first_stage_regs<R, N, NL, NL, T>(s, cur, tid);
            }
        }
        if constexpr (!ONE) {
            mid_stages<R, N, NL, NL, T, 1, 1, F::RAD>(s, tw, tid);
            last_stage_mapped<R, N, NL, T, RM, MP>(s, tw, tid);
        }
        int u, kzz;
        item(it, u, kzz);
        // the first kz of the column block (the same for the whole block): only the blocks that hold
        // kz = 0 or kz = N/2 apply the independent-mode rule of those planes (Pk_library.pyx:322-330)
        const int kzlo = kzz - l;
        // the epilogue takes its own lane layout: TPC consecutive threads share a column (le) and hold
        // consecutive runs of row pairs (jre), so that the threads of a wave flush different bins
        // (with consecutive columns per wave they mostly share one, and their LDS atomics serialise)
        const int le = tid / TPC, jre = tid % TPC;
        kzz = kzlo + le;
        const bool zblock = kzlo == 0 || (even && middle >= kzlo && middle < kzlo + NL);
        if (kzz >= W || (drop0 && kzz == 0)) continue;
        const int kz = kzz;
        const int ku = kfreq(u, N);
        const R cuz = win[u] * win[kzz];
        const bool zplane = (kz == 0) || (kz == middle && even);
        // k_par is constant on the column: k_u (line of sight x or y) or kz
        const int kps = axis == 2 ? kz : ku;
        const int c0 = ku * ku + kz * kz;
        const int cper = c0 - kps * kps;
        const R kps2 = (R)(kps * kps);
        const long long kbase = (long long)u * KUST + kzz;
        // |k|^2 = c0 + u^2 and k_perp^2 = cper + u^2 of this thread's first pair and their bins
        // floor(sqrt); each step of u adds at most 1 to sqrt(c + u^2) (its derivative u / sqrt(c + u^2)
        // is <= 1), so each bin grows by 0 or 1 per step and is carried along without a square root
        const int extra = jre - (TPC - UR);   // >= 0: this thread takes EU + 1 pairs
        const int uq0 = jre * EU + (extra > 0 ? extra : 0);
        const int ne = EU + (extra >= 0 ? 1 : 0);
        int k2 = c0 + uq0 * uq0, kp2 = cper + uq0 * uq0;
        int bin = isqrt24(k2), wb = isqrt24(kp2);
        const int w2o = fixk ? le * nper : 0;
        // the current runs: 3-D bin cur3 and 2-D entry cur2 with their sums and modes; a run is added
        // to the LDS histograms when the bin changes and at the end (if it holds modes)
        int cur3 = bin, cur2 = w2o + wb;
        double a0 = 0.0, a2 = 0.0, a4 = 0.0, ap = 0.0, b1 = 0.0, b2 = 0.0;
        unsigned m3 = 0u, m1 = 0u, m2 = 0u;
        // pairs of rows with opposite k_j: the same |k|, k_perp, mu^2 and window factor.  ZP: the
        // column block holds a kz = 0 or Nyquist column, where a mode may not be independent
        auto pairs = [&](auto zp) {
            constexpr bool ZP = decltype(zp)::value;
#pragma unroll 1
            for (int q = 0; q < ne; ++q) {
                const int uu = uq0 + q;
                if (q > 0) {
                    k2 += 2 * uu - 1;
                    kp2 += 2 * uu - 1;
                    bin += __mul24(bin + 1, bin + 1) <= k2 ? 1 : 0;
                    wb += __mul24(wb + 1, wb + 1) <= kp2 ? 1 : 0;
                }
                const int ja = uu, jb = (N - uu) % N;
                const bool pair = jb != ja;
                const cplx<R> va = s[RM::row(ja) * MP + le];
                const cplx<R> vb = pair ? s[RM::row(jb) * MP + le] : mk<R>(0, 0);
                bool ia = true, ib = pair;
                if (ZP && zplane) {
                    const int xa = last == 0 ? uu : ku, ya = last == 0 ? ku : uu;
                    const int xb = last == 0 ? -uu : ku, yb = last == 0 ? ku : -uu;
                    // k_j = N/2 is +N/2 (kfreq); -uu for the partner row N - uu
                    ia = !(xa < 0 || ((xa == 0 || (xa == middle && even)) && ya < 0));
                    ib = pair && !(xb < 0 || ((xb == 0 || (xb == middle && even)) && yb < 0));
                }
                const R fac = win[uu] * cuz;
                if (keep) {
                    keep[kbase + ja * KEST] = ia ? scale(va, fac) : va;
                    if (pair) keep[kbase + jb * KEST] = ib ? scale(vb, fac) : vb;
                }
                if (ZP && !ia && !ib) continue;
                const unsigned nm = (ia ? 1u : 0u) + (ib ? 1u : 0u);
                const R ra = va.x * va.x + va.y * va.y;
                const R rb = vb.x * vb.x + vb.y * vb.y;
                const R r2 = (ia ? ra : (R)0) + (ib ? rb : (R)0);
                const R mu2 = k2 == 0 ? (R)0 : kps2 * recip((R)k2);
                const R d2 = r2 * (fac * fac);
                const R L2 = ((R)1.5 * mu2 - (R)0.5);
                const R L4 = (((R)35 * mu2 - (R)30) * mu2 + (R)3) * (R)0.125;
                if (bin != cur3) {
                    atomicAdd(&h3[4 * cur3 + 0], a0);
                    atomicAdd(&h3[4 * cur3 + 1], a2);
                    atomicAdd(&h3[4 * cur3 + 2], a4);
                    if (doph) atomicAdd(&h3[4 * cur3 + 3], ap);
                    atomicAdd(&c3[cur3], m3);
                    cur3 = bin;
                    a0 = a2 = a4 = ap = 0.0;
                    m3 = 0u;
                }
                const double dd = (double)d2;
                m3 += nm;
                a0 += dd;
                a2 += (double)(d2 * L2);
                a4 += (double)(d2 * L4);
                if (doph) {
                    // the phase of a mode is unchanged by the (positive) window factor
                    const R pa = phase_sq(va.x, ra), pb = phase_sq(vb.x, rb);
                    ap += (double)((ia ? pa : (R)0) + (ib ? pb : (R)0));
                }
                if (do1 && k2 <= middle * middle) {
                    b1 += dd;
                    m1 += nm;
                }
                if (do2) {
                    const int w2 = w2o + wb;
                    if (w2 != cur2) {
                        atomicAdd(&h2[cur2], b2);
                        atomicAdd(&c2[cur2], m2);
                        cur2 = w2;
                        b2 = 0.0;
                        m2 = 0u;
                    }
                    b2 += dd;
                    m2 += nm;
                }
            }
        };
        if (zblock)
            pairs(std::true_type{});
        else
            pairs(std::false_type{});
        if (m3 != 0u) {
            atomicAdd(&h3[4 * cur3 + 0], a0);
            atomicAdd(&h3[4 * cur3 + 1], a2);
            atomicAdd(&h3[4 * cur3 + 2], a4);
            if (doph) atomicAdd(&h3[4 * cur3 + 3], ap);
            atomicAdd(&c3[cur3], m3);
        }
        if (m1 != 0u) {
            atomicAdd(&h1[abs(kps)], b1);
            atomicAdd(&c1[abs(kps)], m1);
        }
        if (m2 != 0u) {
            atomicAdd(&h2[cur2], b2);
            atomicAdd(&c2[cur2], m2);
        }
    }
    // this block's histograms -> its row of the partials (summed by k_pk_reduce)
    __syncthreads();
    double* row = part + (long long)B.x * RS;
    const int n31 = 5 * n3 + 2 * n1;
    for (int i = tid; i < 4 * n3 + n1; i += T) row[i] = hs[i];
    for (int i = tid; i < n3 + n1; i += T) row[4 * n3 + n1 + i] = (double)c3[i];
    for (int i = tid; i < n2w; i += T) {
        row[n31 + i] = h2[i];
        row[n31 + n2w + i] = (double)c2[i];
    }
}
template <typename R, int N, int NL, int T>
__global__ __launch_bounds__(T) void k_last_bin(LastBinArgs<R> a) {
    last_bin_body<R, N, NL, T>(a, own_blk());
}
template <typename R, int N, int NL, int T>
__global__ __launch_bounds__(T) void k_last_bin_b(const LastBinArgs<R>* __restrict__ tab,
                                                   const unsigned* __restrict__ start, int nj) {
    PYL_BATCH_BLK(start, nj);
    last_bin_body<R, N, NL, T>(tab[bj_], blk_);
}

// Sum the per-block histogram rows of k_last_bin and normalise (Pk_library.pyx:387-421): every workgroup sums its bins
// over all rows and writes their results, so no sums are cleared, added to or read back in memory, and one launch does
// what took four (a clear, the 3-D and 1-D rows, the 2-D rows, the normalisation): 320^3, line of sight z (1008 rows,
// 43 MB) 56 -> 19 us; 32^3 15 -> 4.3 us.  Bound by the latency of its few loads (with 32 threads instead of 64 a sum:
// 27 us) and, at the first size, by reading the rows.
// Workgroups of RT threads, in this order:
//  * RE / 4 3-D bins (RE sums and their counts) each, then RE 1-D bins, the rows split over RT / RE threads a sum: the
//    longest chains, so they start first;
//  * 16 x 16 tiles of 2-D entries, (k_per, k_par) from the blocks whose window holds k_par (fixk = 0: the blocks of
//    u = k_par and u = N - k_par, k_par = |k_u|; fixk = 1: those of kz block k_par / NL, row k_par % NL; the 2-D counts
//    sit n2w entries after the 2-D sums of a row): four threads share an entry's rows, read with k_per fastest and
//    written with k_par fastest, as the row and the output have them.
// Nmodes of every histogram enabled in `flags` come from the binning kernel's counts and are
// compared, bin by bin, with the geometry (the 3-D comparison includes the DC bin, so it contains
// the total test of check_number_modes, Pk_library.pyx:90-102); histograms that were not binned
// report the geometry.
constexpr int RT = 1024;   // threads
constexpr int RE = 16;     // sums of 3-D bins (4 a bin) or 1-D bins of a workgroup
constexpr int R2 = 16;     // edge of a 2-D tile

static unsigned reduce_blocks(const PkDims& d) {
    const unsigned tiles = (unsigned)((d.kmax_par + R2) / R2) * (unsigned)((d.kmax_per + R2) / R2);
    return tiles + (unsigned)((4 * d.n3() + RE - 1) / RE + (d.n1() + RE - 1) / RE);
}

__device__ __forceinline__ double pk_unit(int N, double BoxSize) {
#pragma clang fp contract(off)
    return (BoxSize / ((double)N * N)) * (BoxSize / ((double)N * N)) * (BoxSize / ((double)N * N));
}

// The three normalisations evaluate as written (no fused multiply-add), as the reference's Python arithmetic does:
// the last 1-D bin needs kN^2 - k^2 == 0 exactly.  Each returns 1 where the count is not the geometry's.
__device__ __forceinline__ unsigned finish_3d(const ReduceArgs& A, int i, const double* s, double n) {
#pragma clang fp contract(off)
    const unsigned bad = n != (double)A.n3c[i] ? 1u : 0u;
    A.c3[i] = n;
    if (i == 0) return bad;   // DC: counted and checked, not reported (Pk_library.pyx:412)
    const double kF = 2.0 * M_PI / A.BoxSize, unit = pk_unit(A.N, A.BoxSize);
    double* o = A.out + (i - 1);
    const int kmax = A.n3 - 1;
    o[0] = (A.k3s[i] / n) * kF;
    o[kmax] = (s[0] / n) * unit;
    o[2 * kmax] = (s[1] * 5.0 / n) * unit;
    o[3 * kmax] = (s[2] * 9.0 / n) * unit;
    o[4 * kmax] = (s[3] / n) * unit;
    o[5 * kmax] = n;
    return bad;
}

__device__ __forceinline__ unsigned finish_1d(const ReduceArgs& A, int i, double s, double n) {
#pragma clang fp contract(off)
    const bool do1 = A.flags & PK_1D;
    if (!do1) n = (double)A.n1c[i];
    const unsigned bad = n != (double)A.n1c[i] ? 1u : 0u;
    if (i == 0) return bad;
    const double kF = 2.0 * M_PI / A.BoxSize, unit = pk_unit(A.N, A.BoxSize);
    const double kN = (A.N / 2) * kF;
    const double k = ((double)i * n / n) * kF;
    const double kmaxper = sqrt(kN * kN - k * k);
    double* o = A.out + 6 * (A.n3 - 1) + (i - 1);
    o[0] = k;
    o[A.kmax_par] = s * unit * (M_PI * kmaxper * kmaxper / n) / ((2.0 * M_PI) * (2.0 * M_PI));
    o[2 * A.kmax_par] = n;
    return bad;
}

__device__ __forceinline__ unsigned finish_2d(const ReduceArgs& A, int kp, int kq, double s, double n) {
#pragma clang fp contract(off)
    const int n2 = (A.kmax_par + 1) * A.nper, i = (A.kmax_par + 1) * kq + kp;
    if (!(A.flags & PK_2D)) n = (double)A.n2c[i];
    const unsigned bad = n != (double)A.n2c[i] ? 1u : 0u;
    const double kF = 2.0 * M_PI / A.BoxSize, unit = pk_unit(A.N, A.BoxSize);
    double* o = A.out + 6 * (A.n3 - 1) + 3 * A.kmax_par + i;
    if (A.compact) {
        o[0] = s * unit / n;
        return bad;
    }
    o[0] = 0.5 * (kp + kp + 1) * kF;
    o[n2] = 0.5 * (kq + kq + 1) * kF;
    o[2 * (long long)n2] = s * unit / n;
    o[3 * (long long)n2] = n;
    return bad;
}

__device__ __forceinline__ void reduce_body(const ReduceArgs& A, Blk B) {
    __shared__ double sa[4][R2 * (R2 + 1)], sm[4][R2 * (R2 + 1)];
    const double* __restrict__ part = A.part;
    const int tid = threadIdx.x, n31 = 5 * A.n3 + 2 * A.n1, nchunk = A.nchunk;
    const int nb3 = (4 * A.n3 + RE - 1) / RE, nb1 = (A.n1 + RE - 1) / RE;
    unsigned bad = 0u;
    if ((int)B.x >= nb3 + nb1) {
        const int tp = (A.kmax_par + R2) / R2, tile = (int)B.x - nb3 - nb1;
        const int kp0 = (tile % tp) * R2, kq0 = (tile / tp) * R2;
        const int t = tid & 255, g = tid >> 8;
        const int kq = kq0 + (t & 15), kp = kp0 + (t >> 4);
        double a = 0.0, m = 0.0;
        if ((A.flags & PK_2D) && kp <= A.kmax_par && kq < A.nper) {
            const bool two = !A.fixk && kp > 0 && A.N - kp > A.N / 2;   // rows of -k_u too
            const int E = two ? 2 * nchunk : nchunk;
            const long long b0 = (long long)(A.fixk ? kp / A.NL : kp) * nchunk;
            const long long b1 = (long long)(A.N - kp) * nchunk - nchunk;
            const double* p = part + n31 + (A.fixk ? (kp % A.NL) * A.nper : 0) + kq;
#pragma unroll 4
            for (int e = g; e < E; e += 4) {
                const double* q = p + ((e < nchunk ? b0 : b1) + e) * A.RS;
                a += q[0];
                m += q[A.n2w];
            }
        }
        const int w = (t >> 4) * (R2 + 1) + (t & 15);
        sa[g][w] = a;
        sm[g][w] = m;
        __syncthreads();
        if (tid < 256) {
            const int kpl = tid & 15, kql = tid >> 4, r = kpl * (R2 + 1) + kql;
            if (kp0 + kpl <= A.kmax_par && kq0 + kql < A.nper)
                bad = finish_2d(A, kp0 + kpl, kq0 + kql, (sa[0][r] + sa[1][r]) + (sa[2][r] + sa[3][r]),
                                (sm[0][r] + sm[1][r]) + (sm[2][r] + sm[3][r]));
        }
    } else {
        const int b3 = (int)B.x, b1 = b3 - nb3;
        const bool is3 = b3 < nb3;
        const int e = tid % RE;
        constexpr int ROWS = RT / RE;
        // row entries: 3-D sums (4 n3) | 1-D sums (n1) | 3-D counts (n3) | 1-D counts (n1)
        const int s = is3 ? RE * b3 + e : 4 * A.n3 + RE * b1 + e;
        const bool ins = s < (is3 ? 4 * A.n3 : 4 * A.n3 + A.n1);
        const int c = is3 ? 4 * A.n3 + A.n1 + RE / 4 * b3 + e : 5 * A.n3 + A.n1 + RE * b1 + e;
        const bool inc = is3 ? e < RE / 4 && c < 5 * A.n3 + A.n1 : c < n31;
        double a[4] = {0.0, 0.0, 0.0, 0.0}, m[4] = {0.0, 0.0, 0.0, 0.0};
        if (is3 || (A.flags & PK_1D)) {
            int b = tid / RE;
            for (; b + 3 * ROWS < A.nblocks; b += 4 * ROWS)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const double* row = part + (long long)(b + ROWS * q) * A.RS;
                    if (ins) a[q] += row[s];
                    if (inc) m[q] += row[c];
                }
            for (; b < A.nblocks; b += ROWS) {
                const double* row = part + (long long)b * A.RS;
                if (ins) a[0] += row[s];
                if (inc) m[0] += row[c];
            }
        }
        double ta = (a[0] + a[1]) + (a[2] + a[3]), tm = (m[0] + m[1]) + (m[2] + m[3]);
#pragma unroll
        for (int d = RE; d < 64; d *= 2) {
            ta += __shfl_xor(ta, d);
            tm += __shfl_xor(tm, d);
        }
        double* const pa = &sa[0][0];   // [16 waves][RE + 1]
        double* const pm = &sm[0][0];
        if ((tid & 63) < RE) {
            pa[(tid >> 6) * (RE + 1) + e] = ta;
            pm[(tid >> 6) * (RE + 1) + e] = tm;
        }
        __syncthreads();
        if (tid < 2 * RE) {
            double* const q = tid < RE ? pa : pm;
            double t = 0.0;
            for (int w = 0; w < RT / 64; ++w) t += q[w * (RE + 1) + e];
            q[e] = t;
        }
        __syncthreads();
        if (is3) {
            const int i = RE / 4 * b3 + tid;
            if (tid < RE / 4 && i < A.n3) bad = finish_3d(A, i, &pa[4 * tid], pm[tid]);
        } else {
            const int i = RE * b1 + tid;
            if (tid < RE && i < A.n1) bad = finish_1d(A, i, pa[tid], pm[tid]);
        }
    }
    if (bad) atomicAdd(A.status, bad);
}
__global__ __launch_bounds__(RT) void k_pk_reduce(ReduceArgs a) { reduce_body(a, own_blk()); }
__global__ __launch_bounds__(RT) void k_pk_reduce_b(const ReduceArgs* __restrict__ tab,
                                                    const unsigned* __restrict__ start, int nj) {
    PYL_BATCH_BLK(start, nj);
    reduce_body(tab[bj_], blk_);
}

static int num_cus() {
    static int n = 0;
    if (!n) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
            n = 256;
    }
    return n;
}

int pk_last_axis(int axis) { return axis == 0 ? 1 : 0; }

// launch shape of the binning pass for one grid size and line-of-sight class: blocks own one kz block
// (fixk, line of sight z) or one u; about two blocks per CU, all resident at once, each walking its
// column blocks with prefetch (four per CU with fixk measured faster)
template <typename R, int N, bool FIXK> struct BinShape {
    static constexpr int NL = nl_bin<R, N, FIXK>();
    static constexpr int T = threads_bin<R, N, FIXK>();
    static constexpr int W = N / 2 + 1;   // kz = 0 .. N/2; rows of the spectrum may be padded to P >= W
    int nchunk, grid, n2w, RS;
    size_t shm;
    PkDims d;
    BinShape() {
        d = pk_dims(N, W);
        const int nkzb = (W + NL - 1) / NL;
        const int want = (FIXK ? 4 : 2) * num_cus();
        if (FIXK) {
            nchunk = std::min(N, std::max(1, want / nkzb));
            grid = nkzb * nchunk;
        } else {
            nchunk = std::min(nkzb, std::max(1, (want + N - 1) / N));   // at least `want` blocks when it can
            grid = N * nchunk;
        }
        const int nper = d.kmax_per + 1;
        n2w = (FIXK ? NL : 1) * nper;
        RS = 5 * d.n3() + 2 * d.n1() + 2 * n2w;
        // LDS: float64 sums (4 n3 + n1 + n2w), then 32-bit counts (n3 + n1 + n2w)
        shm = sizeof(double) * (size_t)(4 * d.n3() + d.n1() + n2w) + sizeof(unsigned) * (size_t)(d.n3() + d.n1() + n2w);
    }
};

template <typename R, int N, bool FIXK>
static int last_bin_job_k(const cplx<R>* spec, cplx<R>* keep, int64_t P, const PkGeometry* g, double BoxSize, int p,
                          int flags, const PkCheck& chk, double* out, double* part, LastBinArgs<R>* la, ReduceArgs* ra,
                          unsigned* blocks) {
    const BinShape<R, N, FIXK> sh;
    const cplx<R>* tw = twiddles<R>(N);
    const double* win = window_table(N, p);
    PYL_CHECK(tw && win, E_ALLOC, "table allocation failed");
    const PkDims& d = sh.d;
    const int fixk = FIXK ? 1 : 0;
    *la = LastBinArgs<R>{spec, keep, (long long)P, sh.W, pk_last_axis(g->axis), g->axis, fixk, sh.nchunk, flags,
                         d.kmax_par, d.kmax_per, d.n1(), d.n3(), win, tw, part, sh.RS, chk.status};
    *ra = ReduceArgs{part, sh.RS, sh.grid, d.n3(), d.n1(), sh.n2w, d.kmax_per + 1, d.kmax_par, fixk, sh.nchunk,
                     sh.NL, N, flags, BoxSize, g->n1, g->n2, g->n3, g->k3sum, chk.c3, chk.status, out};
    *blocks = (unsigned)sh.grid;
    return OK;
}

template <typename R, int N, bool FIXK>
static int launch_last_bin_k(const cplx<R>* spec, cplx<R>* keep, int64_t P, const PkGeometry* g, double BoxSize, int p,
                             int flags, const PkCheck& chk, double* out, ReduceArgs* ra, hipStream_t st) {
    const BinShape<R, N, FIXK> sh;
    int rc = OK;
    double* part = (double*)workspace(WS_PART, sizeof(double) * (size_t)sh.grid * sh.RS, &rc);
    if (rc) return rc;
    LastBinArgs<R> la;
    unsigned grid = 0;
    rc = last_bin_job_k<R, N, FIXK>(spec, keep, P, g, BoxSize, p, flags, chk, out, part, &la, ra, &grid);
    if (rc) return rc;
    hipLaunchKernelGGL((k_last_bin<R, N, sh.NL, sh.T>), dim3(grid), dim3(sh.T), sh.shm, st, la);
    PYL_HIP(hipGetLastError());
    return OK;
}

template <typename R, int N, bool FIXK>
static int launch_last_bin_batch_k(const LastBinArgs<R>* tab, const unsigned* start, int nj, unsigned total,
                                   hipStream_t st) {
    const BinShape<R, N, FIXK> sh;
    hipLaunchKernelGGL((k_last_bin_b<R, N, sh.NL, sh.T>), dim3(total), dim3(sh.T), sh.shm, st, tab, start, nj);
    PYL_HIP(hipGetLastError());
    return OK;
}

// blocks own one kz block (fixk) when the line of sight is z, else one u: separate LDS budgets
template <typename R, int N>
static int launch_last_bin(const cplx<R>* spec, cplx<R>* keep, int64_t P, const PkGeometry* g, double BoxSize, int p,
                           int flags, const PkCheck& chk, double* out, ReduceArgs* ra, hipStream_t st) {
    return g->axis == 2
               ? launch_last_bin_k<R, N, true>(spec, keep, P, g, BoxSize, p, flags, chk, out, ra, st)
               : launch_last_bin_k<R, N, false>(spec, keep, P, g, BoxSize, p, flags, chk, out, ra, st);
}

#define PYL_PK_SIZES(X) \
    X(8) X(12) X(16) X(20) X(24) X(32) X(40) X(48) X(64) X(80) X(96) X(128) X(160) X(192) X(256) \
    X(320) X(384) X(512) X(640) X(768) X(1024)

template <typename R>
int pk_last_pass_bin(const cplx<R>* spec, cplx<R>* keep, const PkGeometry* g, int64_t P, double BoxSize, int mas_p,
                     int flags, const PkCheck& chk, double* out, ReduceArgs* ra, hipStream_t st) {
    switch (g->d.N) {
#define PYL_CASE(n) \
    case n:         \
        return launch_last_bin<R, n>(spec, keep, P, g, BoxSize, mas_p, flags, chk, out, ra, st);
        PYL_PK_SIZES(PYL_CASE)
#undef PYL_CASE
        default:
            set_error("grid size %d not supported", g->d.N);
            return E_UNSUPPORTED;
    }
}
template int pk_last_pass_bin<float>(const cplx<float>*, cplx<float>*, const PkGeometry*, int64_t, double, int, int,
                                     const PkCheck&, double*, ReduceArgs*, hipStream_t);
template int pk_last_pass_bin<double>(const cplx<double>*, cplx<double>*, const PkGeometry*, int64_t, double, int, int,
                                      const PkCheck&, double*, ReduceArgs*, hipStream_t);

size_t last_bin_part_doubles(int N, int axis, int prec) {
    switch (N) {
#define PYL_CASE(n)                                                                                          \
    case n:                                                                                                  \
        if (prec == 8)                                                                                       \
            return axis == 2 ? (size_t)BinShape<double, n, true>().grid * BinShape<double, n, true>().RS     \
                             : (size_t)BinShape<double, n, false>().grid * BinShape<double, n, false>().RS;  \
        return axis == 2 ? (size_t)BinShape<float, n, true>().grid * BinShape<float, n, true>().RS           \
                         : (size_t)BinShape<float, n, false>().grid * BinShape<float, n, false>().RS;
        PYL_PK_SIZES(PYL_CASE)
#undef PYL_CASE
        default:
            return 0;
    }
}

template <typename R>
int last_bin_job(const cplx<R>* spec, const PkGeometry* g, int64_t P, double BoxSize, int mas_p, int flags,
                 const PkCheck& chk, double* out, double* part, LastBinArgs<R>* a, ReduceArgs* r, unsigned* blocks) {
    switch (g->d.N) {
#define PYL_CASE(n)                                                                                                   \
    case n:                                                                                                           \
        return g->axis == 2                                                                                           \
                   ? last_bin_job_k<R, n, true>(spec, nullptr, P, g, BoxSize, mas_p, flags, chk, out, part, a, r,     \
                                                blocks)                                                               \
                   : last_bin_job_k<R, n, false>(spec, nullptr, P, g, BoxSize, mas_p, flags, chk, out, part, a, r,    \
                                                 blocks);
        PYL_PK_SIZES(PYL_CASE)
#undef PYL_CASE
        default:
            set_error("grid size %d not supported", g->d.N);
            return E_UNSUPPORTED;
    }
}

template <typename R>
int last_bin_batch(int N, int axis, const LastBinArgs<R>* tab, const unsigned* start, int nj, unsigned total,
                   hipStream_t st) {
    switch (N) {
#define PYL_CASE(n)                                                                                      \
    case n:                                                                                              \
        return axis == 2 ? launch_last_bin_batch_k<R, n, true>(tab, start, nj, total, st)               \
                         : launch_last_bin_batch_k<R, n, false>(tab, start, nj, total, st);
        PYL_PK_SIZES(PYL_CASE)
#undef PYL_CASE
        default:
            set_error("grid size %d not supported", N);
            return E_UNSUPPORTED;
    }
}
template int last_bin_job<float>(const cplx<float>*, const PkGeometry*, int64_t, double, int, int, const PkCheck&,
                                 double*, double*, LastBinArgs<float>*, ReduceArgs*, unsigned*);
template int last_bin_job<double>(const cplx<double>*, const PkGeometry*, int64_t, double, int, int, const PkCheck&,
                                  double*, double*, LastBinArgs<double>*, ReduceArgs*, unsigned*);
template int last_bin_batch<float>(int, int, const LastBinArgs<float>*, const unsigned*, int, unsigned, hipStream_t);
template int last_bin_batch<double>(int, int, const LastBinArgs<double>*, const unsigned*, int, unsigned, hipStream_t);

size_t pk_check_doubles(const PkDims& d) { return (size_t)d.n3() + 1; }

void pk_check_carve(const PkDims& d, double* b, PkCheck* c) {
    c->c3 = b;
    c->status = (unsigned*)(b + d.n3());
}

unsigned pk_reduce_blocks(int N) { return reduce_blocks(pk_dims(N, half_len(N))); }

int pk_reduce_batch(const ReduceArgs* tab, const unsigned* start, int nj, unsigned total, hipStream_t st) {
    hipLaunchKernelGGL(k_pk_reduce_b, dim3(total), dim3(RT), 0, st, tab, start, nj);
    PYL_HIP(hipGetLastError());
    return OK;
}

int pk_reduce(const ReduceArgs& ra, hipStream_t st) {
    hipLaunchKernelGGL(k_pk_reduce, dim3(pk_reduce_blocks(ra.N)), dim3(RT), 0, st, ra);
    PYL_HIP(hipGetLastError());
    return OK;
}

}  // namespace pyl
