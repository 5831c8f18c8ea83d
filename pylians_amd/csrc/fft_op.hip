// The pass along x of a transform pair with an operation on the modes between its two halves: the column is
// transformed forward, multiplied and transformed back while it is in LDS.  As separate passes (forward, product,
// inverse) a 512^3 float32 field took 270 + 412 + 350 us; the spectrum is now read and written once (with the filter,
// 1.6 GB): 443 us.
#include <math.h>

#include <algorithm>

#include "fft.hpp"
#include "fft_engine.hpp"
#include "util.hpp"

namespace pyl {

template <typename R> struct XArgs {
    const cplx<R>* src;
    cplx<R>* dst;
    long long SP, P;
    const cplx<R>* tw;
    XOp<R> op;
};

// the operation on the mode (x, y, kz); b: its filter value (XOP_FILTER); gbin: w_b unit / Nmodes_b per 3-D bin, 0 for
// the bins without weight (XOP_GRAD)
template <typename R, int N, int KIND>
__device__ __forceinline__ cplx<R> mode_op(const XOp<R>& op, cplx<R> a, cplx<R> b, const double* gbin, int x, int y, int kz) {
#pragma clang fp contract(off)
    constexpr int middle = N / 2;
    constexpr bool even = (N % 2) == 0;
    if constexpr (KIND == XOP_FILTER) {
        const R ac = a.x * b.x, bd = a.y * b.y, ad = a.x * b.y, bc = a.y * b.x;
        return mk(ac - bd, ad + bc);
    } else if constexpr (KIND == XOP_WINDOW || KIND == XOP_POWER) {
        if (KIND == XOP_WINDOW && (kz == 0 || (kz == middle && even))) {
            const int kx = kfreq(x, N), ky = kfreq(y, N);
            if (kx < 0 || ((kx == 0 || (kx == middle && even)) && ky < 0)) return a;
        }
        const R f = (R)(op.win[x] * op.win[y] * op.win[kz]);
        a.x = a.x * f;
        a.y = a.y * f;
        if (KIND == XOP_POWER) {
            const R re = a.x * a.x, im = a.y * a.y;
            a.x = re + im;
            a.y = (R)0;
        }
        return a;
    } else {
        const int kx = kfreq(x, N), ky = kfreq(y, N);
        const int k2 = kx * kx + ky * ky + kz * kz;   // <= 3 (N/2)^2 < 2^24
        const int bin = isqrt24(k2);
        // the stored spectrum is window-corrected on the independent modes and raw elsewhere
        const double g = gbin[bin];
        const double c = op.win[x] * op.win[y] * op.win[kz];
        bool ind = true;
        if (kz == 0 || (kz == middle && even)) {
            if (kx < 0) ind = false;
            else if ((kx == 0 || (kx == middle && even)) && ky < 0) ind = false;
        }
        double f = g * (ind ? c : c * c) * op.post;
        if (even && (kx == 0 || kx == middle) && (ky == 0 || ky == middle) && (kz == 0 || kz == middle)) f *= 2.0;
        return scale(a, (R)f);
    }
}

// Register footprint of the last stage: thread tid holds the outputs k = j + m NS of its butterflies
template <int N, int NL, int T> struct Last {
    static constexpr Radices P = make_radices(N);
    static constexpr int RAD = P.r[P.n - 1];
    static constexpr int NS = N / RAD;
    static constexpr int NBF = NS * NL;
    static constexpr int B = (NBF + T - 1) / T;
};

// Keeps the compiler from rearranging what made v with what uses it.  The contraction of a butterfly's products into
// fused multiply-adds depends on its surroundings; with its outputs settled the pass rounds as the plain one does
// (two stages and more, with the compiler in use: tests/test_gpu_mode_equal.py compares the two bit for bit; 8 points,
// one stage, round in their own way).
template <typename R> __device__ __forceinline__ cplx<R> settle(cplx<R> v) {
    asm volatile("" : "+v"(v.x), "+v"(v.y));
    return v;
}

// The radix-5 butterfly of fft_engine.hpp with the fused operations of its two sums written out, as the compiler makes them
// in the plain passes (here it fused the other product).  Named in the plain one instead, they changed the last
// bits of every transform with a factor 5.
template <typename R> __device__ __forceinline__ void dft5(cplx<R>* a) {
    const R c1 = (R)0.30901699437494742410229341718282, c2 = (R)-0.80901699437494742410229341718282;
    const R s1 = (R)0.95105651629515357211643933337938, s2 = (R)0.58778525229247312916870595463907;
    const cplx<R> p1 = a[1] + a[4], d1 = a[1] - a[4], p2 = a[2] + a[3], d2 = a[2] - a[3];
    const cplx<R> m1 = mk(a[0].x + c1 * p1.x + c2 * p2.x, a[0].y + c1 * p1.y + c2 * p2.y);
    const cplx<R> m2 = mk(a[0].x + c2 * p1.x + c1 * p2.x, a[0].y + c2 * p1.y + c1 * p2.y);
    const cplx<R> r1 = mul_mi(mk((R)fma(s1, d1.x, s2 * d2.x), (R)fma(s1, d1.y, s2 * d2.y)));
    const cplx<R> r2 = mul_mi(mk(s2 * d1.x - s1 * d2.x, s2 * d1.y - s1 * d2.y));
    a[0] = a[0] + p1 + p2;
    a[1] = m1 + r1;
    a[4] = m1 - r1;
    a[2] = m2 + r2;
    a[3] = m2 - r2;
}

// Last stage of a forward transform in LDS, each output handed to f(k, value, b, m) and its result left in LDS in
// natural order, conjugated for the inverse transform.
template <typename R, int N, int NL, int T, class FN>
__device__ __forceinline__ void last_stage_op(cplx<R>* s, const cplx<R>* tw, FN&& f, int tid) {
    using L = Last<N, NL, T>;
    constexpr int RAD = L::RAD, NS = L::NS, NBF = L::NBF, B = L::B;
    cplx<R> v[B][RAD];
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int g = tid + b * T;
        if (NBF % T == 0 || g < NBF) {
            const int l = g % NL, j = g / NL;
#pragma unroll
            for (int m = 0; m < RAD; ++m) v[b][m] = s[(j + m * NS) * NL + l];
#pragma unroll
            for (int m = 1; m < RAD; ++m) v[b][m] = cmul(v[b][m], tw[m * j * (N / (NS * RAD))]);
            if constexpr (RAD == 5)
                dft5(v[b]);
            else
                Dft<R, RAD>::run(v[b]);
#pragma unroll
            for (int m = 0; m < RAD; ++m) v[b][m] = settle(v[b][m]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int g = tid + b * T;
        if (NBF % T == 0 || g < NBF) {
            const int l = g % NL, j = g / NL;
#pragma unroll
            for (int m = 0; m < RAD; ++m) s[(j + m * NS) * NL + l] = conjg(f(j + m * NS, v[b][m], b, m));
        }
    }
    __syncthreads();
}

// Persistent blocks of NL columns (y, kz), as the plain column pass (fft.hip)
template <typename R, int N, int NL, int T, int KIND>
__global__ __launch_bounds__(T) void k_cols_op(XArgs<R> A) {
    static_assert(T % NL == 0, "T must be a multiple of NL");
    using F = First<N, NL, T>;
    constexpr bool FWD = KIND != XOP_GRAD;
    constexpr bool PREFETCH = N <= 512;
    constexpr int W = N / 2 + 1;
    __shared__ cplx<R> s[N * NL];
    __shared__ cplx<R> tw[N];
    // 3-D bins floor(|k|): at most sqrt(3) N / 2, so N of them do
    __shared__ double gbin[KIND == XOP_GRAD ? N : 1];
    const int tid = threadIdx.x;
    for (int i = tid; i < N; i += T) tw[i] = A.tw[i];
    if (KIND == XOP_GRAD)
        for (int i = tid; i < N; i += T)
            gbin[i] = i >= 1 && i <= A.op.nb ? A.op.w[i - 1] * A.op.unit / (double)A.op.n3[i] : 0.0;
    const int l = tid % NL;
    const long long P = A.P, SP = A.SP, ncols = (long long)N * P, nblk = (ncols + NL - 1) / NL;
    const long long SEST = (long long)N * SP, EST = (long long)N * P;
    auto column = [&](long long cb, int& y, int& kz) {
        const long long c = cb * NL + l;
        y = (int)(c / P);
        kz = (int)(c % P);
        return c < ncols && kz < W;
    };
    auto load = [&](long long cb, cplx<R> (&v)[F::B][F::RAD]) {
        int y, kz;
        const bool ok = column(cb, y, kz);
        // unconditional (padding reads column 0, which is not stored), so that the loads stay in flight
        const cplx<R>* p = A.src + (ok ? (long long)y * SP + kz : 0);
        first_load<R, N, NL, T>(v, [&](int j, int) { return p[j * SEST]; }, tid);
    };
    cplx<R> nxt[F::B][F::RAD];
    long long cb = blockIdx.x;
    if (PREFETCH && cb < nblk) load(cb, nxt);
    for (; cb < nblk; cb += gridDim.x) {
        cplx<R> cur[F::B][F::RAD];
        if (PREFETCH) {
#pragma unroll
            for (int b = 0; b < F::B; ++b)
#pragma unroll
                for (int m = 0; m < F::RAD; ++m) cur[b][m] = nxt[b][m];
            if (cb + gridDim.x < nblk) load(cb + gridDim.x, nxt);
        } else {
            load(cb, cur);
        }
        int y, kz;
        const bool ok = column(cb, y, kz);
        const cplx<R> none = mk<R>(0, 0);
        auto op = [&](int k, cplx<R> v, cplx<R> f) { return ok ? mode_op<R, N, KIND>(A.op, v, f, gbin, k, y, kz) : v; };
        const cplx<R>* fp = KIND == XOP_FILTER ? A.op.filt + (ok ? (long long)y * A.op.FP + kz : 0) : nullptr;
        const long long FEST = (long long)N * A.op.FP;
        __syncthreads();   // LDS of the previous block consumed (and twiddles loaded)
        if constexpr (FWD) {
            if constexpr (F::NST == 1) {
#pragma unroll
                for (int b = 0; b < F::B; ++b) {
                    const int g = tid + b * T;
                    if (F::NBF % T == 0 || g < F::NBF) {
                        const int j = g / NL;
                        Dft<R, F::RAD>::run(cur[b]);
#pragma unroll
                        for (int m = 0; m < F::RAD; ++m) {
                            const int k = j * F::RAD + m;
                            s[k * NL + l] = conjg(op(k, cur[b][m], KIND == XOP_FILTER ? fp[k * FEST] : none));
                        }
                    }
                }
                __syncthreads();
            } else {
                using L = Last<N, NL, T>;
                first_stage_regs<R, N, NL, NL, T>(s, cur, tid);
                // the filter values of the thread's outputs load during the middle stages (512^3: 60 us off)
                cplx<R> fv[L::B][L::RAD];
                if constexpr (KIND == XOP_FILTER) {
#pragma unroll
                    for (int b = 0; b < L::B; ++b) {
                        const int j = min(tid + b * T, L::NBF - 1) / NL;
#pragma unroll
                        for (int m = 0; m < L::RAD; ++m) fv[b][m] = fp[(j + m * L::NS) * FEST];
                    }
                }
                mid_stages<R, N, NL, NL, T, 1, 1, F::RAD>(s, tw, tid);
                last_stage_op<R, N, NL, T>(
                    s, tw, [&](int k, cplx<R> v, int b, int m) { return op(k, v, KIND == XOP_FILTER ? fv[b][m] : none); },
                    tid);
            }
            first_load<R, N, NL, T>(cur, [&](int j, int) { return settle(s[j * NL + l]); }, tid);
            __syncthreads();
        } else {
#pragma unroll
            for (int b = 0; b < F::B; ++b) {
                const int g = tid + b * T;
                if (F::NBF % T == 0 || g < F::NBF) {
                    const int j = g / NL;
#pragma unroll
                    for (int m = 0; m < F::RAD; ++m) cur[b][m] = conjg(op(j + m * F::STRIDE, cur[b][m], none));
                }
            }
        }
        const long long base = (long long)y * P + kz;
        auto store = [&](int k, int, cplx<R> v) {
            if (ok) A.dst[base + k * EST] = conjg(v);
        };
        if constexpr (F::NST == 1) {
#pragma unroll
            for (int b = 0; b < F::B; ++b) {
                const int g = tid + b * T;
                if (F::NBF % T == 0 || g < F::NBF) {
                    const int j = g / NL;
                    Dft<R, F::RAD>::run(cur[b]);
#pragma unroll
                    for (int m = 0; m < F::RAD; ++m) store(j * F::RAD + m, l, cur[b][m]);
                }
            }
        } else {
            first_stage_regs<R, N, NL, NL, T>(s, cur, tid);
            mid_stages<R, N, NL, NL, T, 1, 1, F::RAD>(s, tw, tid);
            last_stage_store<R, N, NL, NL, T, 1>(s, tw, store, tid);
        }
    }
}

template <typename R, int N, int KIND>
static int launch_op(const XArgs<R>& a, hipStream_t st) {
    using SH = ColShape<R, N>;
    const long long nblk = ((long long)N * a.P + SH::NL - 1) / SH::NL;
    int per_cu = (160 * 1024) / (SH::LDS + (KIND == XOP_GRAD ? 8 * N : 0) + 1024);
    per_cu = per_cu < 1 ? 1 : (per_cu > 8 ? 8 : per_cu);
    const long long nb = std::min<long long>((long long)cu_count() * per_cu, nblk);
    hipLaunchKernelGGL((k_cols_op<R, N, SH::NL, SH::T, KIND>), dim3((unsigned)nb), dim3(SH::T), 0, st, a);
    PYL_HIP(hipGetLastError());
    return OK;
}

template <typename R, int N>
static int launch_op_n(XArgs<R>& a, hipStream_t st) {
    a.tw = twiddles<R>(N);
    PYL_CHECK(a.tw, E_ALLOC, "twiddle table allocation failed");
    switch (a.op.kind) {
        case XOP_WINDOW: return launch_op<R, N, XOP_WINDOW>(a, st);
        case XOP_POWER: return launch_op<R, N, XOP_POWER>(a, st);
        default: break;
    }
    if constexpr (sizeof(R) == 4) {
        if (a.op.kind == XOP_FILTER) return launch_op<R, N, XOP_FILTER>(a, st);
        if (a.op.kind == XOP_GRAD) return launch_op<R, N, XOP_GRAD>(a, st);
    }
    set_error("unknown mode operation %d", a.op.kind);
    return E_ARG;
}

template <typename R>
int fft_pass_x_op(const cplx<R>* src, int64_t SP, cplx<R>* dst, int N, int64_t P, const XOp<R>& op, hipStream_t st) {
    PYL_CHECK(SP >= half_len(N) && P >= half_len(N) && (src != dst || SP == P), E_ARG, "bad spectrum pitch");
    XArgs<R> a{src, dst, (long long)SP, (long long)P, nullptr, op};
    switch (N) {
#define PYL_CASE(n) \
    case n:         \
        return launch_op_n<R, n>(a, st);
        PYL_FFT_SIZES(PYL_CASE)
#undef PYL_CASE
        default:
            set_error("FFT size %d not supported", N);
            return E_UNSUPPORTED;
    }
}
template int fft_pass_x_op<float>(const cplx<float>*, int64_t, cplx<float>*, int, int64_t, const XOp<float>&, hipStream_t);
template int fft_pass_x_op<double>(const cplx<double>*, int64_t, cplx<double>*, int, int64_t, const XOp<double>&,
                                   hipStream_t);

}  // namespace pyl
