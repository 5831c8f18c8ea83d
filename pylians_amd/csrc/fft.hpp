// Host-side interface of the 3-D real FFT (r2c / c2r) built from the LDS Stockham engine.
//
// Layout: real grid r[x][y][z] (N^3, z fastest); half spectrum c[x][y][kz], kz in [0, N/2],
// row pitch P (complex elements; P = N/2+1 gives FFTW's / numpy's rfftn layout).
// Forward = unnormalised (FFTW_FORWARD); inverse = unnormalised times `scale`.
#pragma once
#include "common.hpp"

namespace pyl {

// the transform lengths
#define PYL_FFT_SIZES(X) \
    X(8) X(12) X(16) X(20) X(24) X(32) X(40) X(48) X(64) X(80) X(96) X(128) X(160) X(192) X(256) \
    X(320) X(384) X(512) X(640) X(768) X(1024)

bool fft_size_supported(int N);

// compute units of the current device (cached)
int cu_count();
// workgroups of a persistent launch over `units` pieces of work, at most `most` resident a CU
long long persistent_blocks(long long units, int most);

// twiddle table exp(-2 pi i t/N), t in [0, N), cached per (N, precision); device pointer
template <typename R> const cplx<R>* twiddles(int N);

// pass Z: rows r2c. out rows have P complex.  When `affine`, input values are mapped to the
// overdensity v / rhobar - 1 with rhobar = mass / N^3, mass = dmass[0] (device) or `mass`.
template <typename R>
int fft_pass_z_r2c(const R* in, cplx<R>* out, int N, int64_t P, bool affine, const double* dmass, double mass,
                   hipStream_t st);

// column pass along y (axis 1) or x (axis 0) on a half spectrum, src -> dst (may alias).  K > 0:
// transform just the columns kz < K and leave the others untouched.
template <typename R>
int fft_pass_cols(const cplx<R>* src, cplx<R>* dst, int N, int64_t P, int axis, bool inverse, R scale,
                  hipStream_t st, int K = 0);

// pass Z inverse: rows c2r (unnormalised * scale).  store: 0 = nothing written, 1 = x,
// 2 = x * aux.  When acc != nullptr the kernel also adds sum(x^2) into acc[0] and sum(x * aux)
// into acc[1] (float64; aux == nullptr counts as zero).  K > 0: entries kz >= K are zero and
// are not read.
template <typename R>
int fft_pass_z_c2r(const cplx<R>* in, R* out, int N, int64_t P, R scale, int store, const R* aux,
                   double* acc, hipStream_t st, int K = 0);

// Argument blocks of pass Z (rows r2c) and of the column pass, shared with the batch planner
template <typename R> struct R2cArgs {
    const R* in;
    cplx<R>* out;
    long long nrows, P;
    const cplx<R>* tw;
    int affine;
    const double* dmass;
    double mass, ncell;
};

template <typename R> struct ColArgs {
    const cplx<R>* src;
    cplx<R>* dst;
    long long ncols, CW, CS, EST, PW;
    int W;
    const cplx<R>* tw;
    R sc;
};

// Batched launches over jobs of one grid size N (one launch for all of them): *_job builds a job's
// arguments and block count (no launch), *_batch launches the device table tab[0..nj) whose
// block ranges are start[0..nj] (start[nj] = total).
template <typename R>
int r2c_job(const R* in, cplx<R>* out, int N, int64_t P, bool affine, const double* dmass, double mass,
            R2cArgs<R>* a, unsigned* blocks);
template <typename R>
int r2c_batch(int N, const R2cArgs<R>* tab, const unsigned* start, int nj, unsigned total, hipStream_t st);
template <typename R>
int cols_job(const cplx<R>* src, cplx<R>* dst, int N, int64_t P, int axis, ColArgs<R>* a, unsigned* blocks);
template <typename R>
int cols_batch(int N, const ColArgs<R>* tab, const unsigned* start, int nj, unsigned total, hipStream_t st);

// Row pitch of a library-owned spectrum: N / 2 + 1 rounded up to 128 bytes, so that the strided column passes read
// whole cache lines
template <typename R> inline int64_t padded_pitch(int N) {
    constexpr int64_t A = 128 / (int64_t)sizeof(cplx<R>);
    return (half_len(N) + A - 1) / A * A;
}

// Operation on the modes of a half spectrum, applied inside the pass along x (fft_pass_x_op)
enum { XOP_FILTER = 0, XOP_WINDOW = 1, XOP_POWER = 2, XOP_GRAD = 3 };
template <typename R> struct XOp {
    int kind;
    // XOP_FILTER: v *= filt (half spectrum of row pitch FP), products rounded one by one
    const cplx<R>* filt = nullptr;
    long long FP = 0;
    // XOP_WINDOW: v *= W of the independent modes; XOP_POWER: v = (|W v|^2, 0)
    const double* win = nullptr;
    // XOP_GRAD: v *= H of the power spectrum's adjoint (adjoint.hip): weights w[nb] of the bins, their mode counts n3
    const double* w = nullptr;
    int nb = 0;
    const unsigned long long* n3 = nullptr;
    double unit = 0.0, post = 0.0;
};
// XOP_FILTER, XOP_WINDOW, XOP_POWER: forward transform along x, the operation, inverse transform along x, in one pass
// over the spectrum; XOP_GRAD: the operation, then the inverse transform along x.  src (row pitch SP) -> dst (row
// pitch P; may alias when SP == P).  FILTER and GRAD: float32.
template <typename R>
int fft_pass_x_op(const cplx<R>* src, int64_t SP, cplx<R>* dst, int N, int64_t P, const XOp<R>& op, hipStream_t st);

// full transforms; with K > 0 only the modes kz < K of the r2c are complete (the column passes
// skip the others, which keep the pass-Z values)
template <typename R>
int fft3d_r2c(const R* in, cplx<R>* out, int N, int64_t P, hipStream_t st, int K = 0);
// in is not modified; ws must hold N*N*P complex values (may equal nothing else)
template <typename R>
int fft3d_c2r(const cplx<R>* in, R* out, cplx<R>* ws, int N, int64_t P, R scale, hipStream_t st);

}  // namespace pyl
