// Power-spectrum estimator pieces (Pk_library.pyx:266-425 semantics) for gfx950.
#pragma once
#include "common.hpp"

namespace pyl {

struct PkDims {
    int N, middle, kmax_par, kmax_per, kmax;
    int64_t P;                 // half-spectrum row pitch (complex elements)
    int n1() const { return kmax_par + 1; }
    int n2() const { return (kmax_par + 1) * (kmax_per + 1); }
    int n3() const { return kmax + 1; }
};
PkDims pk_dims(int N, int64_t P);

// Data-independent bin geometry of the independent modes (Pk_library.pyx:322-330):
// integer mode counts per 1-D / 2-D / 3-D bin and the float64 sum of |k| per 3-D bin
// (kF units).  Computed once per (device, N, axis) on the GPU and cached.
struct PkGeometry {
    PkDims d;
    int axis;
    // device arrays
    unsigned long long* n1;    // n1()
    unsigned long long* n2;    // n2()
    unsigned long long* n3;    // n3()
    double* k3sum;             // n3()
    // host copies
    std::vector<unsigned long long> h_n1, h_n2, h_n3;
    std::vector<double> h_k3sum;
};
const PkGeometry* pk_geometry(int N, int axis, int* rc);

// The mode check's part of a call's results, device arrays owned by the caller (pk_check_doubles doubles)
struct PkCheck {
    double* c3;         // n3: modes binned per 3-D bin
    unsigned* status;   // [1]: bins whose count differs from the mode geometry
};
size_t pk_check_doubles(const PkDims& d);
void pk_check_carve(const PkDims& d, double* base, PkCheck* c);

// PK_ASYNC: no host synchronisation for the mode check (the counts are still in the output).
// PK_DROP_KZ0: the binning kernel leaves out the kz = 0 plane -- fault injection for the tests of
// the mode check, never set by the library itself.
enum PkFlags { PK_1D = 1, PK_2D = 2, PK_PHASE = 4, PK_ASYNC = 256, PK_DROP_KZ0 = 512 };

// Argument blocks of the fused last pass + binning and of the reduction of its per-block histograms with the
// normalisation (shared with the batch planner)
template <typename R> struct LastBinArgs {
    const cplx<R>* src;
    cplx<R>* keep;
    long long P;
    int W, last, axis, fixk, nchunk, flags, kmax_par, kmax_per, n1, n3;
    const double* win;
    const cplx<R>* tw;
    double* part;
    int RS;
    unsigned* status;   // cleared here, counted by the reduction
};

struct ReduceArgs {
    const double* part;
    int RS, nblocks, n3, n1, n2w, nper, kmax_par, fixk, nchunk, NL, N, flags;
    double BoxSize;
    const unsigned long long *n1c, *n2c, *n3c;   // the geometry
    const double* k3s;
    double* c3;
    unsigned* status;
    double* out;
    int compact = 0;   // out holds [k3D .. Nmodes1D | Pk2D] only: the rest of the layout the host knows by itself
};

// Axis of the last forward FFT pass for a line of sight `axis`: 1 (y) for axis 0, else 0 (x).
// The half spectrum must have gone through pass Z and the column pass along the other axis.
int pk_last_axis(int axis);
// That last pass fused with the window deconvolution and the binning of the independent modes, into per-block histogram
// rows; `ra` receives the arguments of pk_reduce, which makes the results of them.
// keep (nullable) receives the window-corrected spectrum (Pk_library.pyx:354-355, 423).
template <typename R>
int pk_last_pass_bin(const cplx<R>* spec, cplx<R>* keep, const PkGeometry* g, int64_t P, double BoxSize, int mas_p,
                     int flags, const PkCheck& chk, double* out, ReduceArgs* ra, hipStream_t st);

// Sum of the rows and normalisation of Pk_library.pyx:387-421 on the device, with Nmodes from the binning kernel's
// counts; every bin whose count differs from the geometry is counted into chk.status (the
// check_number_modes test, Pk_library.pyx:90-102, made per bin).  out layout (float64):
//   [k3D (kmax) | P0 (kmax) | P2 (kmax) | P4 (kmax) | Pkphase (kmax) | Nmodes3D (kmax) |
//    k1D (kmax_par) | Pk1D (kmax_par) | Nmodes1D (kmax_par) |
//    kpar (n2) | kper (n2) | Pk2D (n2) | Nmodes2D (n2)]
size_t pk_out_len(const PkDims& d);
int pk_reduce(const ReduceArgs& ra, hipStream_t st);

// Batched last pass + binning over jobs of one grid size N and line of sight class (z or not), and the reduction of
// jobs of any size: last_bin_job builds a job's arguments (part: its per-block histogram rows,
// last_bin_part_doubles(N, axis, prec) of them) and block count, pk_reduce_blocks the blocks of its reduction; the
// launches take tables (block ranges start[0..nj]).
size_t last_bin_part_doubles(int N, int axis, int prec);
template <typename R>
int last_bin_job(const cplx<R>* spec, const PkGeometry* g, int64_t P, double BoxSize, int mas_p, int flags,
                 const PkCheck& chk, double* out, double* part, LastBinArgs<R>* a, ReduceArgs* r, unsigned* blocks);
template <typename R>
int last_bin_batch(int N, int axis, const LastBinArgs<R>* tab, const unsigned* start, int nj, unsigned total,
                   hipStream_t st);
unsigned pk_reduce_blocks(int N);
int pk_reduce_batch(const ReduceArgs* tab, const unsigned* start, int nj, unsigned total, hipStream_t st);

// Deposit algorithm of the fused particles -> P(k) path: cell-binned, direct atomic, or cell-binned
// after a presort by supertile.  deposit_kind: the one `flags` forces (DEP_ATOMIC / DEP_BINNED /
// DEP_SORTED), else the autotuner's (timing trials the first time a size class is seen, which
// overwrite `grid`).  pk_particles: the whole fused path of one job (pyl_pk_particles);
// keep (float32 only, nullable) receives the corrected spectrum.
enum DepositKind { DK_BINNED = 0, DK_ATOMIC = 1, DK_SORTED = 2 };
struct Rsd;
int deposit_kind(const float* pos, const float* W, int64_t n, int dims, double BoxSize, int scheme, bool f64,
                 int flags, void* grid, const double* dmass, hipStream_t st, int* kind, const Rsd& rsd);
int pk_particles(const float* pos, const float* W, int64_t n, int dims, double BoxSize, int scheme, int axis,
                 int prec, int flags, double* out, hipStream_t st, const Rsd& rsd, cplx<float>* keep = nullptr,
                 double* host = nullptr);

// The whole estimator from a real (N,N,N) field: pass Z r2c (affine: delta = rho * N^3 / mass - 1
// applied on the load, mass = dmass[0] when dmass is non-null), the column pass, the fused last pass
// + binning, the normalisation and the mode check (see pyl_pk).  keep (nullable) receives the
// corrected spectrum.  host (nullable): the results go to this host array instead of `out`, which is not used; the call
// then returns when they are there.
template <typename R>
int pk_from_delta(const R* delta, int dims, double BoxSize, int axis, int mas_p, int flags, double* out,
                  cplx<R>* keep, bool affine, const double* dmass, double mass, hipStream_t st,
                  double* host = nullptr);

}  // namespace pyl
