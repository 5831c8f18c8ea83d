// Cell-binned mass assignment onto 2-D grids (projected maps), no global atomics on the grid.
//
// The N x N grid is cut into nt x nt tiles of nearly equal width (at most T2 cells; tile of cell c:
// floor(c nt / N)).  A particle's key is the tile of its lowest stencil cell and the 2-bit mask of the axes along
// which the stencil reaches into the next tile.  Exact counting sort by key, then one workgroup per tile:
// 1. k_map_count    keys counted per workgroup in LDS, a row of counts each
// 2. k_map_scan     exclusive sums down the columns: each workgroup's first slot within every key
// 3. k_map_scatter  a step's records are put in key order in LDS and leave in runs of consecutive addresses
// 4. k_map_tile     the records of a tile and of its three lower neighbours whose mask reaches it are summed in
//                   float64 LDS cells; every grid cell is read and written once, with one rounding
// The direct kernel's global float atomics run at 21 G/s: 5 M TSC particles onto 1000^2 took 2.17 ms; here the
// count takes 12 us (40 MB: memory), the scan 5, the scatter 30 (80 MB, and the barriers of a step: one 1024-thread
// workgroup fits a CU beside its LDS) and the tiles 44 (float64 LDS atomics, S^2 a particle).
#include <algorithm>

#include "deposit.hpp"
#include "profile.hpp"
#include "stencil.hpp"
#include "util.hpp"

namespace pyl {

constexpr int MT = 1024;      // threads per workgroup
constexpr int MKP = 4;        // particles per thread per step
constexpr int MKEYS = 4096;   // most keys
constexpr int MKT = MKEYS / MT;
constexpr int MROWS = 256;    // most workgroups of the count and the scatter

struct MapArgs {
    const float* pos;
    const float* W;
    long long n;
    int N, nt, nk, nb;   // grid edge, tiles per edge, keys (4 nt^2), workgroups
    unsigned tmul;
    double inv;
    unsigned* cnt;   // [nb][nk]
    unsigned* tot;   // [nk]
    unsigned* off;   // [nk + 1] first record of each key
    float* rec;      // [n][2 or 3] records in key order
    double mult;     // weight multiplier
    double div;      // the grid is divided by it afterwards (0: not)
    void* grid;
    int zero;        // overwrite instead of accumulate
};

template <int S>
__device__ __forceinline__ int map_key(const MapArgs& a, float x, float y) {
    double w[4];
    const int bx = wrapN(Axis<S>::eval((double)x * a.inv, w), a.N);
    const int by = wrapN(Axis<S>::eval((double)y * a.inv, w), a.N);
    const int tx = __umulhi(bx, a.tmul), ty = __umulhi(by, a.tmul);
    const int hc = (int)__umulhi(bx + S - 1, a.tmul) - tx + 2 * ((int)__umulhi(by + S - 1, a.tmul) - ty);
    return (tx * a.nt + ty) * 4 + hc;
}
// the steps of MT * MKP particles that workgroup bx owns
__device__ __forceinline__ void map_range(const MapArgs& a, long long& s0, long long& s1) {
    const long long nstep = (a.n + MT * MKP - 1) / (MT * MKP), per = (nstep + a.nb - 1) / a.nb;
    s0 = min(nstep, (long long)blockIdx.x * per);
    s1 = min(nstep, s0 + per);
}

template <int S>
__global__ __launch_bounds__(MT) void k_map_count(MapArgs a) {
    __shared__ unsigned h[MKEYS];
    const int tid = threadIdx.x;
    for (int i = tid; i < a.nk; i += MT) h[i] = 0u;
    __syncthreads();
    long long s0, s1;
    map_range(a, s0, s1);
    for (long long step = s0; step < s1; ++step) {
        float x[MKP], y[MKP];
#pragma unroll
        for (int k = 0; k < MKP; ++k) {
            const long long p = (step * MKP + k) * MT + tid;
            if (p < a.n) {
                x[k] = a.pos[2 * p];
                y[k] = a.pos[2 * p + 1];
            }
        }
#pragma unroll
        for (int k = 0; k < MKP; ++k)
            if ((step * MKP + k) * MT + tid < a.n) atomicAdd(&h[map_key<S>(a, x[k], y[k])], 1u);
    }
    __syncthreads();
    for (int i = tid; i < a.nk; i += MT) a.cnt[(long long)blockIdx.x * a.nk + i] = h[i];
}

// columns [64 bx, 64 bx + 64) of cnt: exclusive sums down the rows in place, and the column totals; the rows
// are split over the 16 waves, and all of a wave's rows are loaded before the first is used
__global__ __launch_bounds__(1024) void k_map_scan(MapArgs a) {
    __shared__ unsigned wsum[16][64];
    constexpr int PER = MROWS / 16;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int c = blockIdx.x * 64 + lane;
    const int per = (a.nb + 15) / 16, r0 = min(a.nb, wv * per), r1 = min(a.nb, r0 + per);
    unsigned s = 0u, v[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) v[j] = c < a.nk && r0 + j < r1 ? a.cnt[(long long)(r0 + j) * a.nk + c] : 0u;
#pragma unroll
    for (int j = 0; j < PER; ++j) s += v[j];
    wsum[wv][lane] = s;
    __syncthreads();
    if (c >= a.nk) return;
    unsigned run = 0u;
    for (int j = 0; j < wv; ++j) run += wsum[j][lane];
    if (wv == 15) a.tot[c] = run + s;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        if (r0 + j < r1) a.cnt[(long long)(r0 + j) * a.nk + c] = run;
        run += v[j];
    }
}

template <int S, bool HASW>
__global__ __launch_bounds__(MT) void k_map_scatter(MapArgs a) {
    constexpr int PS = MT * MKP, R = HASW ? 3 : 2;
    __shared__ float rec[PS * R];
    __shared__ unsigned short keys[PS];
    __shared__ unsigned lc[MKEYS];   // the step's records per key, then the first of them in rec
    __shared__ unsigned gd[MKEYS];   // where rec[i] of the key goes: gd + i
    __shared__ unsigned wsum[MT / 64];
    const int tid = threadIdx.x;
    // thread tid's keys are tid * MKT + j; their cursors: the key's first slot (exclusive sum of the totals)
    // plus what the workgroups before this one put there
    unsigned cur[MKT], t[MKT], sum = 0u;
#pragma unroll
    for (int j = 0; j < MKT; ++j) {
        t[j] = tid * MKT + j < a.nk ? a.tot[tid * MKT + j] : 0u;
        sum += t[j];
    }
    unsigned first = block_exscan(sum, wsum);
#pragma unroll
    for (int j = 0; j < MKT; ++j) {
        const int g = tid * MKT + j;
        cur[j] = 0u;
        lc[g] = 0u;
        if (g < a.nk) {
            if (blockIdx.x == 0) a.off[g] = first;
            cur[j] = first + a.cnt[(long long)blockIdx.x * a.nk + g];
            first += t[j];
        }
    }
    if (blockIdx.x == 0 && tid == 0) a.off[a.nk] = (unsigned)a.n;
    long long s0, s1;
    map_range(a, s0, s1);
    float nx[MKP], ny[MKP], nw[MKP];
    auto load = [&](long long step) {
#pragma unroll
        for (int k = 0; k < MKP; ++k) {
            const long long p = (step * MKP + k) * MT + tid;
            if (p < a.n) {
                nx[k] = a.pos[2 * p];
                ny[k] = a.pos[2 * p + 1];
                nw[k] = HASW ? a.W[p] : 0.f;
            }
        }
    };
    if (s0 < s1) load(s0);
    __syncthreads();
    for (long long step = s0; step < s1; ++step) {
        float x[MKP], y[MKP], w[MKP];
        int key[MKP];
        unsigned r[MKP];
#pragma unroll
        for (int k = 0; k < MKP; ++k) {
            x[k] = nx[k];
            y[k] = ny[k];
            w[k] = nw[k];
        }
        if (step + 1 < s1) load(step + 1);   // in flight during this step
#pragma unroll
        for (int k = 0; k < MKP; ++k) {
            key[k] = -1;
            if ((step * MKP + k) * MT + tid < a.n) {
                key[k] = map_key<S>(a, x[k], y[k]);
                r[k] = atomicAdd(&lc[key[k]], 1u);
            }
        }
        __syncthreads();   // (also: every thread has stored the previous step's records)
        unsigned c[MKT], all = 0u;
#pragma unroll
        for (int j = 0; j < MKT; ++j) {
            c[j] = lc[tid * MKT + j];
            all += c[j];
        }
        unsigned o = block_exscan(all, wsum);
#pragma unroll
        for (int j = 0; j < MKT; ++j) {
            lc[tid * MKT + j] = o;
            gd[tid * MKT + j] = cur[j] - o;
            cur[j] += c[j];
            o += c[j];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < MKP; ++k) {
            if (key[k] < 0) continue;
            const unsigned i = lc[key[k]] + r[k];
            rec[i * R] = x[k];
            rec[i * R + 1] = y[k];
            if (HASW) rec[i * R + 2] = w[k];
            keys[i] = (unsigned short)key[k];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < MKT; ++j) lc[tid * MKT + j] = 0u;
        const int m = (int)min((long long)PS, a.n - step * PS);
        for (int i = tid; i < m; i += MT) {
            const long long d = gd[keys[i]] + (unsigned)i;
            if (d >= a.n) continue;   // unreachable: the count gave every particle its slot
#pragma unroll
            for (int q = 0; q < R; ++q) a.rec[d * R + q] = rec[i * R + q];
        }
        __syncthreads();
    }
}

template <int S, typename G, bool HASW, int T2>
__global__ __launch_bounds__(MT) void k_map_tile(MapArgs a) {
    constexpr int R = HASW ? 3 : 2, ROW = T2 + 1;
    __shared__ double acc[T2 * ROW];
    const int tid = threadIdx.x, nt = a.nt, N = a.N;
    const int tx = blockIdx.x / nt, ty = blockIdx.x % nt;
    const int ox = (tx * N + nt - 1) / nt, oy = (ty * N + nt - 1) / nt;
    const int ex = ((tx + 1) * N + nt - 1) / nt - ox, ey = ((ty + 1) * N + nt - 1) / nt - oy;
    for (int i = tid; i < T2 * ROW; i += MT) acc[i] = 0.0;
    __syncthreads();
    // key ranges that reach the tile: its own four, masks 1 and 3 of the lower neighbour along x, masks 2 and 3
    // of the one along y, mask 3 of the diagonal one
    const int lx = (tx + nt - 1) % nt, ly = (ty + nt - 1) % nt;
    const int own = (tx * nt + ty) * 4, nx = (lx * nt + ty) * 4, ny = (tx * nt + ly) * 4, nd = (lx * nt + ly) * 4;
    const int lo[5] = {own, nx + 1, nx + 3, ny + 2, nd + 3}, hi[5] = {own + 4, nx + 2, nx + 4, ny + 4, nd + 4};
    for (int e = 0; e < 5; ++e) {
        const unsigned r0 = a.off[lo[e]], r1 = a.off[hi[e]];
        // the next record of a thread loads while the present one is added (the last loads record r0 again)
        float nr[R], r[R];
        auto fetch = [&](unsigned i) {
            const float* q = a.rec + (size_t)(i < r1 ? i : r0) * R;
#pragma unroll
            for (int c = 0; c < R; ++c) nr[c] = q[c];
        };
        if (r0 < r1) fetch(r0 + tid);
        for (unsigned i = r0 + tid; i < r1; i += MT) {
#pragma unroll
            for (int c = 0; c < R; ++c) r[c] = nr[c];
            fetch(i + MT);
            double w0[S], w1[S];
            int l0 = wrapN(Axis<S>::eval((double)r[0] * a.inv, w0), N) - ox;
            int l1 = wrapN(Axis<S>::eval((double)r[1] * a.inv, w1), N) - oy;
            if (l0 >= T2) l0 -= N;   // a particle of the lower neighbour across the periodic edge
            if (l1 >= T2) l1 -= N;
            const double ww = HASW ? (double)r[2] * a.mult : a.mult;
#pragma unroll
            for (int l = 0; l < S; ++l) {
                const int c0 = l0 + l;
                if ((unsigned)c0 >= (unsigned)ex) continue;
                const double wl = w0[l] * ww;
#pragma unroll
                for (int m = 0; m < S; ++m)
                    if ((unsigned)(l1 + m) < (unsigned)ey) atomicAdd(&acc[c0 * ROW + l1 + m], wl * w1[m]);
            }
        }
    }
    __syncthreads();
    G* __restrict__ grid = (G*)a.grid;
    for (int i = tid; i < T2 * T2; i += MT) {
        const int r = i / T2, c = i % T2;
        if (r >= ex || c >= ey) continue;
        G* p = grid + (long long)(ox + r) * N + oy + c;
        G v = (G)((a.zero ? 0.0 : (double)*p) + acc[r * ROW + c]);
        if (a.div != 0.0) v = v / (G)a.div;
        *p = v;
    }
}

// Tile edge for a grid edge: about 200 tiles or more where the grid allows (one workgroup a CU), at most MKEYS keys,
// and otherwise large tiles, whose fewer keys give the scatter longer runs (5 M TSC onto 1000^2: 88 us with 64 cells,
// 96 with 32; 4 M onto 700^2, 121 tiles of 64: 99 with 64, 74 with 32)
static int map_tile_edge(int N) { return N <= 256 ? 16 : (N <= 832 ? 32 : (N <= 2048 ? 64 : 128)); }

// The direct kernel takes n S^2 / 21e9 s for unordered particles, and down to a third of that in pixel order (several
// share a line; one cell a particle: less again); this route 22 us of launches and 2.4 ps a cell, and then 8 to 25 ps a
// particle.  The line lies where particles in pixel order are even.  Measured, in pixel order (unordered), direct / this in us:
// 250^2 CIC 160 k 24 / 24 (35 / 21), 500^2 PCS 80 k 28 / 27 (72 / 27), 1000^2 CIC 2^18 22 / 25 (52 / 23), 357 k 28 / 26
// (72 / 24), 4000^2 CIC 441 k 73 / 62 (88 / 64); NGP 500^2 1.9 M 46 / 42 (94 / 32), 1000^2 2.0 M 43 / 43 (100 / 35), 4000^2
// 5.0 M 115 / 112 (245 / 103); 2^23 onto 1000^2, CIC 1528 / 192 (1612 / 101).
bool map_supported(int64_t n, int dims, int scheme) {
    if (dims < 32 || dims > 4096 || n >= (1LL << 31)) return false;
    const double cells = (double)dims * dims;
    return (double)n * scheme * scheme >= (scheme == 1 ? 2.0e6 + 0.3 * cells : 1.25e6 + 0.03 * cells);
}

template <int S, typename G, bool HASW>
static void map_launch(const MapArgs& a, int T2, hipStream_t st) {
    hipLaunchKernelGGL((k_map_count<S>), dim3((unsigned)a.nb), dim3(MT), 0, st, a);
    hipLaunchKernelGGL(k_map_scan, dim3((unsigned)((a.nk + 63) / 64)), dim3(1024), 0, st, a);
    hipLaunchKernelGGL((k_map_scatter<S, HASW>), dim3((unsigned)a.nb), dim3(MT), 0, st, a);
    const dim3 g((unsigned)(a.nt * a.nt));
    switch (T2) {
        case 16: hipLaunchKernelGGL((k_map_tile<S, G, HASW, 16>), g, dim3(MT), 0, st, a); break;
        case 32: hipLaunchKernelGGL((k_map_tile<S, G, HASW, 32>), g, dim3(MT), 0, st, a); break;
        case 64: hipLaunchKernelGGL((k_map_tile<S, G, HASW, 64>), g, dim3(MT), 0, st, a); break;
        default: hipLaunchKernelGGL((k_map_tile<S, G, HASW, 128>), g, dim3(MT), 0, st, a); break;
    }
}

template <int S>
static void map_launch_g(const MapArgs& a, int T2, bool f64, hipStream_t st) {
    if (f64)
        a.W ? map_launch<S, double, true>(a, T2, st) : map_launch<S, double, false>(a, T2, st);
    else
        a.W ? map_launch<S, float, true>(a, T2, st) : map_launch<S, float, false>(a, T2, st);
}

int deposit_map(const float* pos, const float* W, int64_t n, int dims, double BoxSize, int scheme, bool f64, bool zero,
                double mult, double div, void* grid, hipStream_t st) {
    MapArgs a{};
    const int T2 = map_tile_edge(dims);
    a.pos = pos;
    a.W = W;
    a.n = n;
    a.N = dims;
    a.nt = (dims + T2 - 1) / T2;
    a.nk = 4 * a.nt * a.nt;
    PYL_CHECK(a.nk <= MKEYS && a.nt >= 2, E_UNSUPPORTED, "2-D binned deposit: grid edge %d", dims);
    a.tmul = tile_mul(dims, a.nt);
    a.inv = dims / BoxSize;
    a.nb = (int)std::max<int64_t>(1, std::min<int64_t>(MROWS, (n + MT * MKP - 1) / (MT * MKP)));
    a.mult = mult;
    a.div = div;
    a.grid = grid;
    a.zero = zero ? 1 : 0;
    int rc = OK;
    unsigned* w = (unsigned*)workspace(WS_SUP, sizeof(unsigned) * ((size_t)(a.nb + 2) * a.nk + 4), &rc);
    if (rc) return rc;
    a.cnt = w;
    a.tot = w + (size_t)a.nb * a.nk;
    a.off = a.tot + a.nk;
    a.rec = (float*)workspace(WS_STAGE, sizeof(float) * (size_t)n * (W ? 3 : 2) + 64, &rc);
    if (rc) return rc;
    StageTimer t("deposit_map", st);
    switch (scheme) {
        case 1: map_launch_g<1>(a, T2, f64, st); break;
        case 2: map_launch_g<2>(a, T2, f64, st); break;
        case 3: map_launch_g<3>(a, T2, f64, st); break;
        case 4: map_launch_g<4>(a, T2, f64, st); break;
        default: set_error("unknown scheme %d", scheme); return E_ARG;
    }
    PYL_HIP(hipGetLastError());
    return OK;
}

}  // namespace pyl
