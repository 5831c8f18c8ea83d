// Cell-binned mass assignment for gfx950: no global atomics on the grid, every cell written once.
//
// The grid is cut into TILE^3 tiles.  A particle belongs to the tile of its lowest stencil cell; its
// halo class is the 3-bit mask of the axes along which its stencil reaches into the next tile (local
// lowest cell > TILE - S).  Buckets are segmented by (tile, class).
// 1. k_bin    particles -> bucket segments.  A workgroup takes BT * KP consecutive particles at a time,
//             counts them per (tile, class) key in an LDS hash table (the positions of the next
//             step are already loading), reserves room with one global atomic per distinct key and
//             writes the records (position, and weight).  Records beyond
//             a segment's capacity go to an overflow list.
// 2. k_ov     the overflow list is grouped by tile with an exact count + scan (empty in the common
//             case: the kernel then only reads a zero counter).
// 3. k_tile   one workgroup per tile accumulates into TILE^3 float64 LDS cells (ds_add_f64: the per-
//             cell sum is exact to float64, the "compensated" accumulator) the stencil weights that
//             fall inside the tile, from its own particles and from those of its 7 lower neighbours
//             whose class reaches it, then writes every cell once with one rounding.
// The grid edge need not be a multiple of TILE: a ragged edge N is cut into nt = ceil(N / TILE) tiles of
// nearly equal width (TILE / 2 to TILE cells), tile t of cell c being floor(c nt / N).
// Output modes: accumulate into the existing grid (MAS_library.MA semantics), overwrite, or the
// overdensity delta = rho * a - 1 (a = N^3 / mass) evaluated in float64 before the single rounding.
#include <math.h>

#include <algorithm>

#include "binned.hpp"
#include "deposit.hpp"
#include "profile.hpp"
#include "stencil.hpp"
#include "util.hpp"

namespace pyl {

constexpr int BT = 512;    // k_bin: threads per workgroup
constexpr int KP = 4;      // k_bin: particles per thread per step
constexpr int HT = 4096;   // k_bin: LDS hash slots (> BT * KP, so an insertion always finds a slot)
constexpr int TT = 512;    // k_tile: threads per workgroup
constexpr int OT = 1024;   // k_ov: threads per workgroup
constexpr int OB = 256;    // k_ov: workgroups (per job)
// particles per cell from which CIC tiles accumulate in register runs (measured at 512^3 particles: 8 per
// cell 0.94 -> 0.78 ms, 4.1: 0.82 -> 0.75, 2.4: equal, 1.5: 0.75 -> 0.81; NGP gains nothing)
constexpr double RUN_PPC = 3.0;
// row stride of the float64 LDS accumulator of a tile: TILE + 1 doubles, so that particles one row
// apart in y (neighbours in the input along z fill a row, then the next) land on LDS banks 34 apart
// (measured on the 512^3 lattice: k_tile 0.88 -> 0.77 ms; strides 18/20/24 and padded planes were slower)
constexpr int TROW = TILE + 1;
static_assert(HT % BT == 0, "hash slots per thread");
constexpr int HBITS = 12;   // log2(HT): the slot of a key is the top HBITS bits of its multiplicative hash
static_assert(HT == 1 << HBITS, "HT must be 2^HBITS");
static_assert(HT > BT * KP, "every key of a step must find a hash slot");

template <int S>
__device__ __forceinline__ int halo_class(int bx, int by, int bz) {
    return ((bx % TILE) > TILE - S ? 1 : 0) | ((by % TILE) > TILE - S ? 2 : 0) | ((bz % TILE) > TILE - S ? 4 : 0);
}

// AGG: 0 every lane counts itself, 1 runs of equal keys are counted once, 2 a.agg decides (batched
// launches, whose jobs differ; ragged grids).  RAG: the grid edge is no multiple of TILE.
template <int S, bool HASW, int AGG, bool RAG>
__device__ __forceinline__ void bin_body(const BinArgs& a, Blk B) {
    constexpr int R = HASW ? 4 : 3;
    constexpr long long PS = (long long)BT * KP;   // particles per step
    // a slot holds a key of the step, then (after the reservations) the first index of the key's records
    __shared__ int hkey[HT];
    __shared__ unsigned hcnt[HT];
    __shared__ int hused[BT * KP];   // slots that hold a key this step, in insertion order
    __shared__ unsigned nused, nov, ovbase;   // of the step: keys; records beyond their segments, and their first slot
    __shared__ int scap[8], scofs[8];
    const int tid = threadIdx.x;
    const bool grouped = a.sel && *a.sel;
    const float* __restrict__ pos = grouped ? a.spos : a.pos;
    const float* __restrict__ W = grouped ? a.sw : a.W;
    if (tid < 8) {
        scap[tid] = a.cap[tid];
        scofs[tid] = a.cofs[tid];
    }
    for (int i = tid; i < HT; i += BT) {
        hkey[i] = -1;
        hcnt[i] = 0u;
    }
    if (tid == 0) nused = nov = 0u;
    __syncthreads();
    const long long nstep = (a.n + PS - 1) / PS;
    // particle k of this thread in a step: step * PS + k * BT + tid (coalesced for each k)
    float px[KP], py[KP], pz[KP], pw[KP];
    auto load = [&](long long step) {
#pragma unroll
        for (int k = 0; k < KP; ++k) {
            const long long p = step * PS + k * BT + tid;
            if (p < a.n) {
                float c[3] = {pos[3 * p], pos[3 * p + 1], pos[3 * p + 2]};
                if (a.rsd.vel) {
                    const int ax = a.rsd.axis;
                    c[ax] = rsd_shift(c[ax], a.rsd.vel[3 * p + ax], a.rsd.fac, a.rsd.box);
                }
                px[k] = c[0];
                py[k] = c[1];
                pz[k] = c[2];
                pw[k] = HASW ? W[p] : 0.f;
            }
        }
    };
    // each XCD (workgroups go round-robin over the XCDS of the chip) takes one contiguous range of
    // steps, so that records of one segment written at about the same time share an L2, and each
    // workgroup of the XCD a contiguous part of it: consecutive steps of one workgroup append to the
    // same segments, and workgroups running at the same time reserve in different segments (measured
    // 3 % faster than interleaving the workgroups step by step)
    const long long GX = B.gx / XCDS, per = (nstep + XCDS - 1) / XCDS;
    const long long s_beg = (long long)(B.x % XCDS) * per;
    const long long s_end = min(nstep, s_beg + per);
    const long long bper = (per + GX - 1) / GX;
    const long long b_beg = s_beg + (long long)(B.x / XCDS) * bper;
    const long long b_end = min(s_end, b_beg + bper);
    long long step = b_beg;
    if (step < b_end) load(step);
    for (; step < b_end; ++step) {
        float x[KP], y[KP], z[KP], w[KP];
#pragma unroll
        for (int k = 0; k < KP; ++k) {
            x[k] = px[k];
            y[k] = py[k];
            z[k] = pz[k];
            w[k] = pw[k];
        }
        if (step + 1 < b_end) load(step + 1);   // in flight during this step
        int key[KP];
        // slot of the key and the record's rank among the key's of the step, in one register (with two, and the overflow's
        // count, a wave less fits: 128^3 CIC 2^24 268 -> 278 us)
        unsigned sr[KP];
        static_assert(HT <= 1 << 16 && BT * KP <= 1 << 16, "two halves of a word");
#pragma unroll
        for (int k = 0; k < KP; ++k) {
            const long long p = step * PS + k * BT + tid;
            const bool valid = p < a.n;
            key[k] = -1;
            sr[k] = 0u;
            if (valid) {
                double ww[4];
                const int bx = wrapN(Axis<S>::eval((double)x[k] * a.inv, ww), a.N);
                const int by = wrapN(Axis<S>::eval((double)y[k] * a.inv, ww), a.N);
                const int bz = wrapN(Axis<S>::eval((double)z[k] * a.inv, ww), a.N);
                if (RAG) {
                    // the stencil reaches into the next tile when its last cell lies there (tile nt
                    // past the periodic edge)
                    const unsigned m = a.tmul;
                    const int tx = __umulhi(bx, m), ty = __umulhi(by, m), tz = __umulhi(bz, m);
                    const int hc = (int)__umulhi(bx + S - 1, m) - tx + 2 * ((int)__umulhi(by + S - 1, m) - ty) +
                                   4 * ((int)__umulhi(bz + S - 1, m) - tz);
                    key[k] = ((tx * a.nt + ty) * a.nt + tz) * 8 + hc;
                } else {
                    key[k] = (((bx / TILE) * a.nt + by / TILE) * a.nt + bz / TILE) * 8 + halo_class<S>(bx, by, bz);
                }
            }
            // at most BT * KP distinct keys per step in HT slots: the probe always ends
            auto probe = [&](int kk) {
                int s0 = (int)(((unsigned)kk * 2654435761u) >> (32 - HBITS));
                for (;;) {
                    const int prev = atomicCAS(&hkey[s0], -1, kk);
                    if (prev == -1) hused[atomicAdd(&nused, 1u)] = s0;
                    if (prev == -1 || prev == kk) return s0;
                    s0 = (s0 + 1) & (HT - 1);
                }
            };
            if (AGG == 1 || (AGG == 2 && a.agg)) {
                // (uniform over the launch: every lane runs the shuffles) runs of equal keys in
                // consecutive lanes: the first lane of a run probes the table and counts the whole run,
                // the others take the slot and their rank from it.  Invalid lanes (key -1) form runs of
                // their own, which are skipped below.
                const int lane = tid & 63;
                const int kprev = __shfl_up(key[k], 1);
                const unsigned long long hm = __ballot(lane == 0 || kprev != key[k]);
                const unsigned long long le = lane == 63 ? ~0ull : ((2ull << lane) - 1ull);   // lanes <= lane
                const int start = 63 - __clzll((long long)(hm & le));   // lane 0 always starts a run
                const unsigned long long gt = hm & ~le;
                const int end = gt ? __ffsll((long long)gt) - 1 : 64;
                int s0 = 0;
                unsigned base = 0u;
                if (valid && start == lane) {
                    s0 = probe(key[k]);
                    base = atomicAdd(&hcnt[s0], (unsigned)(end - start));
                }
                sr[k] = __shfl((unsigned)s0 | base << 16, start) + ((unsigned)(lane - start) << 16);
            } else if (valid) {
                const int s0 = probe(key[k]);
                sr[k] = (unsigned)s0 | atomicAdd(&hcnt[s0], 1u) << 16;
            }
        }
        __syncthreads();
        // one reservation per key of the step: its records go to [base, base + hcnt) of its segment;
        // the base replaces the key in the slot.  What lies beyond the segment gets consecutive slots of the
        // overflow list, one reservation for the whole step (one atomic a record on that one counter took 1 ms for 4 M
        // of 8 M clustered particles): the count becomes the key's first slot, less its first index there
        const unsigned nu = nused;
        for (unsigned i = tid; i < nu; i += BT) {
            const int sl = hused[i], k = hkey[sl];
            const unsigned cnt = hcnt[sl], base = atomicAdd(&a.fill[k], cnt), first = max(base, (unsigned)scap[k & 7]);
            hkey[sl] = (int)base;
            if (base + cnt > first) hcnt[sl] = atomicAdd(&nov, base + cnt - first) - first;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < KP; ++k) {
            if (key[k] < 0) continue;
            const int c = key[k] & 7;
            const unsigned idx = (unsigned)hkey[sr[k] & 0xffffu] + (sr[k] >> 16);
            if (idx >= (unsigned)scap[c]) continue;
            float* r = a.bucket + ((long long)(key[k] >> 3) * a.CT + scofs[c] + idx) * R;
            r[0] = x[k];
            r[1] = y[k];
            r[2] = z[k];
            if (HASW) r[3] = w[k];
        }
        __syncthreads();
        if (nov) {   // (here, behind the stores, the look at it costs least)
            if (tid == 0) ovbase = atomicAdd(a.ov_count, nov);
            __syncthreads();
#pragma unroll
            for (int k = 0; k < KP; ++k) {
                if (key[k] < 0) continue;
                const unsigned sl = sr[k] & 0xffffu, idx = (unsigned)hkey[sl] + (sr[k] >> 16), cap = (unsigned)scap[key[k] & 7];
                if (idx < cap) continue;
                const unsigned o = ovbase + hcnt[sl] + idx;
                a.ov_idx[o] = (unsigned long long)(idx - cap) << 32 | (unsigned long long)(step * PS + k * BT + tid);
                a.ov_key[o] = (unsigned)key[k];
            }
            __syncthreads();
        }
        for (unsigned i = tid; i < nu; i += BT) {
            const int sl = hused[i];
            hkey[sl] = -1;
            hcnt[sl] = 0u;
        }
        if (tid == 0) nused = nov = 0u;
        __syncthreads();
    }
}

template <int S, bool HASW, int AGG, bool RAG>
__global__ __launch_bounds__(BT) void k_bin(BinArgs a) { bin_body<S, HASW, AGG, RAG>(a, own_blk()); }
template <int S, bool HASW>
__global__ __launch_bounds__(BT) void k_bin_b(const BinArgs* __restrict__ tab,
                                                 const unsigned* __restrict__ start, int nj) {
    PYL_BATCH_BLK(start, nj);
    bin_body<S, HASW, 2, false>(tab[bj_], blk_);
}

// Overflow grouping in one launch: the first workgroup to arrive counts and scans, then all that have records copy
// them.  A tile's records are what its class fills exceed their capacities by, and a record's place among them is its
// index in the segment beyond the capacity, so the list itself is not counted and nothing is added to.  The others wait
// for a workgroup that is running by then (it took its ticket) and waits for none, so the wait ends whatever else the
// card runs; workgroups past the end of the list leave at once.  Nothing overflowed (every group is empty and k_tile
// reads no offset): one read and out, 4.7 us where three launches took 14.  One thread of a waiting workgroup makes its
// fence (the barrier orders the others behind it).
__device__ __forceinline__ unsigned ov_over(const OvArgs& a, long long tile, unsigned (&k)[8]) {
    const uint4 fa = ((const uint4*)a.fill)[2 * tile], fb = ((const uint4*)a.fill)[2 * tile + 1];
    k[0] = fa.x, k[1] = fa.y, k[2] = fa.z, k[3] = fa.w, k[4] = fb.x, k[5] = fb.y, k[6] = fb.z, k[7] = fb.w;
    unsigned s = 0u;
#pragma unroll
    for (int c = 0; c < 8; ++c) s += k[c] -= min(k[c], (unsigned)a.cap[c]);
    return s;
}
// thread t takes the tiles t, t + OT, ...: their groups follow one another in that order
__device__ __forceinline__ void ov_scan(const OvArgs& a) {
    __shared__ unsigned wsum[OT / 64];
    const int tid = threadIdx.x, n = a.ntiles;
    unsigned k[8], s = 0u;
    for (int i = tid; i < n; i += OT) {
        const unsigned o = ov_over(a, i, k);
        a.ocnt[i] = o;
        s += o;
    }
    unsigned run = block_exscan(s, wsum);
    for (int i = tid; i < n; i += OT) {
        a.ooff[i] = run;
        run += a.ocnt[i];
    }
}

template <bool HASW>
__device__ __forceinline__ void ov_body(const OvArgs& a, Blk B) {
    constexpr int R = HASW ? 4 : 3;
    __shared__ unsigned ticket;
    const long long n = *a.ov_count;
    if ((long long)B.x * OT >= n) return;
    if (threadIdx.x == 0) ticket = atomicAdd(&a.turn[0], 1u);
    __syncthreads();
    if (ticket == 0u) {
        ov_scan(a);
        __threadfence();
        __syncthreads();
        if (threadIdx.x == 0) __hip_atomic_store(&a.turn[1], 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    } else {
        if (threadIdx.x == 0) {
            // (an acquire for every look would keep emptying the caches that the scan works in)
            while (__hip_atomic_load(&a.turn[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u)
                __builtin_amdgcn_s_sleep(8);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        __syncthreads();
    }
    const bool sel = a.sel && *a.sel;
    const float* __restrict__ pos = sel ? a.spos : a.pos;
    const float* __restrict__ W = sel ? a.sw : a.W;
    for (long long i = (long long)B.x * OT + threadIdx.x; i < n; i += (long long)B.gx * OT) {
        const unsigned key = a.ov_key[i], t = key >> 3, cls = key & 7u;
        const unsigned long long e = a.ov_idx[i];
        const long long p = (long long)(e & 0xffffffffull);
        unsigned k[8], s = a.ooff[t] + (unsigned)(e >> 32);
        ov_over(a, t, k);
#pragma unroll
        for (unsigned c = 0; c < 8; ++c) s += c < cls ? k[c] : 0u;
        float* r = a.grouped + (long long)s * R;
        float c[3] = {pos[3 * p], pos[3 * p + 1], pos[3 * p + 2]};
        if (a.rsd.vel) c[a.rsd.axis] = rsd_shift(c[a.rsd.axis], a.rsd.vel[3 * p + a.rsd.axis], a.rsd.fac, a.rsd.box);
        r[0] = c[0];
        r[1] = c[1];
        r[2] = c[2];
        if (HASW) r[3] = W[p];
        a.gcls[s] = cls;
    }
}
template <bool HASW>
__global__ __launch_bounds__(OT) void k_ov(OvArgs a) { ov_body<HASW>(a, own_blk()); }
// batched: job blockIdx.y
template <bool HASW>
__global__ __launch_bounds__(OT) void k_ov_b(const OvArgs* __restrict__ tab) {
    const OvArgs& a = tab[blockIdx.y];
    ov_body<HASW>(a, own_blk());
}

enum { OUT_ACC = 0, OUT_SET = 1, OUT_DELTA = 2 };

template <typename G, int MODE>
__device__ __forceinline__ void put(G* __restrict__ grid, long long g, double rho, double a) {
    if (MODE == OUT_ACC)
        grid[g] = (G)((double)grid[g] + rho);
    else if (MODE == OUT_SET)
        grid[g] = (G)rho;
    else
        grid[g] = (G)(rho * a - 1.0);
}


// lowest cell and width (cells, at most TILE) of a tile along each axis
struct TileBox {
    int ox, oy, oz, ex, ey, ez;
};

// the stencil weights of one particle that fall inside the tile t
// (CLIP = false: a particle of the tile itself whose stencil stays inside it)
template <int S, bool HASW, bool CLIP, bool UNIT>
__device__ __forceinline__ void accumulate(double* acc, const float* r, int N, const TileBox& t, double inv,
                                           double mult) {
    double w0[S], w1[S], w2[S];
    int l0 = wrapN(Axis<S>::eval((double)r[0] * inv, w0), N) - t.ox;
    int l1 = wrapN(Axis<S>::eval((double)r[1] * inv, w1), N) - t.oy;
    int l2 = wrapN(Axis<S>::eval((double)r[2] * inv, w2), N) - t.oz;
    // a particle of the lower neighbour across the periodic boundary
    if (l0 >= TILE) l0 -= N;
    if (l1 >= TILE) l1 -= N;
    if (l2 >= TILE) l2 -= N;
    const double ww = HASW ? (double)r[3] * mult : mult;
#pragma unroll
    for (int l = 0; l < S; ++l) {
        const int c0 = l0 + l;
        if (CLIP && (unsigned)c0 >= (unsigned)t.ex) continue;
#pragma unroll
        for (int m = 0; m < S; ++m) {
            const int c1 = l1 + m;
            if (CLIP && (unsigned)c1 >= (unsigned)t.ey) continue;
            const double wlm = UNIT ? w0[l] * w1[m] : w0[l] * w1[m] * ww;   // UNIT: no weights, mult == 1
            double* row = acc + (c0 * TILE + c1) * TROW;
#pragma unroll
            for (int q = 0; q < S; ++q) {
                const int c2 = l2 + q;
                if (!CLIP || (unsigned)c2 < (unsigned)t.ez) atomicAdd(row + c2, wlm * w2[q]);
            }
        }
    }
}

// accumulate() with the 1-D weights and their products in float32 (Axis32); each contribution is
// added to the float64 LDS cell
template <int S, bool HASW, bool CLIP, bool UNIT>
__device__ __forceinline__ void accumulate32(double* acc, const float* r, int N, const TileBox& t, double inv,
                                             float mult) {
    float w0[S], w1[S], w2[S];
    int l0 = wrapN(Axis32<S>::eval((double)r[0] * inv, w0), N) - t.ox;
    int l1 = wrapN(Axis32<S>::eval((double)r[1] * inv, w1), N) - t.oy;
    int l2 = wrapN(Axis32<S>::eval((double)r[2] * inv, w2), N) - t.oz;
    if (l0 >= TILE) l0 -= N;
    if (l1 >= TILE) l1 -= N;
    if (l2 >= TILE) l2 -= N;
    const float ww = HASW ? r[3] * mult : mult;
#pragma unroll
    for (int l = 0; l < S; ++l) {
        const int c0 = l0 + l;
        if (CLIP && (unsigned)c0 >= (unsigned)t.ex) continue;
#pragma unroll
        for (int m = 0; m < S; ++m) {
            const int c1 = l1 + m;
            if (CLIP && (unsigned)c1 >= (unsigned)t.ey) continue;
            const float wlm = UNIT ? w0[l] * w1[m] : w0[l] * w1[m] * ww;
            double* row = acc + (c0 * TILE + c1) * TROW;
#pragma unroll
            for (int q = 0; q < S; ++q) {
                const int c2 = l2 + q;
                if (!CLIP || (unsigned)c2 < (unsigned)t.ez) atomicAdd(row + c2, (double)(wlm * w2[q]));
            }
        }
    }
}

// ACC: ACC_F64 (float64 weights, float64 cell sums), ACC_RUN (the same, with register runs of the
// stencil block for dense CIC inputs) or ACC_F32W (float32 weights and products, float64
// cell sums).  Both run at the same speed on gfx950 (the kernel is bound by loads and LDS
// atomics, not by float64 arithmetic); a float32 LDS cell (ds_add_f32) was measured about six times
// slower than the float64 one (ds_add_f64) in this kernel, and a TwoSum-compensated float32 cell
// (returning atomics) twelve times slower, so the float64 cell is the accumulator of every mode.
enum { ACC_F64 = 0, ACC_F32W = 1, ACC_RUN = 2 };

int dense_acc(int acc, int scheme, int64_t n, int dims) {
    return acc == ACC_F64 && scheme == 2 && (double)n >= RUN_PPC * (double)dims * dims * dims ? ACC_RUN : acc;
}

// k_bin counts runs of equal keys once from AGG_PPC particles per cell up: spatially ordered inputs
// then give runs of tens of lanes per key, whose per-lane LDS atomics on one word serialise (512^3
// lattice particles onto 256^3: 1.68 -> 1.41 ms for the deposit); at one particle per cell 512^3 the
// shuffles cost more than they save (+2 %), and unordered inputs are unchanged either way
constexpr double AGG_PPC = 2.0;
int bin_agg(int64_t n, int dims) { return (double)n >= AGG_PPC * (double)dims * dims * dims ? 1 : 0; }

template <int S, typename G, bool HASW, int MODE, bool UNIT, int ACC, bool RAG>
__device__ __forceinline__ void tile_body(const TileArgs& a, Blk B) {
    constexpr int R = HASW ? 4 : 3;
    constexpr int NE = 72;   // 8 neighbours (d = 0 own) x (8 class segments + 1 overflow group)
    __shared__ double acc[TILE * TILE * TROW];
    __shared__ long long sbase[NE];
    __shared__ unsigned scnt[NE];
    __shared__ unsigned sstart[NE + 1];
    const int tid = threadIdx.x;
    // contiguous runs of tiles per XCD: the lower neighbours whose halo records a tile reads were
    // mostly processed just before on the same XCD
    const int nt = a.nt, ntl = nt * nt * nt, tper = (ntl + XCDS - 1) / XCDS;
    const int t = (int)(B.x % XCDS) * tper + (int)(B.x / XCDS);
    if (t >= ntl) return;
    const int tx = t / (nt * nt), ty = (t / nt) % nt, tz = t % nt;
    for (int i = tid; i < TILE * TILE * TROW; i += TT) acc[i] = 0.0;
    // entry e = d * 9 + c: class segment c (< 8) or the overflow group (c = 8) of the neighbour
    // t - d; a neighbour's particles reach this tile when their class contains d
    if (tid < NE) {
        const int d = tid / 9, c = tid % 9;
        const int dx = d & 1, dy = (d >> 1) & 1, dz = (d >> 2) & 1;
        const long long tn = ((long long)((tx - dx + nt) % nt) * nt + (ty - dy + nt) % nt) * nt + (tz - dz + nt) % nt;
        unsigned n = 0u;
        long long b = 0;
        if (c < 8) {
            if ((c & d) == d) {
                n = min(a.fill[tn * 8 + c], (unsigned)a.cap[c]);
                b = tn * a.CT + a.cofs[c];
            }
        } else {
            n = a.ocnt[tn];
            b = a.ooff[tn];
        }
        scnt[tid] = n;
        sbase[tid] = b;
    }
    __syncthreads();
    if (tid < 64) {
        // exclusive prefix of the 72 counts: lane l holds entries 2l and 2l+1
        const int e0 = 2 * tid, e1 = 2 * tid + 1;
        const unsigned c0 = e0 < NE ? scnt[e0] : 0u, c1 = e1 < NE ? scnt[e1] : 0u;
        unsigned v = c0 + c1;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const unsigned u = __shfl_up(v, o, 64);
            if (tid >= o) v += u;
        }
        const unsigned ex = v - c0 - c1;
        if (e0 < NE) sstart[e0] = ex;
        if (e1 < NE) sstart[e1] = ex + c0;
        if (e1 == NE - 1) sstart[NE] = v;
    }
    __syncthreads();
    const unsigned tot = sstart[NE];
    TileBox box{tx * TILE, ty * TILE, tz * TILE, TILE, TILE, TILE};
    if (RAG) {
        box.ox = (tx * a.N + nt - 1) / nt;
        box.oy = (ty * a.N + nt - 1) / nt;
        box.oz = (tz * a.N + nt - 1) / nt;
        box.ex = ((tx + 1) * a.N + nt - 1) / nt - box.ox;
        box.ey = ((ty + 1) * a.N + nt - 1) / nt - box.oy;
        box.ez = ((tz + 1) * a.N + nt - 1) / nt - box.oz;
    }
    // RP records per thread per step; the records of the next step load while those of this step
    // accumulate.  The loads are unconditional (an exhausted slot reads record 0 and class word 0,
    // both always allocated) and their values are first used a step later, so only they stay in
    // flight across the accumulation.
    constexpr int RP = 2;
    int e = 0;
    float cr[RP][4], nr[RP][4];
    int ce[RP], ne[RP];
    unsigned cg[RP], ng[RP];
    auto fetch = [&](unsigned f) {
#pragma unroll
        for (int j = 0; j < RP; ++j) {
            const unsigned fj = f + j * TT;
            const bool valid = fj < tot;
            if (valid)
                while (fj >= sstart[e + 1]) ++e;
            const bool ovg = e % 9 == 8;
            const long long i = valid ? sbase[e] + (fj - sstart[e]) : 0;
            const float* q = (valid && ovg ? a.grouped : a.bucket) + i * R;
#pragma unroll
            for (int c = 0; c < R; ++c) nr[j][c] = q[c];
            ng[j] = a.gcls[valid && ovg ? i : 0];
            ne[j] = valid ? e : -1;
        }
    };
    auto advance = [&]() {
#pragma unroll
        for (int j = 0; j < RP; ++j) {
#pragma unroll
            for (int c = 0; c < 4; ++c) cr[j][c] = nr[j][c];
            ce[j] = ne[j];
            cg[j] = ng[j];
        }
    };
    // phase 1: the tile's own class-0 records (most of them): one contiguous segment whose stencils
    // stay inside the tile -- no entry search, no clipping, no overflow class word
    const unsigned n0 = scnt[0];
    const float* q0 = a.bucket + sbase[0] * R;
    if constexpr (S == 2 && ACC == ACC_RUN) {
        // Runs (dense inputs): a thread takes groups of RG consecutive records (consecutive particles
        // of the input, mostly neighbours along z) and keeps the float64 sums of its current S^3
        // stencil block in registers.  A record with the same lowest cell adds to them; one cell
        // further along z, the block's lower z face goes to LDS and the block moves up (CIC: 4 LDS
        // atomics instead of 8); any other record sends the whole block to LDS.  With several
        // particles per cell most records add in registers (512^3 particles onto 256^3: 0.95 ->
        // 0.79 ms); with about one per cell the strided group loads and the register blocks cost more
        // than the atomics they save, so the host picks this mode by particles per cell.
        constexpr int RG = 2;
        double blk[S][S][S];
        int b0 = -1, b1 = 0, b2 = 0;   // lowest cell of the block (b0 < 0: none yet)
        float gr[RG][4], gn[RG][4];
        auto fetchg = [&](unsigned g) {
#pragma unroll
            for (int k = 0; k < RG; ++k) {
                const unsigned fk = g * RG + k;
                const float* q = q0 + (size_t)(fk < n0 ? fk : 0u) * R;   // record 0 of the segment always exists
#pragma unroll
                for (int c = 0; c < R; ++c) gn[k][c] = q[c];
            }
        };
        auto all_out = [&]() {
#pragma unroll
            for (int l = 0; l < S; ++l)
#pragma unroll
                for (int m = 0; m < S; ++m) {
                    double* row = acc + ((b0 + l) * TILE + b1 + m) * TROW + b2;
#pragma unroll
                    for (int q = 0; q < S; ++q) atomicAdd(row + q, blk[l][m][q]);
                }
        };
        const unsigned ngr = (n0 + RG - 1) / RG;
        fetchg(tid);
        for (unsigned g = tid; g < ngr; g += TT) {
#pragma unroll
            for (int k = 0; k < RG; ++k)
#pragma unroll
                for (int c = 0; c < 4; ++c) gr[k][c] = gn[k][c];
            fetchg(g + TT);
#pragma unroll
            for (int k = 0; k < RG; ++k) {
                if (g * RG + k >= n0) break;
                double w0[S], w1[S], w2[S];
                int l0 = wrapN(Axis<S>::eval((double)gr[k][0] * a.inv, w0), a.N) - box.ox;
                int l1 = wrapN(Axis<S>::eval((double)gr[k][1] * a.inv, w1), a.N) - box.oy;
                int l2 = wrapN(Axis<S>::eval((double)gr[k][2] * a.inv, w2), a.N) - box.oz;
                if (l0 >= TILE) l0 -= a.N;
                if (l1 >= TILE) l1 -= a.N;
                if (l2 >= TILE) l2 -= a.N;
                if (l0 != b0 || l1 != b1 || l2 != b2) {
                    if (S == 2 && l0 == b0 && l1 == b1 && l2 == b2 + 1) {
#pragma unroll
                        for (int l = 0; l < S; ++l)
#pragma unroll
                            for (int m = 0; m < S; ++m) {
                                atomicAdd(acc + ((b0 + l) * TILE + b1 + m) * TROW + b2, blk[l][m][0]);
                                blk[l][m][0] = blk[l][m][S - 1];
                                blk[l][m][S - 1] = 0.0;
                            }
                    } else {
                        if (b0 >= 0) all_out();
#pragma unroll
                        for (int l = 0; l < S; ++l)
#pragma unroll
                            for (int m = 0; m < S; ++m)
#pragma unroll
                                for (int q = 0; q < S; ++q) blk[l][m][q] = 0.0;
                        b0 = l0;
                        b1 = l1;
                    }
                    b2 = l2;
                }
                const double ww = HASW ? (double)gr[k][3] * a.mult : a.mult;
#pragma unroll
                for (int l = 0; l < S; ++l)
#pragma unroll
                    for (int m = 0; m < S; ++m) {
                        const double wlm = UNIT ? w0[l] * w1[m] : w0[l] * w1[m] * ww;
#pragma unroll
                        for (int q = 0; q < S; ++q) blk[l][m][q] += wlm * w2[q];
                    }
            }
        }
        if (b0 >= 0) all_out();
    } else {
        auto fetch0 = [&](unsigned f) {
#pragma unroll
            for (int j = 0; j < RP; ++j) {
                const unsigned fj = f + j * TT;
                const float* q = q0 + (size_t)(fj < n0 ? fj : 0u) * R;   // record 0 of the segment always exists
#pragma unroll
                for (int c = 0; c < R; ++c) nr[j][c] = q[c];
            }
        };
        fetch0(tid);
        for (unsigned f = tid; f < n0; f += RP * TT) {
#pragma unroll
            for (int j = 0; j < RP; ++j)
#pragma unroll
                for (int c = 0; c < 4; ++c) cr[j][c] = nr[j][c];
            fetch0(f + RP * TT);
#pragma unroll
            for (int j = 0; j < RP; ++j) {
                if (f + j * TT >= n0) break;
                if (ACC == ACC_F32W)
                    accumulate32<S, HASW, false, UNIT>(acc, cr[j], a.N, box, a.inv, (float)a.mult);
                else
                    accumulate<S, HASW, false, UNIT>(acc, cr[j], a.N, box, a.inv, a.mult);
            }
        }
    }
    // phase 2: halo-class segments of this tile and its lower neighbours, overflow groups
    fetch(n0 + tid);
    advance();
    for (unsigned f = n0 + tid; f < tot; f += RP * TT) {
        fetch(f + RP * TT);
#pragma unroll
        for (int j = 0; j < RP; ++j) {
            const int ej = ce[j];
            // entry 0: the tile's own class-0 particles, whose stencils stay inside the tile;
            // an overflow group's record reaches this tile when its class contains the offset
            const unsigned d = (unsigned)(ej / 9);
            const bool ok = ej >= 0 && (ej % 9 < 8 || (cg[j] & d) == d);
            if (ACC == ACC_F32W) {
                if (ok) accumulate32<S, HASW, true, UNIT>(acc, cr[j], a.N, box, a.inv, (float)a.mult);
            } else if (ok) {
                accumulate<S, HASW, true, UNIT>(acc, cr[j], a.N, box, a.inv, a.mult);
            }
        }
        advance();
    }
    __syncthreads();
    G* grid = (G*)a.grid;
    const double am = (MODE == OUT_DELTA) ? (double)a.N * a.N * a.N / (a.dmass ? a.dmass[0] : a.mass) : 0.0;
    const long long N = a.N;
    for (int idx = tid; idx < TILE * TILE * TILE; idx += TT) {
        const int i = idx / (TILE * TILE), j = (idx / TILE) % TILE, k = idx % TILE;
        if (RAG && (i >= box.ex || j >= box.ey || k >= box.ez)) continue;
        const long long g = (((long long)box.ox + i) * N + box.oy + j) * N + box.oz + k;
        put<G, MODE>(grid, g, acc[(i * TILE + j) * TROW + k], am);
    }
}

// RAG: the grid edge is no multiple of TILE: tile t holds the cells [ceil(t N / nt), ceil((t + 1) N / nt))
template <int S, typename G, bool HASW, int MODE, bool UNIT, int ACC, bool RAG>
__global__ __launch_bounds__(TT) void k_tile(TileArgs a) {
    tile_body<S, G, HASW, MODE, UNIT, ACC, RAG>(a, own_blk());
}
template <int S, typename G, bool HASW, int MODE, bool UNIT, int ACC>
__global__ __launch_bounds__(TT) void k_tile_b(const TileArgs* __restrict__ tab,
                                                  const unsigned* __restrict__ start, int nj) {
    PYL_BATCH_BLK(start, nj);
    tile_body<S, G, HASW, MODE, UNIT, ACC, false>(tab[bj_], blk_);
}

// ------------------------------------------------------------------ presort for unordered inputs
// Particles in no spatial order give k_bin one key per particle: one global atomic each and 12-byte
// scattered records.  The presort first groups them by supertile (whole columns of tiles, at most SUPMAX
// groups): k_sup_count counts the groups of every workgroup's particles, k_sup_scatter turns the counts into
// its workgroups' first slots per group and copies the particles there.  No global atomics:
// with one global reservation per group and step instead, 3 M weighted particles took 46 + 46 us, most of
// it in atomics on a hundred addresses.
// k_bin then reads the grouped copy, where neighbouring particles share keys as in an ordered input.
constexpr int PT = 1024;   // presort kernels: threads per workgroup
constexpr int PKP = 8;    // particles per thread per step
// PRESORT_PROBE: particles, and (tile, class) keys of the grid, from which the device looks for a spatial order.  Unordered
// particles, grouped / as they are, us: CIC 128^3 2^17 35 / 27, 2^19 43 / 43, 2^20 50 / 64, 256^3 2^18 75 / 71, 2^20 85 / 109;
// at 2^20 and more 32^3 CIC (64 keys) 267 / 250, 64^3 NGP (64) 52 / 41, 48^3 CIC (216) 113 / 109, 64^3 CIC (512) 71 / 87,
// 128^3 NGP (512) 41 / 44.  A look that finds an order costs 2.
constexpr int64_t PROBE_MIN = 1 << 20;
constexpr long long PROBE_KEYS = 512;
// groups aimed at: more give k_bin fewer keys a step (3 M particles onto 320^3: 60 us with 128, 40 with 256, 29
// with 512), fewer give the scatter longer runs (24 / 24 / 25 us)
constexpr int SUPGROUPS = 512;
constexpr int SUPBLOCKS = 256;   // most workgroups of the count and the scatter

__device__ __forceinline__ void sup_load(const SupArgs& a, long long p, float& x, float& y, float& z) {
    float c[3] = {a.pos[3 * p], a.pos[3 * p + 1], a.pos[3 * p + 2]};
    if (a.rsd.vel) c[a.rsd.axis] = rsd_shift(c[a.rsd.axis], a.rsd.vel[3 * p + a.rsd.axis], a.rsd.fac, a.rsd.box);
    x = c[0];
    y = c[1];
    z = c[2];
}

// supertile of a particle.  The grouping only has to be deterministic (the count and the scatter
// must agree) and spatially coherent, not equal to k_bin's tiles, so float32 cells clamped into
// the grid do (NaN goes to cell 0).
__device__ __forceinline__ int sup_cell(float x, float inv, int N) {
    return (int)fminf(fmaxf(x * inv, 0.0f), (float)(N - 1));
}
__device__ __forceinline__ int sup_of(const SupArgs& a, float x, float y) {
    const float inv = (float)a.inv;
    const unsigned v = (unsigned)((sup_cell(x, inv, a.N) / TILE) * a.nt + sup_cell(y, inv, a.N) / TILE);
    return (int)(a.cmul ? __umulhi(v, a.cmul) : v);
}
// the steps of PT * PKP particles that workgroup B.x of a.nb owns
__device__ __forceinline__ void sup_range(const SupArgs& a, unsigned bx, long long& s0, long long& s1) {
    const long long nstep = (a.n + PT * PKP - 1) / (PT * PKP), per = (nstep + a.nb - 1) / a.nb;
    s0 = min(nstep, (long long)bx * per);
    s1 = min(nstep, s0 + per);
}

// a.sel: the particles are grouped only when they are in no spatial order.  Every workgroup looks at
// the same PROBES pairs of consecutive particles and takes them for unordered
// when more than half of the pairs lie in different tiles along two axes or three: in any order by cell a step goes
// along one axis, also where the particles are so sparse that it leaves the tile (1 M onto 256^3 in cell order: with
// one axis counted they were grouped, 98 us for 71).  The pairs are one from each of PROBES equal parts of the particles,
// at a scattered place: equal distances fell on the ends of the rows of a lattice of 2^k a side.  (1024 pairs took
// 2 us: every lane reads lines of its own.)  Returns whether to group; workgroup 0 notes it.
constexpr int PROBES = 256;
__device__ __forceinline__ bool sup_probe(const SupArgs& a, Blk B) {
    if (!a.sel) return true;
    const float inv = (float)a.inv;
    int diff = 0;
    if (threadIdx.x < PROBES) {
        const unsigned long long lo = (a.n - 1) * (long long)threadIdx.x / PROBES,
                                 hi = (a.n - 1) * (long long)(threadIdx.x + 1) / PROBES;
        const unsigned long long p = lo + ((threadIdx.x * 2654435761u) * (hi - lo) >> 32);   // lo <= p < hi <= n - 1
        const float* r = a.pos + 3 * p;
#pragma unroll
        for (int c = 0; c < 3; ++c) diff += sup_cell(r[c], inv, a.N) / TILE != sup_cell(r[3 + c], inv, a.N) / TILE ? 1 : 0;
    }
    const bool group = 2 * __syncthreads_count(diff >= 2) > PROBES;
    if (B.x == 0 && threadIdx.x == 0) *a.sel = group ? 1u : 0u;
    return group;
}
static_assert(PROBE_MIN > PROBES, "a pair in every part");

__device__ __forceinline__ void sup_count_body(const SupArgs& a, Blk B) {
    __shared__ unsigned h[SUPMAX];
    const int tid = threadIdx.x;
    for (long long i = (long long)B.x * PT + tid; i < a.nclr; i += (long long)B.gx * PT) a.clr[i] = 0u;
    if (!sup_probe(a, B) || (int)B.x >= a.nb) return;
    for (int i = tid; i < a.nsup; i += PT) h[i] = 0u;
    __syncthreads();
    long long s0, s1;
    sup_range(a, B.x, s0, s1);
    for (long long step = s0; step < s1; ++step) {
        int sp[PKP];
#pragma unroll
        for (int k = 0; k < PKP; ++k) {
            const long long p = (step * PKP + k) * PT + tid;
            sp[k] = -1;
            if (p < a.n) {
                float x, y, z;
                sup_load(a, p, x, y, z);
                sp[k] = sup_of(a, x, y);
            }
        }
#pragma unroll
        for (int k = 0; k < PKP; ++k)
            if (sp[k] >= 0) atomicAdd(&h[sp[k]], 1u);
    }
    __syncthreads();
    for (int i = tid; i < a.nsp; i += PT) a.cnt[(long long)B.x * a.nsp + i] = i < a.nsup ? h[i] : 0u;
}

__global__ __launch_bounds__(PT) void k_sup_count(SupArgs a) { sup_count_body(a, own_blk()); }
__global__ __launch_bounds__(PT) void k_sup_count_b(const SupArgs* __restrict__ tab,
                                                     const unsigned* __restrict__ start, int nj) {
    PYL_BATCH_BLK(start, nj);
    sup_count_body(tab[bj_], blk_);
}

// batched launches (a.tot): columns [64 bx, 64 bx + 64) of cnt: exclusive sums down the rows in place, and the column
// totals; the rows are split over the 16 waves
__device__ __forceinline__ void sup_scan_body(const SupArgs& a, unsigned bx) {
    __shared__ unsigned wsum[16][64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int c = (int)bx * 64 + lane;
    const int per = (a.nb + 15) / 16, r0 = min(a.nb, wv * per), r1 = min(a.nb, r0 + per);
    constexpr int PER = SUPBLOCKS / 16;   // all rows of a wave are loaded before the first is used
    unsigned s = 0u, v[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) v[j] = c < a.nsup && r0 + j < r1 ? a.cnt[(long long)(r0 + j) * a.nsp + c] : 0u;
#pragma unroll
    for (int j = 0; j < PER; ++j) s += v[j];
    wsum[wv][lane] = s;
    __syncthreads();
    if (c >= a.nsup) return;
    unsigned run = 0u;
    for (int j = 0; j < wv; ++j) run += wsum[j][lane];
    if (wv == 15) a.tot[c] = run + s;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        if (r0 + j < r1) a.cnt[(long long)(r0 + j) * a.nsp + c] = run;
        run += v[j];
    }
}
// job blockIdx.y
__global__ __launch_bounds__(1024) void k_sup_scan_b(const SupArgs* __restrict__ tab) {
    const SupArgs& a = tab[blockIdx.y];
    sup_scan_body(a, blockIdx.x);
}

// First slots of the groups for workgroup bx: where a group begins, plus what the workgroups before bx put there; thread
// g's return value is group g's.  A single call sums the whole table of counts in every workgroup (up to 1 MB, from L2): as
// long as a launch of its own took, and ordered particles, which need none of this, save that launch.  In a batch one
// launch sums for all jobs (64 jobs: 18.90 ms a replay, 19.04 with the sums in every workgroup).  sc: LDS for
// 2 x 4 PT words.
__device__ __forceinline__ unsigned sup_first(const SupArgs& a, unsigned bx, unsigned* sc, unsigned* wsum) {
    const int tid = threadIdx.x;
    if (a.tot) {
        const unsigned first = block_exscan(tid < a.nsup ? a.tot[tid] : 0u, wsum);
        return tid < a.nsup ? first + a.cnt[(long long)bx * a.nsp + tid] : first;
    }
    const int q4 = a.nsp / 4, parts = min(PT / q4, 32);
    const int part = tid / q4, c4 = tid % q4;
    if (part < parts) {
        uint4 t = make_uint4(0u, 0u, 0u, 0u), b = t;
#pragma unroll 8
        for (int r = part; r < a.nb; r += parts) {
            const uint4 v = ((const uint4*)(a.cnt + (long long)r * a.nsp))[c4];
            const unsigned m = r < (int)bx ? ~0u : 0u;
            t.x += v.x, t.y += v.y, t.z += v.z, t.w += v.w;
            b.x += v.x & m, b.y += v.y & m, b.z += v.z & m, b.w += v.w & m;
        }
        ((uint4*)sc)[part * q4 + c4] = t;
        ((uint4*)sc)[(parts + part) * q4 + c4] = b;
    }
    __syncthreads();
    unsigned tot = 0u, before = 0u;
    if (tid < a.nsup)
        for (int p = 0; p < parts; ++p) {
            tot += sc[p * a.nsp + tid];
            before += sc[(parts + p) * a.nsp + tid];
        }
    return block_exscan(tot, wsum) + before;
}

// A step's particles are put in group order in LDS and leave in runs of consecutive addresses (one store of
// 12 bytes a lane to as many lines kept the store path busy: 10 M weighted particles 161 -> 70 us).
template <bool HASW>
__device__ __forceinline__ void sup_scatter_body(const SupArgs& a, Blk B) {
    constexpr int PS = PT * PKP, R = HASW ? 4 : 3;
    __shared__ float rec[PS * R];
    __shared__ unsigned short grp[PS];
    __shared__ unsigned lc[SUPMAX];   // the step's particles per group
    __shared__ unsigned lo[SUPMAX];   // first of them in rec
    __shared__ unsigned gd[SUPMAX];   // where rec[i] of the group goes: gd + i
    __shared__ unsigned wsum[PT / 64];
    static_assert(SUPMAX == PT && PS <= 65536, "one group a thread");
    const int tid = threadIdx.x;
    if ((a.sel && !*a.sel) || (int)B.x >= a.nb) return;
    static_assert(PS * R >= 2 * 4 * PT, "the sums of the counts fit where the records come");
    unsigned cur = sup_first(a, B.x, (unsigned*)rec, wsum);   // thread g's cursor: the workgroup's next slot in group g
    lc[tid] = 0u;
    long long s0, s1;
    sup_range(a, B.x, s0, s1);
    float nx[PKP], ny[PKP], nz[PKP], nw[PKP];
    auto load = [&](long long step) {
#pragma unroll
        for (int k = 0; k < PKP; ++k) {
            const long long p = (step * PKP + k) * PT + tid;
            if (p < a.n) {
                sup_load(a, p, nx[k], ny[k], nz[k]);
                nw[k] = HASW ? a.W[p] : 0.f;
            }
        }
    };
    if (s0 < s1) load(s0);
    __syncthreads();
    for (long long step = s0; step < s1; ++step) {
        float x[PKP], y[PKP], z[PKP], w[PKP];
        int g[PKP];
        unsigned r[PKP];
#pragma unroll
        for (int k = 0; k < PKP; ++k) {
            x[k] = nx[k];
            y[k] = ny[k];
            z[k] = nz[k];
            w[k] = nw[k];
        }
        if (step + 1 < s1) load(step + 1);   // in flight during this step
#pragma unroll
        for (int k = 0; k < PKP; ++k) {
            g[k] = -1;
            if ((step * PKP + k) * PT + tid < a.n) {
                g[k] = sup_of(a, x[k], y[k]);
                r[k] = atomicAdd(&lc[g[k]], 1u);
            }
        }
        __syncthreads();   // (also: every thread has stored the previous step's records)
        const unsigned c = lc[tid];
        lc[tid] = 0u;
        const unsigned o = block_exscan(c, wsum);
        lo[tid] = o;
        gd[tid] = cur - o;
        cur += c;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < PKP; ++k) {
            if (g[k] < 0) continue;
            const unsigned i = lo[g[k]] + r[k];
            rec[i * R] = x[k];
            rec[i * R + 1] = y[k];
            rec[i * R + 2] = z[k];
            if (HASW) rec[i * R + 3] = w[k];
            grp[i] = (unsigned short)g[k];
        }
        __syncthreads();
        const int m = (int)min((long long)PS, a.n - step * PS);
        for (int i = tid; i < m; i += PT) {
            const long long d = gd[grp[i]] + (unsigned)i;
            if (d >= a.n) continue;   // unreachable: the count pass gave every particle its slot
            a.spos[3 * d] = rec[i * R];
            a.spos[3 * d + 1] = rec[i * R + 1];
            a.spos[3 * d + 2] = rec[i * R + 2];
            if (HASW) a.sw[d] = rec[i * R + 3];
        }
    }
}

template <bool HASW>
__global__ __launch_bounds__(PT) void k_sup_scatter(SupArgs a) { sup_scatter_body<HASW>(a, own_blk()); }
template <bool HASW>
__global__ __launch_bounds__(PT) void k_sup_scatter_b(const SupArgs* __restrict__ tab,
                                                       const unsigned* __restrict__ start, int nj) {
    PYL_BATCH_BLK(start, nj);
    sup_scatter_body<HASW>(tab[bj_], blk_);
}

// ------------------------------------------------------------------ host side
bool binned_supported(int axes, int dims) { return axes == 3 && dims % TILE == 0 && dims >= 2 * TILE; }
// grids whose edge is no multiple of TILE (see tile_mul for the upper limit)
bool binned_ragged(int axes, int dims) { return axes == 3 && dims % TILE != 0 && dims >= 2 * TILE && dims < 32768; }

// A grouped copy of the particles and the device word that tells whether it was made
struct Presort {
    const unsigned* sel = nullptr;
    const float* pos = nullptr;
    const float* W = nullptr;
    bool cleared = false;   // the deposit's counters are cleared on the way
};

// Bucket layout of one deposit: class segment capacities of twice the expected count of a uniform
// distribution plus slack, and the bytes of the counters, buckets and overflow area.
struct Layout {
    int nt, cap[8], cofs[8];
    long long ntiles, CT;
    size_t ncnt;   // counters: fill (8 ntiles) | ocnt | ooff | ov_count | turn (2)
    size_t cnt_bytes, bucket_bytes, ov_bytes;
};

static int layout_of(int64_t n, int dims, int S, bool hasw, Layout* L) {
    const int R = hasw ? 4 : 3;
    L->nt = (dims + TILE - 1) / TILE;
    L->ntiles = (long long)L->nt * L->nt * L->nt;
    const double avg = (double)n / (double)L->ntiles;
    const double ph = (double)(S - 1) * L->nt / dims, p0 = 1.0 - ph;
    L->CT = 0;
    for (int c = 0; c < 8; ++c) {
        const double f = ((c & 1) ? ph : p0) * ((c & 2) ? ph : p0) * ((c & 4) ? ph : p0);
        const long long v = f > 0.0 ? ((long long)(2.0 * avg * f) + 32 + 15) / 16 * 16 : 0;
        PYL_CHECK(v < (1LL << 30), E_UNSUPPORTED, "binned deposit: too many particles per tile");
        L->cap[c] = (int)v;
        L->cofs[c] = (int)L->CT;
        L->CT += v;
    }
    L->ncnt = 10 * (size_t)L->ntiles + 4;
    L->cnt_bytes = sizeof(unsigned) * L->ncnt + 64;
    L->bucket_bytes = sizeof(float) * (size_t)L->ntiles * L->CT * R;
    // overflow: ov_idx (8n: particle index, and the record's index beyond its segment in the upper half) | ov_key (4n) | gcls (4n) | grouped (4Rn)
    L->ov_bytes = (size_t)n * (16 + 4 * R) + 256;
    return OK;
}

template <int S, typename G, bool HASW, int MODE>
static int run_binned(const float* pos, const float* W, int64_t n, int dims, double BoxSize, double mult, void* grid,
                      const double* dmass, double mass, hipStream_t st, const Rsd& rsd, int acc, const Presort& ps) {
    int rc = OK;
    Layout L;
    rc = layout_of(n, dims, S, HASW, &L);
    if (rc) return rc;
    const int nt = L.nt;
    const bool rag = dims % TILE != 0;
    const long long ntiles = L.ntiles, CT = L.CT;
    const int *cap = L.cap, *cofs = L.cofs;
    const size_t ncnt = L.ncnt;
    unsigned* cnt = (unsigned*)workspace(WS_BINS, L.cnt_bytes, &rc);
    if (rc) return rc;
    unsigned *fill = cnt, *ocnt = cnt + 8 * ntiles, *ooff = cnt + 9 * ntiles, *ov_count = cnt + 10 * ntiles;
    float* bucket = (float*)workspace(WS_AUX, L.bucket_bytes, &rc);
    if (rc) return rc;
    char* ov = (char*)workspace(WS_AUX2, L.ov_bytes, &rc);
    if (rc) return rc;
    unsigned long long* ov_idx = (unsigned long long*)ov;
    unsigned* ov_key = (unsigned*)(ov + 8 * (size_t)n);
    unsigned* gcls = (unsigned*)(ov + 12 * (size_t)n);
    float* grouped = (float*)(ov + 16 * (size_t)n + 64);
    if (!ps.cleared && (rc = zero_fill(cnt, sizeof(unsigned) * ncnt, st))) return rc;
    {
        StageTimer tm("deposit_bin", st);
        BinArgs ba{pos, W, (long long)n, dims, nt, dims / BoxSize, fill, bucket, CT, {}, {}, ov_count, ov_idx, ov_key, rsd};
        ba.agg = bin_agg(n, dims);
        ba.tmul = tile_mul(dims, nt);
        ba.sel = ps.sel;
        ba.spos = ps.pos;
        ba.sw = ps.W;
        for (int c = 0; c < 8; ++c) {
            ba.cofs[c] = cofs[c];
            ba.cap[c] = cap[c];
        }
        long long blocks = (n + (long long)BT * KP - 1) / ((long long)BT * KP);
        if (blocks > 2048) blocks = 2048;
        blocks = (blocks + XCDS - 1) / XCDS * XCDS;
        if (rag)
            hipLaunchKernelGGL((k_bin<S, HASW, 2, true>), dim3((unsigned)blocks), dim3(BT), 0, st, ba);
        else if (ba.agg)
            hipLaunchKernelGGL((k_bin<S, HASW, 1, false>), dim3((unsigned)blocks), dim3(BT), 0, st, ba);
        else
            hipLaunchKernelGGL((k_bin<S, HASW, 0, false>), dim3((unsigned)blocks), dim3(BT), 0, st, ba);
        PYL_HIP(hipGetLastError());
    }
    {
        StageTimer tm("deposit_overflow", st);
        OvArgs oa{ov_count, ov_idx, ov_key, fill, {}, ocnt, ooff, ov_count + 1, pos, W, grouped, gcls, rsd,
                  (int)ntiles, ps.sel, ps.pos, ps.W};
        for (int c = 0; c < 8; ++c) oa.cap[c] = cap[c];
        hipLaunchKernelGGL((k_ov<HASW>), dim3(OB), dim3(OT), 0, st, oa);
        PYL_HIP(hipGetLastError());
    }
    {
        StageTimer tm("deposit_tiles", st);
        TileArgs ta{bucket, fill, CT, {}, {}, grouped, gcls, ooff, ocnt, dims, nt, dims / BoxSize, mult, grid, dmass,
                    mass};
        for (int c = 0; c < 8; ++c) {
            ta.cofs[c] = cofs[c];
            ta.cap[c] = cap[c];
        }
        const dim3 tg((unsigned)((ntiles + XCDS - 1) / XCDS * XCDS));
        const bool unit = !HASW && mult == 1.0;
#define PYL_TILE_LAUNCH(U, A, G_) hipLaunchKernelGGL((k_tile<S, G, HASW, MODE, U, A, G_>), tg, dim3(TT), 0, st, ta)
        if (rag) {
            // (never the overdensity; ACC_F32W allows float32 weights, and gets float64 ones)
            if constexpr (MODE != OUT_DELTA) {
                if constexpr (S == 2) {
                    if (acc == ACC_RUN) PYL_TILE_LAUNCH(!HASW, ACC_RUN, true);
                }
                if (acc != ACC_RUN) PYL_TILE_LAUNCH(!HASW, ACC_F64, true);
            }
        } else if (acc == ACC_RUN) {
            if constexpr (S == 2) {
                if (unit) PYL_TILE_LAUNCH(true, ACC_RUN, false); else PYL_TILE_LAUNCH(false, ACC_RUN, false);
            }
        } else if (acc == ACC_F32W) {
            if (unit) PYL_TILE_LAUNCH(true, ACC_F32W, false); else PYL_TILE_LAUNCH(false, ACC_F32W, false);
        } else {
            if (unit) PYL_TILE_LAUNCH(true, ACC_F64, false); else PYL_TILE_LAUNCH(false, ACC_F64, false);
        }
#undef PYL_TILE_LAUNCH
        PYL_HIP(hipGetLastError());
    }
    return OK;
}

template <int S, typename G, int MODE>
static int dispatch_w(const float* pos, const float* W, int64_t n, int dims, double BoxSize, double mult, void* grid,
                      const double* dmass, double mass, hipStream_t st, const Rsd& rsd, int acc, const Presort& ps) {
    return W ? run_binned<S, G, true, MODE>(pos, W, n, dims, BoxSize, mult, grid, dmass, mass, st, rsd, acc, ps)
             : run_binned<S, G, false, MODE>(pos, W, n, dims, BoxSize, mult, grid, dmass, mass, st, rsd, acc, ps);
}

template <typename G, int MODE>
static int dispatch_s(const float* pos, const float* W, int64_t n, int dims, double BoxSize, int scheme, double mult,
                      void* grid, const double* dmass, double mass, hipStream_t st, const Rsd& rsd, int acc,
                      const Presort& ps) {
    switch (scheme) {
        case 1: return dispatch_w<1, G, MODE>(pos, W, n, dims, BoxSize, mult, grid, dmass, mass, st, rsd, acc, ps);
        case 2: return dispatch_w<2, G, MODE>(pos, W, n, dims, BoxSize, mult, grid, dmass, mass, st, rsd, acc, ps);
        case 3: return dispatch_w<3, G, MODE>(pos, W, n, dims, BoxSize, mult, grid, dmass, mass, st, rsd, acc, ps);
        case 4: return dispatch_w<4, G, MODE>(pos, W, n, dims, BoxSize, mult, grid, dmass, mass, st, rsd, acc, ps);
        default: set_error("unknown scheme %d", scheme); return E_ARG;
    }
}

// supertiles: m whole tile columns (nt tiles along z) each, about SUPGROUPS of them and never more than
// SUPMAX; sup_fill sets the geometry of a presort (everything but the buffers), sup_words the unsigned words
// of its counters (counts, totals, the order word)
static void sup_fill(SupArgs* a, int64_t n, int dims) {
    a->nt = (dims + TILE - 1) / TILE;
    const long long cols = (long long)a->nt * a->nt;
    long long m = std::max(1LL, (cols + SUPGROUPS - 1) / SUPGROUPS);
    while ((cols + m - 1) / m > SUPMAX) ++m;
    // v * ceil(2^32 / m) >> 32 = v / m for v < cols: the rounding adds less than cols / 2^32 < 1 / m
    a->cmul = m == 1 ? 0u : (unsigned)(((1ULL << 32) + m - 1) / m);
    a->nsup = (int)((cols + m - 1) / m);
    a->nsp = (a->nsup + 3) / 4 * 4;
    a->N = dims;
    a->n = n;
    a->nb = (int)std::max<int64_t>(1, std::min<int64_t>(SUPBLOCKS, (n + PT * PKP - 1) / (PT * PKP)));
}
static size_t sup_words(const SupArgs& a) { return (size_t)(a.nb + 1) * a.nsp + 4; }
static void sup_carve(SupArgs* a, unsigned* w) {
    a->cnt = w;
}

// groups the particles by supertile into library workspaces (ps->pos, ps->W); the redshift-space shift
// is applied on the way, so the grouped copy is deposited without it.  probe: only when they are in no
// spatial order, which the device decides (ps->sel).  The count clears the deposit's counters, so that ordered
// particles cost no more launches than the clear, the three of the overflow grouping and the rest once did.
static int presort(const float* pos, const float* W, int64_t n, int dims, double BoxSize, int scheme, const Rsd& rsd,
                   bool probe, hipStream_t st, Presort* ps) {
    SupArgs a{};
    sup_fill(&a, n, dims);
    Layout L;
    int rc = layout_of(n, dims, scheme, W != nullptr, &L);
    if (rc) return rc;
    a.clr = (unsigned*)workspace(WS_BINS, L.cnt_bytes, &rc);
    if (rc) return rc;
    a.nclr = (long long)L.ncnt;
    unsigned* words = (unsigned*)workspace(WS_SUP, sizeof(unsigned) * sup_words(a), &rc);
    if (rc) return rc;
    float* sp = (float*)workspace(WS_STAGE, sizeof(float) * (size_t)n * (W ? 4 : 3) + 64, &rc);
    if (rc) return rc;
    sup_carve(&a, words);
    a.pos = pos;
    a.W = W;
    a.inv = dims / BoxSize;
    a.rsd = rsd;
    a.spos = sp;
    a.sw = W ? sp + 3 * n : nullptr;
    a.sel = probe ? a.cnt + (size_t)(a.nb + 1) * a.nsp : nullptr;
    StageTimer tm("deposit_presort", st);
    hipLaunchKernelGGL(k_sup_count, dim3((unsigned)a.nb), dim3(PT), 0, st, a);
    if (W)
        hipLaunchKernelGGL((k_sup_scatter<true>), dim3((unsigned)a.nb), dim3(PT), 0, st, a);
    else
        hipLaunchKernelGGL((k_sup_scatter<false>), dim3((unsigned)a.nb), dim3(PT), 0, st, a);
    PYL_HIP(hipGetLastError());
    ps->sel = a.sel;
    ps->pos = sp;
    ps->W = a.sw;
    ps->cleared = true;
    return OK;
}

// mode: 0 accumulate, 1 overwrite, 2 overdensity (mass = dmass[0] if dmass else mass); acc: cell
// accumulation of a float32 grid (ACC_F64 / ACC_F32W; float64 grids always use ACC_F64)
int deposit_binned(const float* pos, const float* W, int64_t n, int dims, double BoxSize, int scheme, bool f64,
                   int mode, double mult, void* grid, const double* dmass, double mass, hipStream_t st,
                   const Rsd& rsd_in, int sorted, int acc) {
    PYL_CHECK(!rsd_in.vel || (rsd_in.axis >= 0 && rsd_in.axis <= 2), E_ARG, "redshift-space axis must be 0, 1 or 2");
    PYL_CHECK(binned_supported(3, dims) || binned_ragged(3, dims), E_UNSUPPORTED,
              "binned deposit needs 3-D grids of at least %d cells an edge", 2 * TILE);
    PYL_CHECK(binned_supported(3, dims) || (mode != OUT_DELTA && mult == 1.0), E_UNSUPPORTED,
              "binned deposit: overdensities need dims %% %d == 0", TILE);
    PYL_CHECK(n > 0, E_ARG, "binned deposit needs particles");
    PYL_CHECK(n < (1LL << 31), E_UNSUPPORTED, "binned deposit: at most 2^31 particles per call");
    Rsd rsd = rsd_in;
    Presort ps;
    const long long nt = (dims + TILE - 1) / TILE, keys = nt * nt * nt * (scheme > 1 ? 8 : 1);
    if (sorted == PRESORT_PROBE && (rsd.vel || n < PROBE_MIN || keys < PROBE_KEYS)) sorted = PRESORT_NO;
    if (sorted) {
        const int rc = presort(pos, W, n, dims, BoxSize, scheme, rsd_in, sorted == PRESORT_PROBE, st, &ps);
        if (rc && !(sorted == PRESORT_PROBE && rc == E_ALLOC)) return rc;
        if (rc) ps = Presort();   // no room for the grouped copy: deposit the particles as they are
        if (!rc && sorted == PRESORT_YES) {
            pos = ps.pos;
            W = ps.W;
            rsd = Rsd();
            ps = Presort();
            ps.cleared = true;
        }
    }
    auto run = [&](const Presort& q) -> int {
        if (f64) {
            const int a64 = dense_acc(ACC_F64, scheme, n, dims);
            if (mode == OUT_ACC) return dispatch_s<double, OUT_ACC>(pos, W, n, dims, BoxSize, scheme, mult, grid, dmass, mass, st, rsd, a64, q);
            if (mode == OUT_SET) return dispatch_s<double, OUT_SET>(pos, W, n, dims, BoxSize, scheme, mult, grid, dmass, mass, st, rsd, a64, q);
            return dispatch_s<double, OUT_DELTA>(pos, W, n, dims, BoxSize, scheme, mult, grid, dmass, mass, st, rsd, a64, q);
        }
        const int a32 = dense_acc(acc, scheme, n, dims);
        if (mode == OUT_ACC) return dispatch_s<float, OUT_ACC>(pos, W, n, dims, BoxSize, scheme, mult, grid, dmass, mass, st, rsd, a32, q);
        if (mode == OUT_SET) return dispatch_s<float, OUT_SET>(pos, W, n, dims, BoxSize, scheme, mult, grid, dmass, mass, st, rsd, a32, q);
        return dispatch_s<float, OUT_DELTA>(pos, W, n, dims, BoxSize, scheme, mult, grid, dmass, mass, st, rsd, a32, q);
    };
    const int rc = run(ps);
    if (rc != E_ALLOC || !ps.sel) return rc;
    // the buckets do not fit beside the grouped copy: without it
    workspace_drop(WS_STAGE);
    workspace_drop(WS_SUP);
    return run(Presort());
}

// ------------------------------------------------------------------ batched deposit
// Jobs of a batch (pyl_graph_create / pyl_pk_batch) run each stage of the deposit as ONE launch for
// all jobs of a class (same scheme, weights, grid type, accumulation and presort): the arguments of
// job j sit in device tables and its blocks are the range [start[j], start[j+1]) of the launch.
static size_t al256(size_t b) { return (b + 255) / 256 * 256; }

size_t binned_job_bytes(int64_t n, int dims, int scheme, bool hasw, bool sorted) {
    Layout L;
    if (!binned_supported(3, dims) || layout_of(n, dims, scheme, hasw, &L) != OK) return 0;
    size_t b = al256(L.cnt_bytes) + al256(L.bucket_bytes) + al256(L.ov_bytes);
    if (sorted) {
        SupArgs a{};
        sup_fill(&a, n, dims);
        b += al256(sizeof(unsigned) * sup_words(a)) + al256(sizeof(float) * (size_t)n * (hasw ? 4 : 3) + 64);
    }
    return b;
}

int binned_job_plan(const float* pos, const float* W, int64_t n, int dims, double BoxSize, int scheme, void* grid,
                    const double* dmass, double mass, bool sorted, char* mem, BinnedJob* j) {
    PYL_CHECK(binned_supported(3, dims), E_UNSUPPORTED, "binned deposit needs 3-D grids with dims %% %d == 0", TILE);
    PYL_CHECK(n > 0 && n < (1LL << 31), E_UNSUPPORTED, "binned deposit: 1 to 2^31 - 1 particles per job");
    const bool hasw = W != nullptr;
    const int R = hasw ? 4 : 3;
    Layout L;
    int rc = layout_of(n, dims, scheme, hasw, &L);
    if (rc) return rc;
    char* p = mem;
    unsigned* cnt = (unsigned*)p;
    p += al256(L.cnt_bytes);
    float* bucket = (float*)p;
    p += al256(L.bucket_bytes);
    char* ov = p;
    p += al256(L.ov_bytes);
    const long long ntiles = L.ntiles;
    unsigned *fill = cnt, *ocnt = cnt + 8 * ntiles, *ooff = cnt + 9 * ntiles, *ov_count = cnt + 10 * ntiles;
    unsigned long long* ov_idx = (unsigned long long*)ov;
    unsigned* ov_key = (unsigned*)(ov + 8 * (size_t)n);
    unsigned* gcls = (unsigned*)(ov + 12 * (size_t)n);
    float* grouped = (float*)(ov + 16 * (size_t)n + 64);
    const double inv = dims / BoxSize;
    const float* bpos = pos;
    const float* bW = W;
    j->sup = SupArgs{};
    j->sup_blocks = 0;
    if (sorted) {
        SupArgs& a = j->sup;
        sup_fill(&a, n, dims);
        sup_carve(&a, (unsigned*)p);
        a.tot = a.cnt + (size_t)a.nb * a.nsp;
        p += al256(sizeof(unsigned) * sup_words(a));
        float* sp = (float*)p;
        a.pos = pos;
        a.W = W;
        a.inv = inv;
        a.spos = sp;
        a.sw = hasw ? sp + 3 * n : nullptr;
        // a batched launch gives every job a multiple of XCDS blocks; those past a.nb have no particles
        j->sup_blocks = (unsigned)((a.nb + XCDS - 1) / XCDS * XCDS);
        bpos = sp;
        bW = a.sw;
    }
    (void)R;
    j->bin = BinArgs{bpos, bW, (long long)n, dims, L.nt, inv, fill, bucket, L.CT, {}, {}, ov_count, ov_idx, ov_key,
                     Rsd()};
    j->bin.agg = bin_agg(n, dims);
    j->tile = TileArgs{bucket, fill, L.CT, {}, {}, grouped, gcls, ooff, ocnt, dims, L.nt, inv, 1.0, grid, dmass, mass};
    for (int c = 0; c < 8; ++c) {
        j->bin.cofs[c] = j->tile.cofs[c] = L.cofs[c];
        j->bin.cap[c] = j->tile.cap[c] = L.cap[c];
    }
    long long bb = (n + (long long)BT * KP - 1) / ((long long)BT * KP);
    if (bb > 2048) bb = 2048;
    j->bin_blocks = (unsigned)((bb + XCDS - 1) / XCDS * XCDS);
    j->ov = OvArgs{ov_count, ov_idx, ov_key, fill, {}, ocnt, ooff, ov_count + 1, bpos, bW, grouped, gcls, Rsd(),
                   (int)ntiles};
    for (int c = 0; c < 8; ++c) j->ov.cap[c] = L.cap[c];
    j->tile_blocks = (unsigned)((ntiles + XCDS - 1) / XCDS * XCDS);
    j->cnt = cnt;
    j->cnt_bytes = sizeof(unsigned) * L.ncnt;
    return OK;
}

template <int S, bool HASW, typename G, int ACC>
static int batch_launch_s(bool sorted, const BinnedTables& t, hipStream_t st) {
    const unsigned nj = (unsigned)t.nj;
    if (sorted) {
        StageTimer tm("deposit_presort", st);
        hipLaunchKernelGGL(k_sup_count_b, dim3(t.sup_total), dim3(PT), 0, st, t.sup, t.sup_start, t.nj);
        hipLaunchKernelGGL(k_sup_scan_b, dim3(SUPMAX / 64, nj), dim3(1024), 0, st, t.sup);
        hipLaunchKernelGGL((k_sup_scatter_b<HASW>), dim3(t.sup_total), dim3(PT), 0, st, t.sup, t.sup_start, t.nj);
        PYL_HIP(hipGetLastError());
    }
    {
        StageTimer tm("deposit_bin", st);
        hipLaunchKernelGGL((k_bin_b<S, HASW>), dim3(t.bin_total), dim3(BT), 0, st, t.bin, t.bin_start, t.nj);
        PYL_HIP(hipGetLastError());
    }
    {
        StageTimer tm("deposit_overflow", st);
        hipLaunchKernelGGL((k_ov_b<HASW>), dim3(OB, nj), dim3(OT), 0, st, t.ov);
        PYL_HIP(hipGetLastError());
    }
    {
        StageTimer tm("deposit_tiles", st);
        hipLaunchKernelGGL((k_tile_b<S, G, HASW, OUT_DELTA, !HASW, ACC>), dim3(t.tile_total), dim3(TT), 0, st, t.tile,
                           t.tile_start, t.nj);
        PYL_HIP(hipGetLastError());
    }
    return OK;
}

template <int S>
static int batch_launch_w(bool hasw, bool f64, int acc, bool sorted, const BinnedTables& t, hipStream_t st) {
    if constexpr (S == 2) {
        if (acc == ACC_RUN)
            return f64 ? (hasw ? batch_launch_s<S, true, double, ACC_RUN>(sorted, t, st)
                               : batch_launch_s<S, false, double, ACC_RUN>(sorted, t, st))
                       : (hasw ? batch_launch_s<S, true, float, ACC_RUN>(sorted, t, st)
                               : batch_launch_s<S, false, float, ACC_RUN>(sorted, t, st));
    }
    if (f64) return hasw ? batch_launch_s<S, true, double, ACC_F64>(sorted, t, st)
                         : batch_launch_s<S, false, double, ACC_F64>(sorted, t, st);
    if (acc == ACC_F32W) return hasw ? batch_launch_s<S, true, float, ACC_F32W>(sorted, t, st)
                                     : batch_launch_s<S, false, float, ACC_F32W>(sorted, t, st);
    return hasw ? batch_launch_s<S, true, float, ACC_F64>(sorted, t, st)
                : batch_launch_s<S, false, float, ACC_F64>(sorted, t, st);
}

int binned_batch_launch(int scheme, bool hasw, bool f64, int acc, bool sorted, const BinnedTables& t, hipStream_t st) {
    if (t.nj <= 0) return OK;
    switch (scheme) {
        case 1: return batch_launch_w<1>(hasw, f64, acc, sorted, t, st);
        case 2: return batch_launch_w<2>(hasw, f64, acc, sorted, t, st);
        case 3: return batch_launch_w<3>(hasw, f64, acc, sorted, t, st);
        case 4: return batch_launch_w<4>(hasw, f64, acc, sorted, t, st);
        default: set_error("unknown scheme %d", scheme); return E_ARG;
    }
}

}  // namespace pyl
