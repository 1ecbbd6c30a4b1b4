// batch.hip -- many independent systems (packings) stepped together.
//
// Each system is what the reference builds with one AtomVec, OriginBox,
// NeighborList, NListed pair interaction and CollectionDamped /
// CollectionVerlet (src/collection.cpp:356-381, 442-469; src/trackers.cpp:
// 19-85).  The systems' atoms are concatenated; every per-step kernel covers
// all systems at once, and every decision (skin test, rebuild) is taken on
// the device per system, so a step needs no host round trip and a run of
// steps can be captured in a HIP graph.
//
// Per step:  k_batch_force    forces + kick (+ next drift, |x - xref| per atom)
//            k_batch_sort     a fixed grid taking the listed systems in turn:
//                             cell sort in LDS, sorted copies, xref = x
//            k_batch_build    a fixed grid over slices of the listed
//                             systems: the exact list build
//            k_batch_skin     top-2 of |x - xref| per system -> the list of
//                             systems for the next rebuild
// parm_batch_initialize orders every system's slots by cell (k_batch_reorder).
#include "cells.hpp"
#include "common.hpp"
#include "kernels.hpp"
#include "pairs.hpp"

namespace parm {

// First half of a step (drift + half kick) and |x - xref|; empties the skin
// test's worklist.
template <int D, bool DAMPED>
__global__ __launch_bounds__(kBlock) void k_batch_drift(BatchArrays A, StepCoef c,
                                                        unsigned long long *wl) {
    using PT = typename PosStore<D>::T;
    if (blockIdx.x == 0 && threadIdx.x == 0) *wl = 0ull;
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= A.ntot) return;
    PT *pos = static_cast<PT *>(A.pos_out);
    Vec<D> x = PosStore<D>::load(pos[i]);
    double v[D], a[D];
#pragma unroll
    for (int k = 0; k < D; k++) {
        v[k] = A.v[k][i];
        a[k] = A.a[k][i];
    }
    const bool fixed = is_fixed(A.m[i]);
    drift_atom<D, DAMPED>(x, v, a, fixed, c);
    if (!fixed) pos[i] = PosStore<D>::make(x);
#pragma unroll
    for (int k = 0; k < D; k++) A.v[k][i] = v[k];
    const Vec<D> x0 = PosStore<D>::load(static_cast<const PT *>(A.xref)[i]);
    Vec<D> d;
#pragma unroll
    for (int k = 0; k < D; k++) d.c[k] = x.c[k] - x0.c[k];
    A.disp[i] = sqrt(sqnorm<D>(d));
}

// |x - xref| for every atom (update_list(false) outside a step); empties the
// skin test's worklist.
template <int D>
__global__ __launch_bounds__(kBlock) void k_batch_disp(BatchArrays A,
                                                       unsigned long long *wl) {
    using PT = typename PosStore<D>::T;
    if (blockIdx.x == 0 && threadIdx.x == 0) *wl = 0ull;
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= A.ntot) return;
    const Vec<D> x = PosStore<D>::load(static_cast<const PT *>(A.pos_in)[i]);
    const Vec<D> x0 = PosStore<D>::load(static_cast<const PT *>(A.xref)[i]);
    Vec<D> d;
#pragma unroll
    for (int k = 0; k < D; k++) d.c[k] = x.c[k] - x0.c[k];
    A.disp[i] = sqrt(sqnorm<D>(d));
}

// ------------------------------------------------------------ skin test
// The reference's rule (src/trackers.cpp:23-53) per system: rebuild iff the
// two largest displacements sum to >= skin, checked only once something
// moved.  A system that rebuilds puts itself on the worklist: one 64-bit add
// on `wl` returns its place (high word) and its first build slice (low word),
// so the list's slice offsets ascend with its places, whatever the order the
// systems arrive in (their rebuilds are independent).
// W wavefronts per system, each thread kSkinAhead loads at a time: the pass is
// bound by the latency of its loads, not their 8 bytes per atom.  1024 systems
// of 64 - 4096 atoms: 31 us per launch with one wavefront per
// system and one load at a time, 6.7 us.
constexpr int kSkinAhead = 4;

template <int W>
__global__ __launch_bounds__(kBlock) void k_batch_skin(int nsys, BatchArrays A, double skin,
                                                       int slice,
                                                       unsigned long long *__restrict__ wl,
                                                       int32_t *__restrict__ work,
                                                       int32_t *__restrict__ wslice,
                                                       uint32_t *__restrict__ gflag) {
    constexpr int kPer = kBlock / kWave / W;  // systems per workgroup
    constexpr int NT = W * kWave;
    __shared__ double red[kBlock / kWave][2];
    const int s = blockIdx.x * kPer + threadIdx.x / NT;
    const int t = threadIdx.x % NT, lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
    const int off = s < nsys ? A.geom[s].off : 0, n = s < nsys ? A.geom[s].n : 0;
    Top2 m;
    bool bad = false;
    for (int k = t; k < n; k += NT * kSkinAhead) {
        double d[kSkinAhead];
#pragma unroll
        for (int q = 0; q < kSkinAhead; q++)
            d[q] = k + q * NT < n ? A.disp[off + k + q * NT] : 0.0;
#pragma unroll
        for (int q = 0; q < kSkinAhead; q++) {
            m.add(d[q]);
            bad |= !isfinite(d[q]);
        }
    }
    m = wave_top2(m);
    if (__ballot(bad) != 0ull && lane == 0) atomicOr(gflag, kFlagNonFinite);
    if (W > 1) {
        if (lane == 0) {
            red[w][0] = m.a;
            red[w][1] = m.b;
        }
        __syncthreads();
        if (t == 0) {
#pragma unroll
            for (int q = 1; q < W; q++) {
                m.add(red[w + q][0]);
                m.add(red[w + q][1]);
            }
        }
    }
    if (t == 0 && s < nsys && m.a > 0 && m.b + m.a >= skin) {
        const unsigned long long at =
            atomicAdd(wl, (1ull << 32) | (unsigned long long)((n + slice - 1) / slice));
        work[at >> 32] = s;
        wslice[at >> 32] = (int32_t)(at & 0xffffffffull);
    }
}

// -------------------------------------------------------------- rebuild
// The systems to rebuild at the end of a step are those on the worklist of
// the skin test (or all, listed by k_batch_all): wl holds their count (high
// word) and their build slices (low word), work the systems, wslice the first
// slice of each.  Two launches on fixed grids, so the launch shapes do not
// depend on how many systems rebuild (the step stays graph-capturable) and no
// workgroup is started for a system that keeps its list:
//   k_batch_sort   one workgroup of kSortThreads per listed system: cell
//                  keys, a stable counting sort of the system's atoms by
//                  cell in LDS, the cell starts, sorted copies of the
//                  positions, diameters, keys and list words, xref = x;
//   k_batch_build  one workgroup per slice of a listed system's atoms,
//                  several lanes per atom: the exact list build over the
//                  stencil rows of the periodic cell grid
//                  (candidates in row order, then sorted order:
//                  deterministic).  A large system's build is spread over
//                  many workgroups.
// With `alt` (the positions one step ahead), |alt - xref| is recomputed for
// the next skin test.
constexpr int kBatchMaxCells = kBatchMaxCellsPerSystem;
constexpr int kSortThreads = 1024;
constexpr int kAllThreads = 1024;
constexpr int kBuildThreads = 256;

// Every system on the worklist, in order.
__global__ __launch_bounds__(kAllThreads) void k_batch_all(
    int nsys, int slice, const BatchGeom *__restrict__ geom,
    unsigned long long *__restrict__ wl, int32_t *__restrict__ work,
    int32_t *__restrict__ wslice) {
    __shared__ int wsum[kAllThreads / kWave];
    const int t = threadIdx.x;
    const int per = (nsys + kAllThreads - 1) / kAllThreads;
    const int s0 = t * per;
    int loc = 0;
    for (int q = 0; q < per; q++)
        if (s0 + q < nsys) loc += (geom[s0 + q].n + slice - 1) / slice;
    const int lane = t % kWave, w = t / kWave;
    int incl = loc;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const int y = __shfl_up(incl, o);
        if (lane >= o) incl += y;
    }
    if (lane == kWave - 1) wsum[w] = incl;
    __syncthreads();
    int run = incl - loc, tot = 0;
    for (int q = 0; q < kAllThreads / kWave; q++) {
        if (q < w) run += wsum[q];
        tot += wsum[q];
    }
    for (int q = 0; q < per; q++) {
        const int s = s0 + q;
        if (s < nsys) {
            work[s] = s;
            wslice[s] = run;
            run += (geom[s].n + slice - 1) / slice;
        }
    }
    if (t == 0) *wl = ((unsigned long long)nsys << 32) | (unsigned long long)tot;
}

// A system of up to kSortKeep atoms per thread, no cell of it with more than
// kRankMax atoms, is sorted from registers: one load of the positions, each
// atom's arrival on its cell's counter, then its rank among the cell's atoms
// by their indices (so the order is the stable one).  The general form
// reloads the positions per chunk and takes its ranks from ballots, the
// wavefronts in turn: 16 barriers per chunk.  1024 systems of
// 64 - 4096: 28 us per launch in the general form, 14 us.
constexpr int kSortKeep = 4;
constexpr int kRankMax = 64;

// The per-slot outputs of the sort.
template <int D>
struct SortOut {
    int32_t *keys;     // cell of each sorted slot
    uint32_t *ent;     // list word of its atom: (index << type_bits) | type
    int32_t *cstart;
    typename PosStore<D>::T *xs;
    double *dsort;
};

template <int D>
__device__ __forceinline__ void sort_system(const int s, const BatchArrays &A,
                                            const typename PosStore<D>::T *__restrict__ pos,
                                            int count_rebuild, int type_bits,
                                            const SortOut<D> &S, uint32_t *__restrict__ which,
                                            unsigned long long *__restrict__ nent, int *hist,
                                            int *slots) {
    using PT = typename PosStore<D>::T;
    constexpr int NT = kSortThreads;
    const BatchGeom G = A.geom[s];
    const int off = G.off, n = G.n, ncell = G.grid.ncell;
    const int t = threadIdx.x;
    const bool keep = n <= kSortKeep * NT;
    PT *const xref = static_cast<PT *>(A.xref_w);
    PT xk[kSortKeep];
    double dk[kSortKeep];
    int32_t tk[kSortKeep];
    int kk[kSortKeep], ak[kSortKeep];  // key, arrival on the cell's counter
#pragma unroll
    for (int q = 0; q < kSortKeep; q++) {
        const int k = t + q * NT;
        if (keep && k < n) {
            xk[q] = pos[off + k];
            dk[q] = A.diam[off + k];
            tk[q] = A.type[off + k];
        }
    }
    for (int c = t; c < ncell; c += NT) hist[c] = 0;
    __syncthreads();
    // keys and counts
    if (keep) {
#pragma unroll
        for (int q = 0; q < kSortKeep; q++) {
            const int k = t + q * NT;
            kk[q] = ak[q] = 0;
            if (k < n) {
                kk[q] = (int)cell_of<D>(PosStore<D>::load(xk[q]), G.grid);
                ak[q] = atomicAdd(&hist[kk[q]], 1);
                xref[off + k] = xk[q];
            }
        }
    } else {
        for (int k = t; k < n; k += NT) {
            const PT x = pos[off + k];
            atomicAdd(&hist[(int)cell_of<D>(PosStore<D>::load(x), G.grid)], 1);
            xref[off + k] = x;
        }
    }
    __syncthreads();
    // exclusive scan of the counts: each thread sums a run of kScanPer
    // cells, a block scan of the run sums, then each thread writes its run
    int crowd = 0;
    {
        constexpr int kScanPer = kBatchMaxCells / NT;
        __shared__ int wsum[NT / kWave];
        const int c0 = t * kScanPer;
        int loc = 0;
#pragma unroll
        for (int q = 0; q < kScanPer; q++) {
            const int h = c0 + q < ncell ? hist[c0 + q] : 0;
            crowd |= h > kRankMax;
            loc += h;
        }
        const int lane = t % kWave, w = t / kWave;
        int incl = loc;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const int y = __shfl_up(incl, o);
            if (lane >= o) incl += y;
        }
        if (lane == kWave - 1) wsum[w] = incl;
        crowd = __syncthreads_or(crowd);
        int run = incl - loc;
        for (int q = 0; q < w; q++) run += wsum[q];
#pragma unroll
        for (int q = 0; q < kScanPer; q++) {
            const int c = c0 + q;
            if (c < ncell) {
                const int h = hist[c];
                S.cstart[G.cell_off + c] = off + run;
                hist[c] = run;
                run += h;
            }
        }
        if (t == 0) {
            S.cstart[G.cell_off + ncell] = off + n;
            hist[ncell] = n;
        }
    }
    __syncthreads();
    auto place = [&](int slot, int k, int key, const PT &x, double d, int32_t type) {
        S.xs[off + slot] = x;
        S.dsort[off + slot] = d;
        S.keys[off + slot] = key;
        S.ent[off + slot] = ((uint32_t)(off + k) << type_bits) | (uint32_t)type;
    };
    if (keep && !crowd) {
#pragma unroll
        for (int q = 0; q < kSortKeep; q++)
            if (t + q * NT < n) slots[hist[kk[q]] + ak[q]] = t + q * NT;
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kSortKeep; q++) {
            const int k = t + q * NT;
            if (k < n) {
                const int a = hist[kk[q]], b = hist[kk[q] + 1];
                int r = a;
                for (int e = a; e < b; e++) r += slots[e] < k;
                place(r, k, kk[q], xk[q], dk[q], tk[q]);
            }
        }
    } else {
        // stable scatter, one chunk of NT atoms at a time: within a wavefront
        // the rank among equal keys comes from ballots over the key bits; the
        // wavefronts of the chunk then take their turn, in order, on the cell
        // counters (the wavefront's reads of hist[key] precede, in its program
        // order, the update by its last lane of that key)
        constexpr int kKeyBits = 12;
        static_assert(kBatchMaxCells <= (1 << kKeyBits), "cell keys fit the ballot match");
        const int lane = t % kWave, wv = t / kWave;
        const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
        for (int base = 0; base < n; base += NT) {
            const int k = base + t;
            const bool valid = k < n;
            PT x{};
            double d = 0.0;
            int32_t type = 0;
            if (valid) {
                x = pos[off + k];
                d = A.diam[off + k];
                type = A.type[off + k];
            }
            const int key = valid ? (int)cell_of<D>(PosStore<D>::load(x), G.grid) : 0;
            unsigned long long eq = __ballot(valid);
#pragma unroll
            for (int b = 0; b < kKeyBits; b++) {
                const bool bit = (key >> b) & 1;
                const unsigned long long bb = __ballot(bit);
                eq &= bit ? bb : ~bb;
            }
            const int r = __popcll(eq & below);
            const bool lastk = valid && (eq >> lane) == 1ull;
            const int cntk = __popcll(eq);
            int slot = 0;
            for (int w2 = 0; w2 < NT / kWave; w2++) {
                if (wv == w2) {
                    if (valid) slot = hist[key] + r;
                    if (lastk) hist[key] += cntk;
                }
                __syncthreads();
            }
            if (valid) place(slot, k, key, x, d, type);
        }
    }
    if (t == 0) {
        nent[s] = 0ull;
        if (count_rebuild) which[s] += 1u;
    }
    // the next listed system reuses the LDS
    __syncthreads();
}

// wl_next: the worklist that the step's skin test fills, emptied here (its
// last readers were the launches of the step before).
template <int D>
__global__ __launch_bounds__(kSortThreads) void k_batch_sort(
    BatchArrays A, const typename PosStore<D>::T *__restrict__ pos, int count_rebuild,
    int type_bits, SortOut<D> S, uint32_t *__restrict__ which,
    unsigned long long *__restrict__ nent, const unsigned long long *__restrict__ wl,
    unsigned long long *__restrict__ wl_next, const int32_t *__restrict__ work) {
    __shared__ int hist[kBatchMaxCells + 1];
    __shared__ int slots[kSortKeep * kSortThreads];
    const int count = (int)(*wl >> 32);
    if (wl_next && blockIdx.x == 0 && threadIdx.x == 0) *wl_next = 0ull;
    for (int q = blockIdx.x; q < count; q += gridDim.x)
        sort_system<D>(work[q], A, pos, count_rebuild, type_bits, S, which, nent, hist, slots);
}

// G lanes per atom.  The build is bound by the latency of its chain of
// dependent loads (cell bounds, then candidates), not by arithmetic: at a step
// a few systems rebuild.  A stencil row of three x-adjacent cells is one
// contiguous range (two where it wraps), so an atom takes 9 rows, not 27
// cells; the group's lanes load all rows' bounds together and test G
// candidates per round.  48 liquids of 300 - 1000 atoms: 179 us per launch with
// one thread per atom, 27 us with 8 lanes of four candidates.  (Loading the
// next round's candidates before testing this one's is no faster: 200 liquids
// 7.67 against 7.57 ms per 100 steps.)
template <int D, int G>
__global__ __launch_bounds__(kBuildThreads) void k_batch_build(
    BatchArrays A, const typename PosStore<D>::T *__restrict__ alt, double skin,
    int type_bits, int tpa, int cap, int npad, uint32_t *__restrict__ nbr,
    int32_t *__restrict__ ncount, const int32_t *__restrict__ keys,
    const uint32_t *__restrict__ ent, const int32_t *__restrict__ cstart,
    const typename PosStore<D>::T *__restrict__ xs, const double *__restrict__ dsort,
    unsigned long long *__restrict__ nent, uint32_t *__restrict__ gflag,
    const unsigned long long *__restrict__ wl, const int32_t *__restrict__ work,
    const int32_t *__restrict__ wslice) {
    constexpr int kSlice = kBuildThreads / G;  // atoms per slice
    constexpr int RPL = (9 + G - 1) / G;       // rows whose bounds a lane loads
    __shared__ unsigned long long red[kBuildThreads / kWave];
    const int count = (int)(*wl >> 32), total = (int)(*wl & 0xffffffffull);
    const int t = threadIdx.x;
    const int sub = t % G, lane = t % kWave;
    const int gbase = lane - sub;  // first lane of this atom's group
    const unsigned long long below = (1ull << sub) - 1ull;
    for (int gs = blockIdx.x; gs < total; gs += gridDim.x) {
        // the listed system holding slice gs: the last q with wslice[q] <= gs
        int lo = 0, hi = count;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (wslice[mid] <= gs)
                lo = mid;
            else
                hi = mid;
        }
        const int s = work[lo];
        const BatchGeom G_ = A.geom[s];
        const int off = G_.off, n = G_.n, nc0 = G_.grid.nc[0], nc1 = G_.grid.nc[1],
                  nc2 = G_.grid.nc[2];
        const int u = (gs - wslice[lo]) * kSlice + t / G;
        unsigned long long mycnt = 0;
        if (u < n) {
            const int i = (int)(ent[off + u] >> type_bits);
            const Vec<D> xi = PosStore<D>::load(xs[off + u]);
            const double di = dsort[off + u];
            int key = keys[off + u];
            const int c0 = key % nc0;
            key /= nc0;
            const int c1 = D >= 2 ? key % nc1 : 0;
            const int c2 = D == 3 ? key / nc1 : 0;
            const int ny = (D >= 2 && nc1 >= 3) ? 3 : 1, nz = (D == 3 && nc2 >= 3) ? 3 : 1;
            const int nrows = ny * nz;
            // the row's x cells as at most two contiguous cell ranges
            int xa0 = 0, xb0 = 0, xa1 = 0, xb1 = -1;
            if (nc0 >= 3) {
                xa0 = c0 > 0 ? c0 - 1 : 0;
                xb0 = c0 < nc0 - 1 ? c0 + 1 : c0;
                if (c0 == 0) xa1 = xb1 = nc0 - 1;
                if (c0 == nc0 - 1) xa1 = xb1 = 0;
            }
            // lane sub loads the bounds of rows sub, sub + G, ...
            int bnd[RPL][4];
#pragma unroll
            for (int q = 0; q < RPL; q++) {
                const int r = sub + q * G;
                bnd[q][0] = bnd[q][1] = bnd[q][2] = bnd[q][3] = 0;
                if (r < nrows) {
                    int q1 = c1 + (ny == 3 ? r % 3 - 1 : 0), q2 = c2 + (nz == 3 ? r / ny - 1 : 0);
                    q1 = q1 < 0 ? q1 + nc1 : (q1 >= nc1 ? q1 - nc1 : q1);
                    q2 = q2 < 0 ? q2 + nc2 : (q2 >= nc2 ? q2 - nc2 : q2);
                    const int row = G_.cell_off + (D == 3 ? q2 * nc1 + q1 : q1) * nc0;
                    bnd[q][0] = cstart[row + xa0];
                    bnd[q][1] = cstart[row + xb0 + 1];
                    if (xb1 >= 0) {
                        bnd[q][2] = cstart[row + xa1];
                        bnd[q][3] = cstart[row + xb1 + 1];
                    }
                }
            }
            int cnt = 0;
            for (int r = 0; r < nrows; r++) {
                int rb[4];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    int v = bnd[0][k];
#pragma unroll
                    for (int q = 1; q < RPL; q++) v = r / G == q ? bnd[q][k] : v;
                    rb[k] = __shfl(v, gbase + r % G);
                }
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    for (int base = rb[2 * h]; base < rb[2 * h + 1]; base += G) {
                        // (a lane past the range reads the atom's own slot,
                        // which is not tested)
                        const int v = base + sub < rb[2 * h + 1] ? base + sub : off + u;
                        const Vec<D> xj = PosStore<D>::load(xs[v]);
                        const double dj = dsort[v];
                        const uint32_t ej = ent[v];
                        bool pass = false;
                        if (v != off + u) {
                            // minimum image by rint: equal to the reference's
                            // remainder up to rounding far inside the 1e-6
                            // band, where the reference's predicate decides
                            double d2 = 0.0;
#pragma unroll
                            for (int k = 0; k < D; k++) {
                                double dk = xi.c[k] - xj.c[k];
                                dk -= G_.box.L[k] * rint(dk * G_.box.invL[k]);
                                d2 = fma(dk, dk, d2);
                            }
                            const double cut = (di + dj) / 2 + skin;
                            const double c2c = cut * cut;
                            pass = d2 < c2c * (1.0 - 1e-6) ||
                                   (d2 <= c2c * (1.0 + 1e-6) &&
                                    in_list<D>(xi, xj, di, dj, G_.box, skin));
                        }
                        const unsigned long long m =
                            (__ballot(pass) >> gbase) & ((1ull << G) - 1ull);
                        if (pass) {
                            const int w = cnt + __popcll(m & below);
                            if (w < cap) nbr[untiled_entry(w, i, tpa, npad)] = ej;
                        }
                        cnt += __popcll(m);
                    }
                }
            }
            if (sub == 0) {
                ncount[i] = cnt < cap ? cnt : cap;
                if (cnt > cap) atomicOr(gflag, kFlagOverflow);
                mycnt = (unsigned long long)cnt;
                if (alt) {
                    const Vec<D> xa = PosStore<D>::load(alt[i]);
                    Vec<D> dd;
#pragma unroll
                    for (int d = 0; d < D; d++) dd.c[d] = xa.c[d] - xi.c[d];
                    A.disp[i] = sqrt(sqnorm<D>(dd));
                }
            }
        }
        unsigned long long sum = mycnt;
#pragma unroll
        for (int o = kWave / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
        if (t % kWave == 0) red[t / kWave] = sum;
        __syncthreads();
        if (t == 0) {
            unsigned long long tot = 0;
            for (int q = 0; q < kBuildThreads / kWave; q++) tot += red[q];
            atomicAdd(&nent[s], tot);
        }
        __syncthreads();
    }
}

// Every per-atom column in sorted order (slot k takes the slot in ent[k]):
// FORWARD gathers into the scratch arrays, the other way copies back, so the
// columns stay where they are (a captured run of steps holds their addresses).
// The caller's order is none in space: with it, an atom's neighbours are
// anywhere among its system's positions, each a cache line of its own for one
// gather.  1024 packed systems of 64 - 4096 given in random order: the force
// launch 208 -> 182 us.
template <int D>
struct OrderScratch {
    typename PosStore<D>::T *pos;
    double *v, *a, *m, *diam;  // v, a: D x ntot
    int32_t *type, *orig;
};

template <int D, bool FORWARD>
__global__ __launch_bounds__(kBlock) void k_batch_reorder(
    BatchArrays A, typename PosStore<D>::T *__restrict__ pos, double *__restrict__ m,
    double *__restrict__ diam, int32_t *__restrict__ type, int32_t *__restrict__ orig,
    const uint32_t *__restrict__ ent, int type_bits, OrderScratch<D> S) {
    const int k = blockIdx.x * kBlock + threadIdx.x;
    const size_t n = (size_t)A.ntot;
    if (k >= A.ntot) return;
    if (FORWARD) {
        const int i = (int)(ent[k] >> type_bits);
        S.pos[k] = pos[i];
#pragma unroll
        for (int d = 0; d < D; d++) {
            S.v[d * n + k] = A.v[d][i];
            S.a[d * n + k] = A.a[d][i];
        }
        S.m[k] = m[i];
        S.diam[k] = diam[i];
        S.type[k] = type[i];
        S.orig[k] = orig[i];
    } else {
        pos[k] = S.pos[k];
#pragma unroll
        for (int d = 0; d < D; d++) {
            A.v[d][k] = S.v[d * n + k];
            A.a[d][k] = S.a[d * n + k];
        }
        m[k] = S.m[k];
        diam[k] = S.diam[k];
        type[k] = S.type[k];
        orig[k] = S.orig[k];
    }
}

// Per-system sums of the per-atom energies, virials and contact / overlap
// counts (NListed::energy, pressure, contacts, overlaps per system): one
// wavefront per system, compensated sums for the energy and the virial.
__global__ __launch_bounds__(kBlock) void k_batch_sys_sums(int nsys, BatchArrays A,
                                                           const double *__restrict__ eatom,
                                                           double *__restrict__ out) {
    const int s = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
    const int lane = threadIdx.x % kWave;
    if (s >= nsys) return;
    const int off = A.geom[s].off, n = A.geom[s].n;
    const double4 *ea = reinterpret_cast<const double4 *>(eatom);
    KSum e, w;
    double c = 0.0, o = 0.0;
    for (int k = lane; k < n; k += kWave) {
        const double4 q = ea[off + k];
        e.add(q.x);
        c += q.y;
        w.add(q.z);
        o += q.w;
    }
    CSum ce{e.s, e.c}, cw{w.s, w.c};
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) {
        ce = csum_merge(ce, CSum{__shfl_xor(ce.s, d), __shfl_xor(ce.c, d)});
        cw = csum_merge(cw, CSum{__shfl_xor(cw.s, d), __shfl_xor(cw.c, d)});
        c += __shfl_xor(c, d);
        o += __shfl_xor(o, d);
    }
    if (lane == 0) {
        out[s] = ce.s + ce.c;
        out[nsys + s] = cw.s + cw.c;
        out[2 * (size_t)nsys + s] = c / 2;
        out[3 * (size_t)nsys + s] = o / 2;
    }
}

// ======================================================== host launchers
static inline int nblk1(long n) { return (int)((n + kBlock - 1) / kBlock); }

hipError_t launch_batch_force(int ndim, int precision, int stage, bool energy,
                              const BatchArrays &A, const ListView &Lv, const PairView &P,
                              const StepCoef &c, double *eatom, hipStream_t s) {
    if (A.ntot <= 0) return hipSuccess;
    const bool rep = P.kind == kPairRepulsion, dbl = precision == kFP64;
#define PARM_F(D, K, Q) batch_force_part<D, K, Q>(stage, energy, A, Lv, P, c, eatom, s)
    if (ndim == 3) {
        if (rep) {
            if (dbl) PARM_F(3, kPairRepulsion, kFP64); else PARM_F(3, kPairRepulsion, kMixed);
        } else {
            if (dbl) PARM_F(3, kPairLJ, kFP64); else PARM_F(3, kPairLJ, kMixed);
        }
    } else {
        if (rep) {
            if (dbl) PARM_F(2, kPairRepulsion, kFP64); else PARM_F(2, kPairRepulsion, kMixed);
        } else {
            if (dbl) PARM_F(2, kPairLJ, kFP64); else PARM_F(2, kPairLJ, kMixed);
        }
    }
#undef PARM_F
    return hipGetLastError();
}

hipError_t launch_batch_drift(int ndim, bool damped, const BatchArrays &A,
                              const StepCoef &c, unsigned long long *wl, hipStream_t s) {
    if (A.ntot <= 0) return hipSuccess;
    dim3 g(nblk1(A.ntot)), b(kBlock);
    if (ndim == 3) {
        if (damped)
            hipLaunchKernelGGL((k_batch_drift<3, true>), g, b, 0, s, A, c, wl);
        else
            hipLaunchKernelGGL((k_batch_drift<3, false>), g, b, 0, s, A, c, wl);
    } else {
        if (damped)
            hipLaunchKernelGGL((k_batch_drift<2, true>), g, b, 0, s, A, c, wl);
        else
            hipLaunchKernelGGL((k_batch_drift<2, false>), g, b, 0, s, A, c, wl);
    }
    return hipGetLastError();
}

hipError_t launch_batch_disp(int ndim, const BatchArrays &A, unsigned long long *wl,
                             hipStream_t s) {
    if (A.ntot <= 0) return hipSuccess;
    dim3 g(nblk1(A.ntot)), b(kBlock);
    if (ndim == 3)
        hipLaunchKernelGGL(k_batch_disp<3>, g, b, 0, s, A, wl);
    else
        hipLaunchKernelGGL(k_batch_disp<2>, g, b, 0, s, A, wl);
    return hipGetLastError();
}

// Build lanes per atom: those whose round is a stencil row or more leave the
// shortest chain, as long as the wavefronts that they make fit the chip.
// A dense batch (a liquid: ~50 atoms to a row) takes 32: 48 / 200 / 800
// liquids of 300 - 1000, passes of 100 steps with 8 x 4 (lanes x candidates
// per lane and round), 16 x 2 and 32 x 1: 5.23 / 4.22 / 3.82, 9.03 / 7.87 /
// 7.45, 20.6 / 19.6 / 19.8 ms.  A sparse one (packed spheres: ~8 to a row) of
// 16 / 64 / 256 / 1024 systems of 64 - 4096, passes of 200 steps: 16 lanes
// 5.8 / 9.6 / 19.6 / - , 8 lanes 6.2 / 9.8 / 18.6 / 61.4, 4 lanes 7.0 / 11.2 /
// 19.7 / 59.4 ms.  The lines in between: 20 atoms to a row, 2^18 and 2^20 atoms.
int batch_build_lanes(int ntot, int cells) {
    if (3.0 * ntot > 20.0 * cells) return 32;
    return ntot <= (1 << 18) ? 16 : (ntot <= (1 << 20) ? 8 : 4);
}

// One wavefront per system of up to kSkinWaveAtoms atoms on average (two
// rounds of its loads), else a workgroup.
constexpr long kSkinWaveAtoms = 2 * kSkinAhead * kWave;

hipError_t launch_batch_skin(int nsys, const BatchArrays &A, double skin, int lanes,
                             unsigned long long *wl, int32_t *work, int32_t *wslice,
                             uint32_t *gflag, hipStream_t s) {
    constexpr int kWaves = kBlock / kWave;
    if (A.ntot <= kSkinWaveAtoms * nsys)
        hipLaunchKernelGGL(k_batch_skin<1>, dim3((nsys + kWaves - 1) / kWaves), dim3(kBlock), 0,
                           s, nsys, A, skin, kBuildThreads / lanes, wl, work, wslice, gflag);
    else
        hipLaunchKernelGGL(k_batch_skin<kWaves>, dim3(nsys), dim3(kBlock), 0, s, nsys, A, skin,
                           kBuildThreads / lanes, wl, work, wslice, gflag);
    return hipGetLastError();
}

hipError_t launch_batch_all(int nsys, const BatchArrays &A, int lanes, unsigned long long *wl,
                            int32_t *work, int32_t *wslice, hipStream_t s) {
    hipLaunchKernelGGL(k_batch_all, dim3(1), dim3(kAllThreads), 0, s, nsys, kBuildThreads / lanes,
                       A.geom, wl, work, wslice);
    return hipGetLastError();
}

template <int D>
static hipError_t batch_rebuild(const BatchArrays &A, const BatchLists &B, const void *pos,
                                const void *alt, int count_rebuild, double skin,
                                const unsigned long long *wl, unsigned long long *wl_next,
                                uint32_t *gflag, hipStream_t s) {
    using PT = typename PosStore<D>::T;
    const SortOut<D> S{B.keys, B.ent, B.cstart, (PT *)B.xs, B.dsort};
    hipLaunchKernelGGL(k_batch_sort<D>, dim3(B.sort_grid), dim3(kSortThreads), 0, s, A,
                       (const PT *)pos, count_rebuild, B.type_bits, S, B.which, B.nent, wl,
                       wl_next, B.work);
    if (B.sort_only) return hipGetLastError();
    if (!B.nbr) return hipErrorInvalidValue;
#define PARM_BB(GG)                                                                           \
    case GG:                                                                                  \
        hipLaunchKernelGGL((k_batch_build<D, GG>), dim3(B.build_grid), dim3(kBuildThreads),   \
                           0, s, A, (const PT *)alt, skin, B.type_bits, B.tpa, B.cap, B.npad, \
                           B.nbr, B.ncount, B.keys, B.ent, B.cstart, (const PT *)B.xs,        \
                           B.dsort, B.nent, gflag, wl, B.work, B.wslice);                     \
        break
    switch (B.lanes) {
        PARM_BB(4);
        PARM_BB(8);
        PARM_BB(16);
        PARM_BB(32);
        default:
            return hipErrorInvalidValue;
    }
#undef PARM_BB
    return hipGetLastError();
}

hipError_t launch_batch_rebuild(int ndim, const BatchArrays &A, const BatchLists &B,
                                const void *pos, const void *alt, int count_rebuild,
                                double skin, const unsigned long long *wl,
                                unsigned long long *wl_next, uint32_t *gflag, hipStream_t s) {
    return ndim == 3 ? batch_rebuild<3>(A, B, pos, alt, count_rebuild, skin, wl, wl_next, gflag,
                                        s)
                     : batch_rebuild<2>(A, B, pos, alt, count_rebuild, skin, wl, wl_next, gflag,
                                        s);
}

template <int D>
static hipError_t batch_reorder(const BatchArrays &A, const BatchLists &B, void *pos,
                                void *pos_alt, double *m, double *diam, int32_t *type,
                                int32_t *orig, double *stage, double *eatom, hipStream_t s) {
    using PT = typename PosStore<D>::T;
    const size_t n = (size_t)A.ntot;
    // (the sorted positions in xs are free from here on; an atom's share of
    // xs, at least two doubles, holds its diameter, type and index)
    OrderScratch<D> S{};
    S.pos = (PT *)pos_alt;
    S.v = stage;
    S.a = eatom;
    S.m = eatom + 3 * n;
    S.diam = (double *)B.xs;
    S.type = (int32_t *)(S.diam + n);
    S.orig = S.type + n;
    const dim3 g(nblk1(A.ntot)), b(kBlock);
    hipLaunchKernelGGL((k_batch_reorder<D, true>), g, b, 0, s, A, (PT *)pos, m, diam, type, orig,
                       B.ent, B.type_bits, S);
    hipLaunchKernelGGL((k_batch_reorder<D, false>), g, b, 0, s, A, (PT *)pos, m, diam, type,
                       orig, B.ent, B.type_bits, S);
    return hipGetLastError();
}

hipError_t launch_batch_reorder(int ndim, const BatchArrays &A, const BatchLists &B, void *pos,
                                void *pos_alt, double *m, double *diam, int32_t *type,
                                int32_t *orig, double *stage, double *eatom, hipStream_t s) {
    return ndim == 3 ? batch_reorder<3>(A, B, pos, pos_alt, m, diam, type, orig, stage, eatom, s)
                     : batch_reorder<2>(A, B, pos, pos_alt, m, diam, type, orig, stage, eatom, s);
}

hipError_t launch_batch_sys_sums(int nsys, const BatchArrays &A, const double *eatom,
                                 double *out, hipStream_t s) {
    const int per = kBlock / kWave;
    hipLaunchKernelGGL(k_batch_sys_sums, dim3((nsys + per - 1) / per), dim3(kBlock), 0, s,
                       nsys, A, eatom, out);
    return hipGetLastError();
}

}  // namespace parm
