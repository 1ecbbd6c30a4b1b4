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
//            k_batch_worklist the systems whose skin flag is set, as a list
//            k_batch_sort     a fixed grid taking the listed systems in turn:
//                             cell sort in LDS, sorted copies, xref = x
//            k_batch_build    a fixed grid over slices of the listed
//                             systems: the exact list build, a thread per atom
//            k_batch_skin     one wavefront per system: top-2 of |x - xref|
//                             -> the system's flag for the next rebuild
#include "common.hpp"
#include "kernels.hpp"
#include "pairs.hpp"

namespace parm {

// First half of a step (drift + half kick) and |x - xref|.
template <int D, bool DAMPED>
__global__ __launch_bounds__(kBlock) void k_batch_drift(BatchArrays A, StepCoef c) {
    using PT = typename PosStore<D>::T;
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

// |x - xref| for every atom (update_list(false) outside a step).
template <int D>
__global__ __launch_bounds__(kBlock) void k_batch_disp(BatchArrays A) {
    using PT = typename PosStore<D>::T;
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
// One wavefront per system: the reference's rule (src/trackers.cpp:23-53),
// rebuild iff the two largest displacements sum to >= skin, checked only
// once something moved.  The flag is overwritten, never accumulated.
__global__ __launch_bounds__(kBlock) void k_batch_skin(int nsys, BatchArrays A,
                                                       double skin,
                                                       uint32_t *__restrict__ flags,
                                                       uint32_t *__restrict__ gflag) {
    const int s = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
    const int lane = threadIdx.x % kWave;
    if (s >= nsys) return;
    const int off = A.geom[s].off, n = A.geom[s].n;
    Top2 t;
    bool bad = false;
    for (int k = lane; k < n; k += kWave) {
        const double d = A.disp[off + k];
        t.add(d);
        bad |= !isfinite(d);
    }
    t = wave_top2(t);
    const unsigned long long anybad = __ballot(bad);
    if (lane == 0) {
        flags[s] = (t.a > 0 && t.b + t.a >= skin) ? 1u : 0u;
        if (anybad) atomicOr(gflag, kFlagNonFinite);
    }
}

// -------------------------------------------------------------- rebuild
// The systems to rebuild at the end of a step are those whose skin flag is
// set (or all, when forced).  k_batch_worklist turns the flags into a list
// (system ids in ascending order, count first) and counts each listed
// system's build slices (exclusive prefix in wslice).  Then
// two launches on fixed grids, so the launch shapes do not depend on how
// many systems rebuild (the step stays graph-capturable) and no workgroup is
// started for a system that keeps its list:
//   k_batch_sort   one workgroup of kSortThreads per listed system: cell
//                  keys, a stable counting sort of the system's atoms by
//                  cell in LDS, the cell starts, sorted copies of the
//                  positions and diameters, xref = x;
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
constexpr int kWorklistThreads = 1024;
constexpr int kBuildThreads = 256;

__global__ __launch_bounds__(kWorklistThreads) void k_batch_worklist(
    int nsys, const uint32_t *__restrict__ flags, int force, int slice,
    const BatchGeom *__restrict__ geom, int32_t *__restrict__ work,
    int32_t *__restrict__ wslice) {
    __shared__ int wsum[kWorklistThreads / kWave][2];
    const int t = threadIdx.x;
    const int per = (nsys + kWorklistThreads - 1) / kWorklistThreads;
    const int s0 = t * per;
    int loc = 0, lsl = 0;
    for (int q = 0; q < per; q++) {
        const int s = s0 + q;
        if (s < nsys && (force || flags[s] != 0u)) {
            loc++;
            lsl += (geom[s].n + slice - 1) / slice;
        }
    }
    const int lane = t % kWave, w = t / kWave;
    int incl = loc, isl = lsl;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const int y = __shfl_up(incl, o), z = __shfl_up(isl, o);
        if (lane >= o) {
            incl += y;
            isl += z;
        }
    }
    if (lane == kWave - 1) {
        wsum[w][0] = incl;
        wsum[w][1] = isl;
    }
    __syncthreads();
    int pos = incl - loc, psl = isl - lsl, tot = 0, totsl = 0;
    for (int q = 0; q < kWorklistThreads / kWave; q++) {
        if (q < w) {
            pos += wsum[q][0];
            psl += wsum[q][1];
        }
        tot += wsum[q][0];
        totsl += wsum[q][1];
    }
    for (int q = 0; q < per; q++) {
        const int s = s0 + q;
        if (s < nsys && (force || flags[s] != 0u)) {
            work[1 + pos] = s;
            wslice[pos] = psl;
            pos++;
            psl += (geom[s].n + slice - 1) / slice;
        }
    }
    if (t == 0) {
        work[0] = tot;
        wslice[tot] = totsl;
    }
}

template <int D>
__device__ __forceinline__ void sort_system(
    const int s, const BatchArrays &A, const typename PosStore<D>::T *__restrict__ pos,
    int count_rebuild, int32_t *__restrict__ keys, int32_t *__restrict__ cellidx,
    int32_t *__restrict__ cstart, typename PosStore<D>::T *__restrict__ xs,
    double *__restrict__ dsort, uint32_t *__restrict__ flags, uint32_t *__restrict__ which,
    unsigned long long *__restrict__ nent, int *hist) {
    using PT = typename PosStore<D>::T;
    constexpr int NT = kSortThreads;
    const BatchGeom G = A.geom[s];
    const int off = G.off, n = G.n, ncell = G.grid.ncell;
    const int t = threadIdx.x;
    for (int c = t; c < ncell; c += NT) hist[c] = 0;
    __syncthreads();
    // keys and counts
    for (int k = t; k < n; k += NT) {
        const Vec<D> x = PosStore<D>::load(pos[off + k]);
        int key = 0;
#pragma unroll
        for (int d = D - 1; d >= 0; d--) {
            double sv = x.c[d] * G.grid.invL[d];
            sv -= floor(sv);
            int cd = (int)(sv * (double)G.grid.nc[d]);
            cd = cd < 0 ? 0 : (cd >= G.grid.nc[d] ? G.grid.nc[d] - 1 : cd);
            key = key * G.grid.nc[d] + cd;
        }
        keys[off + k] = key;
        atomicAdd(&hist[key], 1);
    }
    __syncthreads();
    // exclusive scan of the counts: each thread sums a run of kScanPer
    // cells, a block scan of the run sums, then each thread writes its run
    {
        constexpr int kScanPer = kBatchMaxCells / NT;
        __shared__ int wsum[NT / kWave];
        const int c0 = t * kScanPer;
        int loc = 0;
        for (int q = 0; q < kScanPer; q++) loc += (c0 + q < ncell) ? hist[c0 + q] : 0;
        const int lane = t % kWave, w = t / kWave;
        int incl = loc;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const int y = __shfl_up(incl, o);
            if (lane >= o) incl += y;
        }
        if (lane == kWave - 1) wsum[w] = incl;
        __syncthreads();
        int run = incl - loc;
        for (int q = 0; q < w; q++) run += wsum[q];
        __syncthreads();
        for (int q = 0; q < kScanPer; q++) {
            const int c = c0 + q;
            if (c < ncell) {
                const int h = hist[c];
                cstart[G.cell_off + c] = off + run;
                hist[c] = run;
                run += h;
            }
        }
        if (t == 0) cstart[G.cell_off + ncell] = off + n;
    }
    __syncthreads();
    // stable scatter, one chunk of NT atoms at a time: within a wavefront the
    // rank among equal keys comes from ballots over the key bits; the
    // wavefronts of the chunk then take their turn, in order, on the cell
    // counters (the wavefront's reads of hist[key] precede, in its program
    // order, the update by its last lane of that key)
    {
        constexpr int kKeyBits = 12;
        static_assert(kBatchMaxCells <= (1 << kKeyBits), "cell keys fit the ballot match");
        const int lane = t % kWave, wv = t / kWave;
        const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
        for (int base = 0; base < n; base += NT) {
            const int k = base + t;
            const bool valid = k < n;
            const int key = valid ? keys[off + k] : 0;
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
            for (int w2 = 0; w2 < NT / kWave; w2++) {
                if (wv == w2) {
                    if (valid) cellidx[off + hist[key] + r] = off + k;
                    if (lastk) hist[key] += cntk;
                }
                __syncthreads();
            }
        }
    }
    // sorted copies of the positions and diameters, and xref = x (the
    // reference stores lastlocs inside the rebuild loop)
    for (int u = t; u < n; u += NT) {
        const int i = cellidx[off + u];
        xs[off + u] = pos[i];
        dsort[off + u] = A.diam[i];
    }
    for (int k = t; k < n; k += NT) static_cast<PT *>(A.xref_w)[off + k] = pos[off + k];
    if (t == 0) {
        nent[s] = 0ull;
        if (count_rebuild) which[s] += 1u;
        flags[s] = 0u;
    }
    // the next listed system reuses the LDS
    __syncthreads();
}

template <int D>
__global__ __launch_bounds__(kSortThreads) void k_batch_sort(
    BatchArrays A, const typename PosStore<D>::T *__restrict__ pos, int count_rebuild,
    int32_t *__restrict__ keys, int32_t *__restrict__ cellidx, int32_t *__restrict__ cstart,
    typename PosStore<D>::T *__restrict__ xs, double *__restrict__ dsort,
    uint32_t *__restrict__ flags, uint32_t *__restrict__ which,
    unsigned long long *__restrict__ nent, const int32_t *__restrict__ work) {
    __shared__ int hist[kBatchMaxCells];
    const int count = work[0];
    for (int q = blockIdx.x; q < count; q += gridDim.x)
        sort_system<D>(work[1 + q], A, pos, count_rebuild, keys, cellidx, cstart, xs, dsort,
                       flags, which, nent, hist);
}

// G lanes per atom, U candidates per lane and round.  The build is bound by
// the latency of its chain of dependent loads (cell bounds, then candidates),
// not by arithmetic: at a step a few dozen systems rebuild.  A stencil row of
// three x-adjacent cells is one contiguous range (two where it wraps), so an
// atom takes 9 rows, not 27 cells; the group's lanes load all rows' bounds
// together and test G * U candidates per round.  48 liquids of 300 - 1000 atoms:
// 179 us per launch with one thread per atom, a step 210 -> 69 us; 1024
// packings of 64 - 4096 (4 x 2 lanes): 200 steps 85.1 -> 80.0 ms.
template <int D, int G, int U>
__global__ __launch_bounds__(kBuildThreads) void k_batch_build(
    BatchArrays A, const typename PosStore<D>::T *__restrict__ alt, double skin,
    int type_bits, int tpa, int cap, int npad, uint32_t *__restrict__ nbr,
    int32_t *__restrict__ ncount, const int32_t *__restrict__ keys,
    const int32_t *__restrict__ cellidx, const int32_t *__restrict__ cstart,
    const typename PosStore<D>::T *__restrict__ xs, const double *__restrict__ dsort,
    unsigned long long *__restrict__ nent, uint32_t *__restrict__ gflag,
    const int32_t *__restrict__ work, const int32_t *__restrict__ wslice) {
    constexpr int kSlice = kBuildThreads / G;  // atoms per slice
    constexpr int RPL = (9 + G - 1) / G;       // rows whose bounds a lane loads
    __shared__ unsigned long long red[kBuildThreads / kWave];
    const int count = work[0];
    const int total = wslice[count];
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
        const int s = work[1 + lo];
        const BatchGeom G_ = A.geom[s];
        const int off = G_.off, n = G_.n, nc0 = G_.grid.nc[0], nc1 = G_.grid.nc[1],
                  nc2 = G_.grid.nc[2];
        const int u = (gs - wslice[lo]) * kSlice + t / G;
        unsigned long long mycnt = 0;
        if (u < n) {
            const int i = cellidx[off + u];
            const Vec<D> xi = PosStore<D>::load(xs[off + u]);
            const double di = dsort[off + u];
            int key = keys[i];
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
                const int owner = gbase + (r % G);
                int rb[4];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    int v = bnd[0][k];
#pragma unroll
                    for (int q = 1; q < RPL; q++) v = r / G == q ? bnd[q][k] : v;
                    rb[k] = __shfl(v, owner);
                }
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int a = rb[2 * h], b = rb[2 * h + 1];
                    for (int base = a; base < b; base += G * U) {
                        // the round's loads in flight together; a slot past
                        // the range reads the atom's own (and is not tested)
                        Vec<D> xj[U];
                        double dj[U];
#pragma unroll
                        for (int q = 0; q < U; q++) {
                            const int v = base + q * G + sub;
                            const int vv = v < b ? v : off + u;
                            xj[q] = PosStore<D>::load(xs[vv]);
                            dj[q] = dsort[vv];
                        }
#pragma unroll
                        for (int q = 0; q < U; q++) {
                            if (base + q * G >= b) break;  // uniform over the group
                            const int v = base + q * G + sub;
                            bool pass = false;
                            if (v < b && v != off + u) {
                                // minimum image by rint: equal to the
                                // reference's remainder up to rounding far
                                // inside the 1e-6 band, where the reference's
                                // predicate decides
                                double d2 = 0.0;
#pragma unroll
                                for (int k = 0; k < D; k++) {
                                    double dk = xi.c[k] - xj[q].c[k];
                                    dk -= G_.box.L[k] * rint(dk * G_.box.invL[k]);
                                    d2 = fma(dk, dk, d2);
                                }
                                const double cut = (di + dj[q]) / 2 + skin;
                                const double c2c = cut * cut;
                                pass = d2 < c2c * (1.0 - 1e-6) ||
                                       (d2 <= c2c * (1.0 + 1e-6) &&
                                        in_list<D>(xi, xj[q], di, dj[q], G_.box, skin));
                            }
                            const unsigned long long m =
                                (__ballot(pass) >> gbase) & ((1ull << G) - 1ull);
                            if (pass) {
                                const int w = cnt + __popcll(m & below);
                                if (w < cap) {
                                    const int j = cellidx[v];
                                    nbr[untiled_entry(w, i, tpa, npad)] =
                                        ((uint32_t)j << type_bits) | (uint32_t)A.type[j];
                                }
                            }
                            cnt += __popcll(m);
                        }
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
                              const StepCoef &c, hipStream_t s) {
    if (A.ntot <= 0) return hipSuccess;
    dim3 g(nblk1(A.ntot)), b(kBlock);
    if (ndim == 3) {
        if (damped)
            hipLaunchKernelGGL((k_batch_drift<3, true>), g, b, 0, s, A, c);
        else
            hipLaunchKernelGGL((k_batch_drift<3, false>), g, b, 0, s, A, c);
    } else {
        if (damped)
            hipLaunchKernelGGL((k_batch_drift<2, true>), g, b, 0, s, A, c);
        else
            hipLaunchKernelGGL((k_batch_drift<2, false>), g, b, 0, s, A, c);
    }
    return hipGetLastError();
}

hipError_t launch_batch_disp(int ndim, const BatchArrays &A, hipStream_t s) {
    if (A.ntot <= 0) return hipSuccess;
    dim3 g(nblk1(A.ntot)), b(kBlock);
    if (ndim == 3)
        hipLaunchKernelGGL(k_batch_disp<3>, g, b, 0, s, A);
    else
        hipLaunchKernelGGL(k_batch_disp<2>, g, b, 0, s, A);
    return hipGetLastError();
}

hipError_t launch_batch_skin(int nsys, const BatchArrays &A, double skin, uint32_t *flags,
                             uint32_t *gflag, hipStream_t s) {
    const int per = kBlock / kWave;
    hipLaunchKernelGGL(k_batch_skin, dim3((nsys + per - 1) / per), dim3(kBlock), 0, s, nsys,
                       A, skin, flags, gflag);
    return hipGetLastError();
}

// Build lanes per atom and candidates per lane and round: a dense system (a
// liquid: ~50 atoms in a stencil row) 8 x 4, a sparse one (packed spheres: ~8)
// 4 x 2, whose round is a row (200 steps of 1024 packings: 80.0 ms, 87.1 ms with
// 8 x 4; one thread per atom 85.1 ms).  The caller's line between them, 20
// atoms to a row of three cells, lies where a row is two to three sparse
// rounds and over half a dense one.
constexpr int kBuildLanes = 8, kBuildAhead = 4;
constexpr int kBuildLanesSparse = 4, kBuildAheadSparse = 2;

hipError_t launch_batch_rebuild(int ndim, int nsys, const BatchArrays &A, const void *pos,
                                const void *alt, int force, int count_rebuild, double skin,
                                int type_bits, int tpa, int cap, int npad, uint32_t *nbr,
                                int32_t *ncount, int32_t *keys, int32_t *cellidx,
                                int32_t *cstart, void *xs, double *dsort, uint32_t *flags,
                                uint32_t *which, unsigned long long *nent, uint32_t *gflag,
                                int32_t *work, int32_t *wslice, int sort_grid, int build_grid,
                                bool sparse, hipStream_t s) {
    if (nsys <= 0) return hipSuccess;
    // (see k_batch_build)
    const int lanes = sparse ? kBuildLanesSparse : kBuildLanes;
    hipLaunchKernelGGL(k_batch_worklist, dim3(1), dim3(kWorklistThreads), 0, s, nsys, flags,
                       force, kBuildThreads / lanes, A.geom, work, wslice);
    const int gs = sort_grid < nsys ? sort_grid : nsys;
#define PARM_BB(DD, PT, GG, UU)                                                               \
    hipLaunchKernelGGL((k_batch_build<DD, GG, UU>), dim3(build_grid), dim3(kBuildThreads), 0, \
                       s, A, (const PT *)alt, skin, type_bits, tpa, cap, npad, nbr, ncount,   \
                       keys, cellidx, cstart, (const PT *)xs, dsort, nent, gflag, work, wslice)
#define PARM_BR(DD, PT)                                                                       \
    hipLaunchKernelGGL(k_batch_sort<DD>, dim3(gs), dim3(kSortThreads), 0, s, A,               \
                       (const PT *)pos, count_rebuild, keys, cellidx, cstart, (PT *)xs,       \
                       dsort, flags, which, nent, work);                                      \
    if (sparse)                                                                               \
        PARM_BB(DD, PT, kBuildLanesSparse, kBuildAheadSparse);                                \
    else                                                                                      \
        PARM_BB(DD, PT, kBuildLanes, kBuildAhead)
    if (ndim == 3) {
        PARM_BR(3, double4);
    } else {
        PARM_BR(2, double2);
    }
#undef PARM_BR
#undef PARM_BB
    return hipGetLastError();
}

hipError_t launch_batch_sys_sums(int nsys, const BatchArrays &A, const double *eatom,
                                 double *out, hipStream_t s) {
    const int per = kBlock / kWave;
    hipLaunchKernelGGL(k_batch_sys_sums, dim3((nsys + per - 1) / per), dim3(kBlock), 0, s,
                       nsys, A, eatom, out);
    return hipGetLastError();
}

}  // namespace parm
