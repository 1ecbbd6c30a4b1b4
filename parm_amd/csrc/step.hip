// step.hip -- the per-atom step kernels (drift, skin test, observables, state
// transfers), the reductions of workgroup partials, and the dispatch of the
// force launches (force.hip, step_tiled.hip).
//
// Reference behaviour restated (paths relative to the reference root):
//   Collection::set_forces               src/collection.cpp:159-179
//   CollectionVerlet::timestep           src/collection.cpp:442-469
//   CollectionDamped::timestep           src/collection.cpp:356-381
//   NeighborList::update_list skin test  src/trackers.cpp:23-53
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"
#include "pairs.hpp"
#include "stepcore.hpp"

namespace parm {

// Sums: one workgroup per field (the last one, with TOP, takes the top-2 and
// non-finite fields), so a field's partials are read by 256 threads on a CU of
// their own: thread t adds partials t, t + 256, ... (Neumaier), then a fixed
// butterfly per wave and a fixed combine over waves (compensated two-sum), so
// the result is deterministic.  Each result goes to device memory and, for the
// host, to a pinned record whose number says that it is there: the host polls
// the records.  Latency bounds it: one workgroup of 1024 threads over all
// fields took 17 us for 16 as for 16,384 partials, and the copy of the
// results and the wait for the stream another 35.  6 frames of 100,003 atoms
// (two reductions each) 1.84 -> 1.66 ms.
constexpr int kFinSumThreads = 256;

__device__ __forceinline__ void put_sum(const ReduceBuf &R, int k, double v) {
    R.out[k] = v;
    if (R.rec) {
        __hip_atomic_store(&R.rec[k].v, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(&R.rec[k].seq, R.rseq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

template <bool TOP>
__global__ __launch_bounds__(kFinSumThreads) void k_finalize_sums(int nparts, ReduceBuf R) {
    constexpr int NW = kFinSumThreads / kWave;
    const int tid = threadIdx.x, lane = tid % kWave, w = tid / kWave;
    const int k = blockIdx.x;
    const size_t ps = (size_t)R.pstride;
    __shared__ double fin[NW][3];
    if (TOP && k == kTop1) {
        Top2 t;
        double nf = 0.0;
#pragma unroll 4
        for (int b = tid; b < nparts; b += kFinSumThreads) {
            Top2 o;
            o.a = R.part[kTop1 * ps + b];
            o.b = R.part[kTop2 * ps + b];
            t.merge(o);
            nf += R.part[kNonFinite * ps + b];
        }
        t = wave_top2(t);
        nf = wave_count(nf);
        if (lane == 0) {
            fin[w][0] = t.a;
            fin[w][1] = t.b;
            fin[w][2] = nf;
        }
        __syncthreads();
        if (tid == 0) {
            for (int q = 1; q < NW; q++) {
                Top2 o;
                o.a = fin[q][0];
                o.b = fin[q][1];
                t.merge(o);
                nf += fin[q][2];
            }
            put_sum(R, kTop1, t.a);
            put_sum(R, kTop2, t.b);
            put_sum(R, kNonFinite, nf);
        }
        return;
    }
    KSum q;
    const double *p = R.part + k * ps;
#pragma unroll 8
    for (int b = tid; b < nparts; b += kFinSumThreads) q.add(p[b]);
    CSum c{q.s, q.c};
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1)
        c = csum_merge(c, CSum{__shfl_xor(c.s, off), __shfl_xor(c.c, off)});
    if (lane == 0) {
        fin[w][0] = c.s;
        fin[w][1] = c.c;
    }
    __syncthreads();
    if (tid == 0) {
        for (int v = 1; v < NW; v++) c = csum_merge(c, CSum{fin[v][0], fin[v][1]});
        put_sum(R, k, c.s + c.c);
    }
}

// The skin test on demand: one workgroup over the partials, the flag stored in
// device memory and, with its number, in the pinned word the host polls.
constexpr int kFinal = 1024;

__global__ __launch_bounds__(kFinal) void k_finalize(int nparts, ReduceBuf R) {
    const int tid = threadIdx.x;
    const int lane = tid % kWave, w = tid / kWave;
    constexpr int NW = kFinal / kWave;
    const size_t ps = (size_t)R.pstride;
    Top2 bt;
    double nf = 0.0;
    // deep unroll: a partial array of ~10^4 workgroups is read in one or
    // two rounds of loads in flight
#pragma unroll 16
    for (int b = tid; b < nparts; b += kFinal) {
        Top2 o;
        o.a = R.part[kTop1 * ps + b];
        o.b = R.part[kTop2 * ps + b];
        bt.merge(o);
        nf += R.part[kNonFinite * ps + b];
    }
    bt = wave_top2(bt);
    nf = wave_count(nf);
    __shared__ double fin2[NW][3];
    if (lane == 0) {
        fin2[w][0] = bt.a;
        fin2[w][1] = bt.b;
        fin2[w][2] = nf;
    }
    __syncthreads();
    if (tid == 0) {
        Top2 tt;
        double nft = 0.0;
        for (int q = 0; q < NW; q++) {
            Top2 o;
            o.a = fin2[q][0];
            o.b = fin2[q][1];
            tt.merge(o);
            nft += fin2[q][2];
        }
        R.out[kTop1] = tt.a;
        R.out[kTop2] = tt.b;
        R.out[kNonFinite] = nft;
        const uint32_t fl = skin_flag(tt, nft, R.skin);
        *R.flag = fl;
        __hip_atomic_store(R.hflag, (R.g.seq << kFlagBits) | fl, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// The skin test's reduction over up to kFinBlocks workgroups of kFinThreads:
// workgroup g merges partials g, g + G, ... (top-2 and non-finite count; the
// merge does not depend on order), stores its result, and the last
// workgroup to finish (a counter: release and acquire at device scope, cheap
// here, where little is written) merges the G results and raises the flag.
// One workgroup over 16,384 partials (1M atoms) takes ~10 us; G of them, each
// reading a few hundred, a fraction of that.  The counter is returned to 0 by
// the last workgroup, so the next launch finds it cleared.
constexpr int kFinThreads = 256;

__device__ __forceinline__ void fin_block_top2(Top2 &t, double &nf) {
    constexpr int NW = kFinThreads / kWave;
    t = wave_top2(t);
    nf = wave_count(nf);
    __shared__ double sh[NW][3];
    const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
    if (lane == 0) {
        sh[w][0] = t.a;
        sh[w][1] = t.b;
        sh[w][2] = nf;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        Top2 tt;
        double n2 = 0.0;
        for (int q = 0; q < NW; q++) {
            Top2 o;
            o.a = sh[q][0];
            o.b = sh[q][1];
            tt.merge(o);
            n2 += sh[q][2];
        }
        t = tt;
        nf = n2;
    }
}

__global__ __launch_bounds__(kFinThreads) void k_finalize_skin(int nparts, ReduceBuf R) {
    const size_t ps = (size_t)R.pstride;
    const int G = (int)gridDim.x, g = (int)blockIdx.x;
    Top2 t;
    double nf = 0.0;
#pragma unroll 4
    for (int b = g * kFinThreads + (int)threadIdx.x; b < nparts; b += G * kFinThreads) {
        Top2 o;
        o.a = R.part[kTop1 * ps + b];
        o.b = R.part[kTop2 * ps + b];
        t.merge(o);
        nf += R.part[kNonFinite * ps + b];
    }
    fin_block_top2(t, nf);
    __shared__ int last;
    if (threadIdx.x == 0) {
        R.gpart[g] = t.a;
        R.gpart[kFinBlocks + g] = t.b;
        R.gpart[2 * kFinBlocks + g] = nf;
        __threadfence();
        last = atomicAdd(R.cnt, 1u) == (unsigned)(G - 1);
    }
    __syncthreads();
    if (!last) return;
    __threadfence();
    Top2 u;
    double nu = 0.0;
    if ((int)threadIdx.x < G) {
        u.a = R.gpart[threadIdx.x];
        u.b = R.gpart[kFinBlocks + threadIdx.x];
        nu = R.gpart[2 * kFinBlocks + threadIdx.x];
    }
    fin_block_top2(u, nu);
    if (threadIdx.x == 0) {
        __hip_atomic_store(R.cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        R.out[kTop1] = u.a;
        R.out[kTop2] = u.b;
        R.out[kNonFinite] = nu;
        const uint32_t fl = skin_flag(u, nu, R.skin);
        *R.flag = fl;
        __hip_atomic_store(R.hflag, (R.g.seq << kFlagBits) | fl, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// For skin tests on demand (the step loop reduces its own inside the next step
// launch).  From about this many partials (1M atoms) on several workgroups are
// the quicker; below, the counter's fences and the second merge cost more than
// they save.  parm_nlist_update with nothing to rebuild, one workgroup / several:
// 32,768 atoms 12.5 / 13.5 us, 262,144 13.7 / 14.6, 1M 24.1 / 23.5, 2M 34.9 / 32.4,
// 4M 61 / 51, 16M 221 / 192.
constexpr int kFinMultiMin = 4 * kFinal;

static void launch_finalize(int nparts, const ReduceBuf &R, hipStream_t s) {
    if (R.cnt && R.gpart && nparts >= kFinMultiMin) {
        const int G = std::max(1, std::min(kFinBlocks, (nparts + kFinThreads - 1) / kFinThreads));
        hipLaunchKernelGGL(k_finalize_skin, dim3(G), dim3(kFinThreads), 0, s, nparts, R);
        return;
    }
    hipLaunchKernelGGL(k_finalize, dim3(1), dim3(kFinal), 0, s, nparts, R);
}

hipError_t launch_finalize_sums(bool top, int nparts, const ReduceBuf &R, hipStream_t s) {
    if (top)
        hipLaunchKernelGGL(k_finalize_sums<true>, dim3(kTop1 + 1), dim3(kFinSumThreads), 0, s,
                           nparts, R);
    else
        hipLaunchKernelGGL(k_finalize_sums<false>, dim3(kTop1), dim3(kFinSumThreads), 0, s,
                           nparts, R);
    return hipGetLastError();
}

// Standalone first half of a step (drift + half kick) and skin test.
template <int D, bool DAMPED>
__global__ __launch_bounds__(kBlock) void k_drift(AtomArrays A, StepCoef c,
                                                  ReduceBuf R) {
    using PT = typename PosStore<D>::T;
    const int i = blockIdx.x * kBlock + threadIdx.x;
    Top2 top;
    double nonfinite = 0.0;
    if (i < A.n) {
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
        if (A.rank[i] >= 0) skin_atom<D>(x, A.xref, i, top, nonfinite);
    }
    double v[kRedWidth];
#pragma unroll
    for (int k = 0; k < kRedWidth; k++) v[k] = 0.0;
    v[kNonFinite] = nonfinite;
    block_partial<false, true, kBlock / kWave>(v, top, R, blockIdx.x);
}

// Skin test only (after a rebuild, or for update_list(false) on demand).
template <int D>
__global__ __launch_bounds__(kBlock) void k_skin(AtomArrays A, ReduceBuf R) {
    using PT = typename PosStore<D>::T;
    const int i = blockIdx.x * kBlock + threadIdx.x;
    Top2 top;
    double nonfinite = 0.0;
    if (i < A.n && A.rank[i] >= 0) {
        const Vec<D> x = PosStore<D>::load(static_cast<const PT *>(A.pos_in)[i]);
        skin_atom<D>(x, A.xref, i, top, nonfinite);
    }
    double v[kRedWidth];
#pragma unroll
    for (int k = 0; k < kRedWidth; k++) v[k] = 0.0;
    v[kNonFinite] = nonfinite;
    block_partial<false, true, kBlock / kWave>(v, top, R, blockIdx.x);
}

// Atom-wise observables (AtomGroup::kinetic_energy / momentum / mass,
// src/box.cpp:239-260, 401-411) and force statistics.
template <int D, int MODE>
__global__ __launch_bounds__(kBlock) void k_atom_sums(AtomArrays A, Vec<D> ov,
                                                      ReduceBuf R) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    double v[kRedWidth];
#pragma unroll
    for (int k = 0; k < kRedWidth; k++) v[k] = 0.0;
    Top2 top;
    if (i < A.n) {
        const double m = A.m[i];
        if (MODE == 0) {
            if (!(m == 0 || isinf(m))) {
                double c[D];
#pragma unroll
                for (int k = 0; k < D; k++) c[k] = A.v[k][i] - ov.c[k];
                double dd;
                if constexpr (D == 3)
                    dd = (c[0] * c[0] + c[1] * c[1]) + c[2] * c[2];
                else
                    dd = c[0] * c[0] + c[1] * c[1];
                v[0] = m / 2 * dd;
            }
            if (!is_fixed(m)) {
#pragma unroll
                for (int k = 0; k < D; k++) v[1 + k] = A.v[k][i] * m;
                v[4] = m;
            }
        } else {
            Vec<D> f;
#pragma unroll
            for (int k = 0; k < D; k++) f.c[k] = A.f[k][i];
            const double fn = sqrt(sqnorm<D>(f));
            v[0] = fn;
            top.add(fn);
        }
    }
    block_partial<true, MODE == 1, kBlock / kWave>(v, top, R, blockIdx.x);
}

template <int D>
__global__ __launch_bounds__(kBlock) void k_upload(AtomArrays A, int what,
                                                   const int32_t *__restrict__ orig,
                                                   const double *__restrict__ src) {
    using PT = typename PosStore<D>::T;
    const int s = blockIdx.x * kBlock + threadIdx.x;
    if (s >= A.n) return;
    const size_t o = (size_t)orig[s] * D;
    if (what == 0) {
        Vec<D> x;
#pragma unroll
        for (int k = 0; k < D; k++) x.c[k] = src[o + k];
        static_cast<PT *>(A.pos_out)[s] = PosStore<D>::make(x);
        return;
    }
    double *const *dst = what == 1 ? A.v : (what == 2 ? A.a : A.f);
#pragma unroll
    for (int k = 0; k < D; k++) dst[k][s] = src[o + k];
}

template <int D>
__global__ __launch_bounds__(kBlock) void k_download(AtomArrays A, int what,
                                                     const int32_t *__restrict__ orig,
                                                     double *__restrict__ dst) {
    using PT = typename PosStore<D>::T;
    const int s = blockIdx.x * kBlock + threadIdx.x;
    if (s >= A.n) return;
    const size_t o = (size_t)orig[s] * D;
    if (what == 0) {
        const Vec<D> x = PosStore<D>::load(static_cast<const PT *>(A.pos_in)[s]);
#pragma unroll
        for (int k = 0; k < D; k++) dst[o + k] = x.c[k];
        return;
    }
    double *const *src = what == 1 ? A.v : (what == 2 ? A.a : A.f);
#pragma unroll
    for (int k = 0; k < D; k++) dst[o + k] = src[k][s];
}

// ======================================================== host launchers
int reduce_blocks(int n) { return n <= 0 ? 1 : (n + kBlock - 1) / kBlock; }
int force_blocks(int n, int tpa) { return reduce_blocks(n * tpa); }
int force_partials(int n, const ListView &Lv) {
    return Lv.tiled && Lv.built ? Lv.ntiles : force_blocks(n, Lv.tpa);
}

size_t tiled_force_lds(int ndim, int prec, int kind, int ntypes, int smax) {
    const bool raw = prec == kFP64 && kind == kPairRepulsion;
    if (raw) return (size_t)smax * sizeof(double4);
    if (kind == kPairLJ) {
        // (lj_slots_bytes in step_tiled.hip) + type bytes
        const size_t real = prec == kFP64 ? sizeof(double) : sizeof(float);
        const size_t b = ((size_t)(smax + 1) * ndim * real + 15) & ~(size_t)15;
        return ntypes > 1 ? b + (size_t)smax + 1 : b;
    }
    if (ntypes == 1 && kind != kPairNone) return (size_t)smax * ndim * sizeof(double);
    return (size_t)smax * (sizeof(double4) + sizeof(int32_t));
}

// F(D, KIND, PREC) for the runtime dimension, pair kind and precision.
#define PARM_DISPATCH(F)                                                          \
    do {                                                                          \
        const bool rep = P.kind == kPairRepulsion, dbl = precision == kFP64;      \
        if (ndim == 3) {                                                          \
            if (rep) {                                                            \
                if (dbl) F(3, kPairRepulsion, kFP64); else F(3, kPairRepulsion, kMixed); \
            } else {                                                              \
                if (dbl) F(3, kPairLJ, kFP64); else F(3, kPairLJ, kMixed);        \
            }                                                                     \
        } else {                                                                  \
            if (rep) {                                                            \
                if (dbl) F(2, kPairRepulsion, kFP64); else F(2, kPairRepulsion, kMixed); \
            } else {                                                              \
                if (dbl) F(2, kPairLJ, kFP64); else F(2, kPairLJ, kMixed);        \
            }                                                                     \
        }                                                                         \
    } while (0)

hipError_t launch_force(int ndim, int precision, int stage, bool energy,
                        const AtomArrays &A, const ListView &Lv, const PairView &P,
                        const Box &box, const StepCoef &c, const ReduceBuf &R,
                        hipStream_t s) {
    if (energy != (stage == kStageSums)) return hipErrorInvalidValue;
    if (A.n <= 0) return hipSuccess;
    if (Lv.tiled && Lv.built) {
        if (Lv.ntiles <= 0) return hipSuccess;
#define PARM_F(D, K, Q) return force_tiled_part<D, K, Q>(stage, A, Lv, P, box, c, R, s)
        PARM_DISPATCH(PARM_F);
#undef PARM_F
    } else {
#define PARM_F(D, K, Q) return force_part<D, K, Q>(stage, energy, A, Lv, P, box, c, R, s)
        PARM_DISPATCH(PARM_F);
#undef PARM_F
    }
}

hipError_t launch_drift(int ndim, int stage, const AtomArrays &A, const StepCoef &c,
                        const ReduceBuf &R, hipStream_t s) {
    if (A.n <= 0) return hipSuccess;
    dim3 g(reduce_blocks(A.n)), b(kBlock);
    const bool damped = (stage == kStageDampedKick || stage == kStageDampedKickDrift);
    if (ndim == 3) {
        if (damped)
            hipLaunchKernelGGL((k_drift<3, true>), g, b, 0, s, A, c, R);
        else
            hipLaunchKernelGGL((k_drift<3, false>), g, b, 0, s, A, c, R);
    } else {
        if (damped)
            hipLaunchKernelGGL((k_drift<2, true>), g, b, 0, s, A, c, R);
        else
            hipLaunchKernelGGL((k_drift<2, false>), g, b, 0, s, A, c, R);
    }
    return hipGetLastError();
}

hipError_t launch_atom_sums(int ndim, int mode, const AtomArrays &A,
                            const double *originv, const ReduceBuf &R, hipStream_t s) {
    dim3 g(reduce_blocks(A.n)), b(kBlock);
    if (ndim == 3) {
        Vec<3> ov{{0, 0, 0}};
        if (originv)
            for (int k = 0; k < 3; k++) ov.c[k] = originv[k];
        if (mode == 0)
            hipLaunchKernelGGL((k_atom_sums<3, 0>), g, b, 0, s, A, ov, R);
        else
            hipLaunchKernelGGL((k_atom_sums<3, 1>), g, b, 0, s, A, ov, R);
    } else {
        Vec<2> ov{{0, 0}};
        if (originv)
            for (int k = 0; k < 2; k++) ov.c[k] = originv[k];
        if (mode == 0)
            hipLaunchKernelGGL((k_atom_sums<2, 0>), g, b, 0, s, A, ov, R);
        else
            hipLaunchKernelGGL((k_atom_sums<2, 1>), g, b, 0, s, A, ov, R);
    }
    return launch_finalize_sums(mode != 0, (int)g.x, R, s);
}

hipError_t launch_upload(int ndim, int what, const AtomArrays &A, const int32_t *orig,
                         const double *src, hipStream_t s) {
    if (A.n <= 0) return hipSuccess;
    dim3 g(reduce_blocks(A.n)), b(kBlock);
    if (ndim == 3)
        hipLaunchKernelGGL(k_upload<3>, g, b, 0, s, A, what, orig, src);
    else
        hipLaunchKernelGGL(k_upload<2>, g, b, 0, s, A, what, orig, src);
    return hipGetLastError();
}

hipError_t launch_download(int ndim, int what, const AtomArrays &A,
                           const int32_t *orig, double *dst, hipStream_t s) {
    if (A.n <= 0) return hipSuccess;
    dim3 g(reduce_blocks(A.n)), b(kBlock);
    if (ndim == 3)
        hipLaunchKernelGGL(k_download<3>, g, b, 0, s, A, what, orig, dst);
    else
        hipLaunchKernelGGL(k_download<2>, g, b, 0, s, A, what, orig, dst);
    return hipGetLastError();
}

hipError_t launch_skin(int ndim, const AtomArrays &A, const ReduceBuf &R, bool finalize,
                       hipStream_t s) {
    if (A.n <= 0) return hipSuccess;
    dim3 g(reduce_blocks(A.n)), b(kBlock);
    if (ndim == 3)
        hipLaunchKernelGGL((k_skin<3>), g, b, 0, s, A, R);
    else
        hipLaunchKernelGGL((k_skin<2>), g, b, 0, s, A, R);
    if (finalize) launch_finalize((int)g.x, R, s);
    return hipGetLastError();
}

}  // namespace parm
