// batch_force.hip -- pair forces of all systems of a batch (batch.hip), fused
// with the integrator stages.  One dimension, pair kind and precision per
// object file (PARM_PART_*, set by the Makefile).
#include "common.hpp"
#include "kernels.hpp"
#include "pairs.hpp"

namespace parm {

// ---------------------------------------------------------------- forces
constexpr int kBatchAhead = 4;  // list entries per lane evaluated before the loop

template <int D, int KIND, int PREC, bool SINGLE, bool HARM, int STAGE, bool ENERGY,
          int TPA>
__global__ __launch_bounds__(kBlock) void k_batch_force(BatchArrays A, ListView Lv,
                                                        PairView P, StepCoef c,
                                                        double *__restrict__ eatom) {
    using PT = typename PosStore<D>::T;
    constexpr bool DRIFT =
        (STAGE == kStageVerletKickDrift || STAGE == kStageDampedKickDrift);
    constexpr bool DAMPED =
        (STAGE == kStageDampedKick || STAGE == kStageDampedKickDrift);
    // consecutive workgroups (consecutive atoms: one system's, mostly) on one
    // XCD, so each system's positions, which its atoms' neighbour gathers
    // read, are held in one L2 rather than in all eight
    const int gt = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    const int i = gt / TPA;
    const int sub = gt % TPA;
    const bool act = i < A.ntot;
    PairAcc acc;
    double fi[D];
    float f32[D];
#pragma unroll
    for (int k = 0; k < D; k++) {
        fi[k] = 0.0;
        f32[k] = 0.0f;
    }
    const PT *pos = static_cast<const PT *>(A.pos_in);
    Vec<D> xi;
    Box box{};
    if (act) {
        xi = PosStore<D>::load(pos[i]);
        box = A.geom[A.sys[i]].box;
    }
    // the integrator inputs of the atom (lane sub == 0 applies the stage),
    // loaded now to arrive during the pair loop
    double m_i = 1.0, v_i[D], x0_i[D];
#pragma unroll
    for (int k = 0; k < D; k++) v_i[k] = x0_i[k] = 0.0;
    if (act && sub == 0 && STAGE != kStageSums && STAGE != kStageForceOnly) {
        m_i = A.m[i];
        if (STAGE != kStageForceA) {
#pragma unroll
            for (int k = 0; k < D; k++) v_i[k] = A.v[k][i];
        }
        if (DRIFT) {
            const Vec<D> x0 = PosStore<D>::load(static_cast<const PT *>(A.xref)[i]);
#pragma unroll
            for (int k = 0; k < D; k++) x0_i[k] = x0.c[k];
        }
    }
    if (act && Lv.built) {
        const size_t stride = (size_t)Lv.npad * TPA;
        const uint32_t *nb = Lv.nbr + (size_t)i * TPA + sub;
        // the lane's first kBatchAhead entries: their list words are read
        // together with the entry count (any word within the list array's
        // wcap per lane is in bounds; those past the count are not used),
        // then their neighbours' positions are gathered together
        uint32_t w[kBatchAhead];
#pragma unroll
        for (int k = 0; k < kBatchAhead; k++)
            w[k] = k < Lv.wcap ? nb[(size_t)k * stride] : 0u;
        const int cnt = Lv.ncount[i];
        const int tb = Lv.type_bits;
        const uint32_t tmask = (1u << tb) - 1u;
        const PairParam *row = P.tab;
        PairParam p0;
        if (SINGLE)
            p0 = P.p0;
        else
            row = P.tab + (size_t)A.type[i] * P.ntypes;
        PT pw[kBatchAhead];
#pragma unroll
        for (int k = 0; k < kBatchAhead; k++)
            if (sub + k * TPA < cnt) pw[k] = pos[w[k] >> tb];
#pragma unroll
        for (int k = 0; k < kBatchAhead; k++) {
            if (sub + k * TPA < cnt) {
                const Vec<D> r = diff<D>(xi, PosStore<D>::load(pw[k]), box);
                visit<D, KIND, PREC, ENERGY, HARM>(SINGLE ? p0 : row[w[k] & tmask], r, fi,
                                                   f32, acc);
            }
        }
        // the rest: the next two entries loaded while the current two are
        // evaluated
        int q = sub + kBatchAhead * TPA;
        size_t off = (size_t)kBatchAhead * stride;
        uint32_t n0 = q < cnt ? nb[off] : 0u;
        uint32_t n1 = q + TPA < cnt ? nb[off + stride] : 0u;
        for (; q + TPA < cnt; q += 2 * TPA, off += 2 * stride) {
            const uint32_t e0 = n0;
            const uint32_t e1 = n1;
            if (q + 2 * TPA < cnt) n0 = nb[off + 2 * stride];
            if (q + 3 * TPA < cnt) n1 = nb[off + 3 * stride];
            const PT pj0 = pos[e0 >> tb];
            const PT pj1 = pos[e1 >> tb];
            const Vec<D> r0 = diff<D>(xi, PosStore<D>::load(pj0), box);
            visit<D, KIND, PREC, ENERGY, HARM>(SINGLE ? p0 : row[e0 & tmask], r0, fi, f32,
                                               acc);
            const Vec<D> r1 = diff<D>(xi, PosStore<D>::load(pj1), box);
            visit<D, KIND, PREC, ENERGY, HARM>(SINGLE ? p0 : row[e1 & tmask], r1, fi, f32,
                                               acc);
        }
        if (q < cnt) {
            const uint32_t e0 = n0;
            const Vec<D> r0 = diff<D>(xi, PosStore<D>::load(pos[e0 >> tb]), box);
            visit<D, KIND, PREC, ENERGY, HARM>(SINGLE ? p0 : row[e0 & tmask], r0, fi, f32,
                                               acc);
        }
    }
    if (PREC != kFP64) {
#pragma unroll
        for (int k = 0; k < D; k++) fi[k] = (double)f32[k];
    }
    double e = acc.e, nc = acc.contacts, w = acc.w, no = acc.overlaps;
#pragma unroll
    for (int o = 1; o < TPA; o <<= 1) {
#pragma unroll
        for (int k = 0; k < D; k++) fi[k] += __shfl_xor(fi[k], o);
        if (ENERGY) {
            e += __shfl_xor(e, o);
            nc += __shfl_xor(nc, o);
            w += __shfl_xor(w, o);
            no += __shfl_xor(no, o);
        }
    }
    if (!act || sub != 0) return;
    if (ENERGY) {
        // the full list visits each pair from both atoms: halves per atom
        double4 *ea = reinterpret_cast<double4 *>(eatom);
        ea[i] = double4{0.5 * e, nc, 0.5 * w, no};
    }
    if (STAGE == kStageSums) return;
    // fused kick + drift: f and a are stored by the run's last (plain kick)
    // launch only; nothing reads them in between
    if constexpr (!DRIFT) {
#pragma unroll
        for (int k = 0; k < D; k++) A.f[k][i] = fi[k];
    }
    if (STAGE == kStageForceOnly) return;
    const double m = m_i;
    const bool fixed = is_fixed(m);
    double a[D];
#pragma unroll
    for (int k = 0; k < D; k++) a[k] = fixed ? 0.0 : fi[k] / m;
    if constexpr (!DRIFT) {
#pragma unroll
        for (int k = 0; k < D; k++) A.a[k][i] = a[k];
    }
    if (STAGE == kStageForceA) return;
    double v[D];
#pragma unroll
    for (int k = 0; k < D; k++) v[k] = v_i[k];
    if (!fixed) {
#pragma unroll
        for (int k = 0; k < D; k++) v[k] = v[k] + a[k] * (DAMPED ? c.k4 : c.k2);
    }
    if (DRIFT) {
        Vec<D> xn = xi;
        drift_atom<D, DAMPED>(xn, v, a, fixed, c);
        static_cast<PT *>(A.pos_out)[i] = PosStore<D>::make(xn);
        Vec<D> d;
#pragma unroll
        for (int k = 0; k < D; k++) d.c[k] = xn.c[k] - x0_i[k];
        A.disp[i] = sqrt(sqnorm<D>(d));
    }
#pragma unroll
    for (int k = 0; k < D; k++) A.v[k][i] = v[k];
}

static inline int nblk1(long n) { return (int)((n + kBlock - 1) / kBlock); }

template <int D, int KIND, int PREC, bool SINGLE, bool HARM, int STAGE, int TPA>
static void bforce_tt(bool energy, const BatchArrays &A, const ListView &Lv,
                      const PairView &P, const StepCoef &c, double *eatom, hipStream_t s) {
    // energies are accumulated by the sums stage only
    (void)energy;
    dim3 g(nblk1((long)A.ntot * TPA)), b(kBlock);
    hipLaunchKernelGGL(
        (k_batch_force<D, KIND, PREC, SINGLE, HARM, STAGE, STAGE == kStageSums, TPA>), g, b,
        0, s, A, Lv, P, c, eatom);
}

template <int D, int KIND, int PREC, bool SINGLE, bool HARM, int STAGE>
static void bforce_t(bool energy, const BatchArrays &A, const ListView &Lv,
                     const PairView &P, const StepCoef &c, double *eatom, hipStream_t s) {
    switch (Lv.tpa) {
    case 1:
        bforce_tt<D, KIND, PREC, SINGLE, HARM, STAGE, 1>(energy, A, Lv, P, c, eatom, s);
        break;
    case 2:
        bforce_tt<D, KIND, PREC, SINGLE, HARM, STAGE, 2>(energy, A, Lv, P, c, eatom, s);
        break;
    case 32:
        bforce_tt<D, KIND, PREC, SINGLE, HARM, STAGE, 32>(energy, A, Lv, P, c, eatom, s);
        break;
    case 16:
        bforce_tt<D, KIND, PREC, SINGLE, HARM, STAGE, 16>(energy, A, Lv, P, c, eatom, s);
        break;
    case 8:
        bforce_tt<D, KIND, PREC, SINGLE, HARM, STAGE, 8>(energy, A, Lv, P, c, eatom, s);
        break;
    default:
        bforce_tt<D, KIND, PREC, SINGLE, HARM, STAGE, 4>(energy, A, Lv, P, c, eatom, s);
        break;
    }
}

template <int D, int KIND, int PREC, bool SINGLE, bool HARM>
static void bforce_s(int stage, bool energy, const BatchArrays &A, const ListView &Lv,
                     const PairView &P, const StepCoef &c, double *eatom, hipStream_t s) {
    switch (stage) {
#define PARM_BSTAGE(S)                                                          \
    case S:                                                                     \
        bforce_t<D, KIND, PREC, SINGLE, HARM, S>(energy, A, Lv, P, c, eatom, s); \
        break;
        PARM_BSTAGE(kStageForceOnly)
        PARM_BSTAGE(kStageForceA)
        PARM_BSTAGE(kStageVerletKick)
        PARM_BSTAGE(kStageVerletKickDrift)
        PARM_BSTAGE(kStageDampedKick)
        PARM_BSTAGE(kStageDampedKickDrift)
        PARM_BSTAGE(kStageSums)
#undef PARM_BSTAGE
    }
}

template <int D, int KIND, int PREC>
static void bforce_k(int stage, bool energy, const BatchArrays &A, const ListView &Lv,
                     const PairView &P, const StepCoef &c, double *eatom, hipStream_t s) {
    if constexpr (KIND == kPairRepulsion) {
        if (P.harmonic) {
            if (P.single)
                bforce_s<D, KIND, PREC, true, true>(stage, energy, A, Lv, P, c, eatom, s);
            else
                bforce_s<D, KIND, PREC, false, true>(stage, energy, A, Lv, P, c, eatom, s);
            return;
        }
    }
    {
        if (P.single)
            bforce_s<D, KIND, PREC, true, false>(stage, energy, A, Lv, P, c, eatom, s);
        else
            bforce_s<D, KIND, PREC, false, false>(stage, energy, A, Lv, P, c, eatom, s);
    }
}

template <int D, int KIND, int PREC>
void batch_force_part(int stage, bool energy, const BatchArrays &A, const ListView &Lv,
                      const PairView &P, const StepCoef &c, double *eatom, hipStream_t s) {
    bforce_k<D, KIND, PREC>(stage, energy, A, Lv, P, c, eatom, s);
}
template void batch_force_part<PARM_PART_D, PARM_PART_KIND, PARM_PART_PREC>(
    int, bool, const BatchArrays &, const ListView &, const PairView &, const StepCoef &,
    double *, hipStream_t);

}  // namespace parm
