// force.hip -- pair forces over the untiled device list, fused with the
// integrator stages and the skin test of step.hip.
//
// Reference behaviour restated (paths relative to the reference root):
//   NListed<A,P>::set_forces / energy / pressure / stress
//                                   src/interaction.hpp:2153-2291
//   LJAttractRepulsePair::forces/energy  src/interaction.hpp:1270-1298
//   RepulsionPair::forces/energy         src/interaction.hpp:1538-1556
//
// The device list is a FULL list (each pair appears in both atoms' rows), so
// each thread gathers the force on its own atom without atomics and in a
// fixed order.  The per-pair force from j on i uses r = diff(x_i, x_j); the
// visit from j computes -r bit for bit, so the two visits are exact negatives
// and only the summation order differs from the reference's half-list
// scatter.  Energies, virials and contact counts are halved.
//
// One dimension, pair kind and precision per object file (PARM_PART_*, set
// by the Makefile), so that the instantiations compile side by side.
#include "common.hpp"
#include "kernels.hpp"
#include "pairs.hpp"
#include "stepcore.hpp"

namespace parm {

// TPA lanes share one atom: lane `sub` visits list entries sub, sub + TPA, ...
// The list is stored in groups of TPA entries per atom (entry q of slot i at
// ((q / TPA) * npad + i) * TPA + q % TPA), so the 64 lanes of a wave read
// 64 consecutive words per step of the loop.  Two entries per lane are in
// flight at a time (both list words, then both position gathers) to hide
// memory latency.  The TPA partial forces are summed with a fixed butterfly,
// so the result is deterministic.
// With kAheadLanes lanes or more (few atoms: latency, not registers or
// bandwidth, bounds them) a lane's first kAhead entries are all in flight
// before the first is evaluated, instead of two at a time: 1000 LJ atoms at 8
// lanes, 200 steps 2320 -> 2130 us (4 or 8 ahead: within 3 % of 6).  A repulsion
// with a general exponent takes two: its rows are short, and each entry
// evaluated ahead is another copy of pow (2,003 disks, 200 steps: six 2615 us, two
// 2540).
constexpr int kAheadLanes = 8, kAhead = 6;

template <int D, int KIND, int PREC, bool SINGLE, bool HARM, int STAGE, bool ENERGY,
          int TPA>
__global__ __launch_bounds__(kBlock) void k_force(AtomArrays A, ListView Lv,
                                                  PairView P, Box box, StepCoef c,
                                                  ReduceBuf R) {
    using PT = typename PosStore<D>::T;
    constexpr bool STEP = STAGE == kStageVerletKickDrift || STAGE == kStageDampedKickDrift ||
                          STAGE == kStageVerletKick || STAGE == kStageDampedKick;
    // a step launch's first workgroup reduces the previous launch's skin test
    const int extra = STEP && R.g.nprev > 0 ? 1 : 0;
    if (STEP && extra && blockIdx.x == 0) {
        reduce_prev<kBlock / kWave>(R);
        return;
    }
    const int blk = (int)blockIdx.x - extra;
    const int gt = xcd_block(blk, (int)gridDim.x - extra) * kBlock + threadIdx.x;
    const int i = gt / TPA;
    const int sub = gt % TPA;
    const bool act = i < A.n;
    PairAcc acc;
    double fi[D];
    // (mixed) the FP32 sums of the even and the odd entries: one lane adds up
    // as two lanes do, so the result does not depend on which of them the
    // autotuner takes
    constexpr bool PAIRSUM = PREC != kFP64 && TPA == 1;
    constexpr int AHEAD = TPA < kAheadLanes ? 0 : (KIND == kPairRepulsion && !HARM ? 2 : kAhead);
    float f32[D], f32o[D];
#pragma unroll
    for (int k = 0; k < D; k++) {
        fi[k] = 0.0;
        f32[k] = f32o[k] = 0.0f;
    }

    const PT *pos = static_cast<const PT *>(A.pos_in);
    Vec<D> xi;
    if (act) xi = PosStore<D>::load(pos[i]);
    // the integrator inputs of the atom, loaded now to arrive during the
    // pair loop (lane sub == 0 applies the stage)
    AtomIn<D> ain;
    if (act && sub == 0) atom_load<D, STAGE, false>(A, i, ain);
    const bool member = act && A.rank[i] >= 0;
    // (the gate word arrives with the atom's own data)
    if (STEP && step_stopped(R.g)) return;
    if (member && Lv.built) {
        // lane sub's entries m = 0 .. nl-1 sit at (m * npad + i) * TPA + sub
        const size_t stride = (size_t)Lv.npad * TPA;
        const uint32_t *nb = Lv.nbr + (size_t)i * TPA + sub;
        uint32_t w[AHEAD > 0 ? AHEAD : 1];
        PT pw[AHEAD > 0 ? AHEAD : 1];
#pragma unroll
        for (int k = 0; k < AHEAD; k++) w[k] = k < Lv.wcap ? nb[(size_t)k * stride] : 0u;
        const int nl = Lv.lcount[(size_t)i * TPA + sub];
        const int tb = Lv.type_bits;
        const uint32_t tmask = (1u << tb) - 1u;
        const PairParam *row = P.tab;
        PairParam p0;
        if (SINGLE)
            p0 = P.p0;
        else
            row = P.tab + (size_t)A.type[i] * P.ntypes;
        int m = 0;
        size_t off = 0;
        if (AHEAD > 0) {
            // the lane's first entries: their list words, read with the entry
            // count (any word below wcap is in bounds; those past the count
            // are not used), then their gathers, all in flight together
#pragma unroll
            for (int k = 0; k < AHEAD; k++) pw[k] = k < nl ? pos[w[k] >> tb] : PT{};
#pragma unroll
            for (int k = 0; k < AHEAD; k++)
                if (k < nl) {
                    const Vec<D> r = diff<D>(xi, PosStore<D>::load(pw[k]), box);
                    visit<D, KIND, PREC, ENERGY, HARM>(SINGLE ? p0 : row[w[k] & tmask], r, fi,
                                                       f32, acc);
                }
            m = AHEAD;
            off = AHEAD * stride;
        }
        for (; m + 1 < nl; m += 2, off += 2 * stride) {
            const uint32_t e0 = nb[off];
            const uint32_t e1 = nb[off + stride];
            const PT pj0 = pos[e0 >> tb];
            const PT pj1 = pos[e1 >> tb];
            const Vec<D> r0 = diff<D>(xi, PosStore<D>::load(pj0), box);
            visit<D, KIND, PREC, ENERGY, HARM>(SINGLE ? p0 : row[e0 & tmask], r0, fi,
                                               f32, acc);
            const Vec<D> r1 = diff<D>(xi, PosStore<D>::load(pj1), box);
            visit<D, KIND, PREC, ENERGY, HARM>(SINGLE ? p0 : row[e1 & tmask], r1, fi,
                                               PAIRSUM ? f32o : f32, acc);
        }
        if (m < nl) {
            const uint32_t e0 = nb[off];
            const Vec<D> r0 = diff<D>(xi, PosStore<D>::load(pos[e0 >> tb]), box);
            visit<D, KIND, PREC, ENERGY, HARM>(SINGLE ? p0 : row[e0 & tmask], r0, fi,
                                               f32, acc);
        }
    }
    if (PREC != kFP64) {
#pragma unroll
        for (int k = 0; k < D; k++)
            fi[k] = PAIRSUM ? (double)f32[k] + (double)f32o[k] : (double)f32[k];
    }
    // sum the TPA partial forces of the atom (all lanes take part)
#pragma unroll
    for (int o = 1; o < TPA; o <<= 1) {
#pragma unroll
        for (int k = 0; k < D; k++) fi[k] += __shfl_xor(fi[k], o);
    }

    Top2 top;
    double nonfinite = 0.0, dots[4] = {0.0, 0.0, 0.0, 0.0};
    if (act && sub == 0) {
        ain.x = xi;
        atom_store<D, STAGE>(A, i, fi, ain, c, top, nonfinite, dots);
    }
    group_partials<D, STAGE, ENERGY, kBlock / kWave>(acc, top, nonfinite, dots, R, blk);
}

template <int D, int KIND, int PREC, bool SINGLE, bool HARM, int STAGE, int TPA>
static hipError_t launch_force_tt(bool energy, const AtomArrays &A, const ListView &Lv,
                                  const PairView &P, const Box &box, const StepCoef &c,
                                  const ReduceBuf &R, hipStream_t s) {
    constexpr bool DRIFT =
        (STAGE == kStageVerletKickDrift || STAGE == kStageDampedKickDrift);
    // energies and virials are accumulated by these stages only
    constexpr bool ENERGY = STAGE == kStageSums || STAGE == kStageNlcg;
    (void)energy;
    const int nb = force_blocks(A.n, TPA);
    constexpr bool STEP = DRIFT || STAGE == kStageVerletKick || STAGE == kStageDampedKick;
    dim3 g(nb + (STEP && R.g.nprev > 0 ? 1 : 0)), b(kBlock);
    hipLaunchKernelGGL((k_force<D, KIND, PREC, SINGLE, HARM, STAGE, ENERGY, TPA>), g, b, 0,
                       s, A, Lv, P, box, c, R);
    // (before any other call: the next one's outcome would take its place)
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (R.done) (void)hipEventRecord(R.done, s);
    return ENERGY ? launch_finalize_sums(false, nb, R, s) : hipSuccess;
}

template <int D, int KIND, int PREC, bool SINGLE, bool HARM, int STAGE>
static hipError_t launch_force_t(bool energy, const AtomArrays &A, const ListView &Lv,
                                 const PairView &P, const Box &box, const StepCoef &c,
                                 const ReduceBuf &R, hipStream_t s) {
    switch (Lv.tpa) {
    case 1:
        return launch_force_tt<D, KIND, PREC, SINGLE, HARM, STAGE, 1>(energy, A, Lv, P, box, c,
                                                                      R, s);
    case 2:
        return launch_force_tt<D, KIND, PREC, SINGLE, HARM, STAGE, 2>(energy, A, Lv, P, box, c,
                                                                      R, s);
    case 32:
        return launch_force_tt<D, KIND, PREC, SINGLE, HARM, STAGE, 32>(energy, A, Lv, P, box, c,
                                                                      R, s);
    case 16:
        return launch_force_tt<D, KIND, PREC, SINGLE, HARM, STAGE, 16>(energy, A, Lv, P, box, c,
                                                                      R, s);
    case 8:
        return launch_force_tt<D, KIND, PREC, SINGLE, HARM, STAGE, 8>(energy, A, Lv, P, box, c,
                                                                      R, s);
    default:
        return launch_force_tt<D, KIND, PREC, SINGLE, HARM, STAGE, 4>(energy, A, Lv, P, box, c,
                                                                      R, s);
    }
}

template <int D, int KIND, int PREC, bool SINGLE, bool HARM>
static hipError_t launch_force_s(int stage, bool energy, const AtomArrays &A,
                                 const ListView &Lv, const PairView &P, const Box &box,
                                 const StepCoef &c, const ReduceBuf &R, hipStream_t s) {
    switch (stage) {
#define PARM_STAGE(S)                                                                 \
    case S:                                                                           \
        return launch_force_t<D, KIND, PREC, SINGLE, HARM, S>(energy, A, Lv, P, box,  \
                                                              c, R, s);
        PARM_STAGE(kStageForceOnly)
        PARM_STAGE(kStageForceA)
        PARM_STAGE(kStageVerletKick)
        PARM_STAGE(kStageVerletKickDrift)
        PARM_STAGE(kStageDampedKick)
        PARM_STAGE(kStageDampedKickDrift)
        PARM_STAGE(kStageSums)
        PARM_STAGE(kStageForceAdd)
        PARM_STAGE(kStageNlcg)
#undef PARM_STAGE
    }
    return hipErrorInvalidValue;
}

template <int D, int KIND, int PREC>
static hipError_t launch_force_k(int stage, bool energy, const AtomArrays &A,
                                 const ListView &Lv, const PairView &P, const Box &box,
                                 const StepCoef &c, const ReduceBuf &R, hipStream_t s) {
    if constexpr (KIND == kPairRepulsion) {
        if (P.harmonic) {
            return P.single ? launch_force_s<D, KIND, PREC, true, true>(stage, energy, A, Lv,
                                                                        P, box, c, R, s)
                            : launch_force_s<D, KIND, PREC, false, true>(stage, energy, A, Lv,
                                                                         P, box, c, R, s);
        }
    }
    return P.single ? launch_force_s<D, KIND, PREC, true, false>(stage, energy, A, Lv, P, box,
                                                                 c, R, s)
                    : launch_force_s<D, KIND, PREC, false, false>(stage, energy, A, Lv, P, box,
                                                                  c, R, s);
}

template <int D, int KIND, int PREC>
hipError_t force_part(int stage, bool energy, const AtomArrays &A, const ListView &Lv,
                      const PairView &P, const Box &box, const StepCoef &c,
                      const ReduceBuf &R, hipStream_t s) {
    return launch_force_k<D, KIND, PREC>(stage, energy, A, Lv, P, box, c, R, s);
}
template hipError_t force_part<PARM_PART_D, PARM_PART_KIND, PARM_PART_PREC>(
    int, bool, const AtomArrays &, const ListView &, const PairView &, const Box &,
    const StepCoef &, const ReduceBuf &, hipStream_t);

}  // namespace parm
