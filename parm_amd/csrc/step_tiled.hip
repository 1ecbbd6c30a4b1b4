// step_tiled.hip -- pair forces over the tiled list (tiles.hpp), fused with
// the integrator stages exactly as k_force in force.hip.
//
// Reference behaviour restated (paths relative to the reference root):
//   NListed<A,P>::set_forces / energy / pressure / stress
//                                   src/interaction.hpp:2153-2291
//   LJAttractRepulsePair::forces/energy  src/interaction.hpp:1270-1298
//   RepulsionPair::forces/energy         src/interaction.hpp:1538-1556
//
// One workgroup per tile, TPA lanes per atom (kWave * TPA threads).  The
// tile's stencil (its runs, precomputed at the rebuild) is staged in LDS once
// per launch; each list entry is a staged slot, so a neighbour position is an
// LDS read instead of a gather from memory, and the list itself is 2 bytes
// per entry.  Three staging modes:
//   RAW   (FP64 repulsion): the positions themselves; each pair takes the
//         reference's minimum image diff(x_i, x_j), so every pair force is
//         the untiled kernel's bit for bit.
//   REL64 (FP64 LJ, mixed repulsion): the FP64 minimum-image offset of each
//         atom from the tile's middle atom.  A pair displacement is the
//         difference of two offsets (both in [-L/2, L/2], so one fold gives
//         the minimum image; when every offset of the tile is under L/4 the
//         difference already is, and the fold is skipped).  It differs from
//         diff(x_i, x_j) only by rounding (~1e-16 relative); the LJ in/out
//         decision within 1e-14 of the cutoff is taken on the exact d2, so the
//         set of interacting pairs is the reference's.
//         With several types a slot's type is a byte of its own and the pair
//         parameters are a table in LDS.
//   REL32 (mixed LJ): the same offsets rounded to FP32 and differenced in
//         FP32 (half the LDS traffic; the rounding of offsets of a few sigma
//         costs ~1e-6 sigma in r).  Repulsion does not use it: its force
//         eps (1 - R/sigma)/sigma cancels at small overlaps.
// Mixed precision decides in/out within 1e-5 of the cutoff in FP64 on the
// exact d2, as the untiled mixed path does.
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "pairs.hpp"
#include "stepcore.hpp"
#include "tiles.hpp"

namespace parm {

// FP64 LJAttractRepulsePair on a displacement r that may differ from the
// reference's by rounding; exact_d2() is the reference's d2, used only within
// 1e-14 of the cutoff (where lim_lo / lim_hi bracket it).
template <int D, bool ENERGY, typename Exact>
__device__ __forceinline__ void lj64x(const PairParam &pp, const Vec<D> &r,
                                      const Exact &exact_d2, double (&f)[D], PairAcc &acc) {
    // fused d2: within an ulp of the reference's (x*x + y*y) + z*z, far
    // inside the band in which exact_d2 decides
    double d2 = r.c[0] * r.c[0];
#pragma unroll
    for (int k = 1; k < D; k++) d2 = fma(r.c[k], r.c[k], d2);
    if (!(d2 < pp.lim_lo)) {
        if (d2 > pp.lim_hi) return;
        if (exact_d2() / pp.sig2 > pp.cut2) return;
    }
    double rsix, fmagR;
    const double fs = lj64_fs(pp, d2, rsix, fmagR);
#pragma unroll
    for (int k = 0; k < D; k++) f[k] = fma(fs, r.c[k], f[k]);
    if (ENERGY) {
        const double mid = 1.0 - rsix;
        const double e = pp.eps * (mid * mid) - pp.p5;
        acc.e += e;
        acc.w += fmagR;
#pragma unroll
        for (int a = 0; a < D; a++)
#pragma unroll
            for (int b = 0; b < D; b++) acc.s[a * D + b] += r.c[a] * (r.c[b] * fs);
        acc.contacts += (e != 0.0) ? 1.0 : 0.0;
        acc.overlaps += (e > 0.0) ? 1.0 : 0.0;
    }
}

// x folded into the primary image, x - L rint(x / L): one rounding, of
// magnitude ulp(L / 2), whatever image the unwrapped x is in.
template <int D>
__device__ __forceinline__ Vec<D> fold_image(const Vec<D> &x, const Box &b) {
    Vec<D> r;
#pragma unroll
    for (int k = 0; k < D; k++) r.c[k] = fma(-b.L[k], rint(x.c[k] * b.invL[k]), x.c[k]);
    return r;
}

// Minimum-image offset of x from the origin o (o already folded):
// d - L rint(d / L) with d = x - o.  `far` is set when x lies more than a box
// length from o along some dimension: x - o then rounds at its own
// magnitude, and offset_folded (x folded into the primary image first, every
// rounding at ulp(L)) should be taken instead.  The staged offsets need not
// round like the reference's remainder (they are differenced again).
template <int D>
__device__ __forceinline__ Vec<D> offset_from(const Vec<D> &x, const Vec<D> &o, const Box &b,
                                              bool &far) {
    Vec<D> r;
#pragma unroll
    for (int k = 0; k < D; k++) {
        const double d = x.c[k] - o.c[k];
        far |= fabs(d) > b.L[k];
        r.c[k] = fma(-b.L[k], rint(d * b.invL[k]), d);
    }
    return r;
}

template <int D>
__device__ __forceinline__ Vec<D> offset_folded(const Vec<D> &x, const Vec<D> &o,
                                                const Box &b) {
    const Vec<D> xf = fold_image<D>(x, b);
    Vec<D> r;
#pragma unroll
    for (int k = 0; k < D; k++) {
        const double d = xf.c[k] - o.c[k];
        r.c[k] = fma(-b.L[k], rint(d * b.invL[k]), d);
    }
    return r;
}

// The upper word of a double as a float: for magnitudes, the float order of
// upper words is the order of the doubles up to the lower word.
__device__ __forceinline__ float hi_float(double x) {
    return __uint_as_float((unsigned)((unsigned long long)__double_as_longlong(x) >> 32));
}

// List words per lane read ahead of the pair loop (two entries a word), and
// the entries the LJ loop evaluates side by side.
constexpr int kChunkWords = 4;
constexpr int kGroup = 4;
static_assert(kChunkWords % (kGroup / 2) == 0, "groups tile a chunk");

// One row of the LJ pair table (several types).
template <int PREC>
struct LjRow;
template <>
struct LjRow<kFP64> {
    double sig2, p6, lo, hi;
    __device__ static LjRow make(const PairParam &p) {
        return LjRow{p.sig2, p.p6, p.lim_lo, p.lim_hi};
    }
};
template <>
struct LjRow<kMixed> {
    float sig2, p6, lo, hi;
    __device__ static LjRow make(const PairParam &p) {
        return LjRow{p.sig2_f, p.p6_f, p.lim_f * 0.99999f, p.lim_f * 1.00001f};
    }
};

// Dynamic LDS of the LJ staging, in this order: smax + 1 slots of D offsets
// (the last one a stand-in for entries past a lane's count: see the pair
// loop), then with several types the pair table (TABLDS) and a type byte per
// slot.
template <int D, int PREC>
__host__ __device__ constexpr size_t lj_slots_bytes(int smax) {
    return (((size_t)(smax + 1) * D * (PREC == kFP64 ? 8 : 4)) + 15) & ~(size_t)15;
}

// TABLDS (LJ of several types, force stages): the pair table is copied to LDS;
// otherwise a pair's row comes from memory.  LDS is the faster as long as it has
// room for the table beside the stencil (up to about 24 types in FP64, 45 in
// FP32), and at that size both take the same: 262,144 atoms of 8 / 20 / 24 types
// in FP64 68.7 / 73.3 / 90.7 us per launch from LDS, 75.0 / 85.8 / 90.1 from
// memory; 28 / 32 / 64 types from memory 98 / 103 / 132, where the untiled list
// takes 168 / 173 / 201.
template <int D, int KIND, int PREC, bool SINGLE, bool HARM, int STAGE, int TPA, bool TABLDS>
__global__ __launch_bounds__(kWave *TPA) void k_force_tiled(AtomArrays A, ListView Lv,
                                                            PairView P, Box box, StepCoef c,
                                                            ReduceBuf R) {
    using PT = typename PosStore<D>::T;
    constexpr bool ENERGY = STAGE == kStageSums || STAGE == kStageNlcg;
    constexpr bool RAW = PREC == kFP64 && KIND != kPairLJ;
    constexpr bool REL32 = PREC != kFP64 && KIND == kPairLJ;
    // COMPACT (LJ, or one pair type, offsets staged): a slot is the D offsets
    // only (FP64: 8 D bytes, FP32: 4 D bytes), no atom index (the rare
    // exact-d2 path finds the atom from the runs): less LDS per workgroup,
    // more workgroups per CU.  LJ with several types keeps a type byte per
    // slot beside them.
    constexpr bool LJ = KIND == kPairLJ;
    constexpr bool COMPACT = LJ || (SINGLE && !RAW);
    using Real = typename std::conditional<REL32, float, double>::type;
    constexpr int NT = kWave * TPA;
    extern __shared__ double4 st64[];
    __shared__ int2 runs[kRunSlots];  // run_entry form (tiles.hpp)
    __shared__ int wides[TPA];
    double *stc64 = reinterpret_cast<double *>(st64);
    float *stc32 = reinterpret_cast<float *>(st64);
    Real *stc = reinterpret_cast<Real *>(st64);
    LjRow<PREC> *ljtab = reinterpret_cast<LjRow<PREC> *>(reinterpret_cast<char *>(st64) +
                                                         lj_slots_bytes<D, PREC>(Lv.smax));
    uint8_t *ljtype = reinterpret_cast<uint8_t *>(
        ljtab + (TABLDS ? (size_t)P.ntypes * P.ntypes : (size_t)0));
    int32_t *stj = reinterpret_cast<int32_t *>(st64 + Lv.smax);  // unless COMPACT or RAW

    constexpr bool STEP = STAGE == kStageVerletKickDrift || STAGE == kStageDampedKickDrift ||
                          STAGE == kStageVerletKick || STAGE == kStageDampedKick;
    // a step launch's first workgroup reduces the previous launch's skin test
    const int extra = STEP && R.g.nprev > 0 ? 1 : 0;
    if (STEP && extra && blockIdx.x == 0) {
        reduce_prev<TPA>(R);
        return;
    }
    const int blk = (int)blockIdx.x - extra;
    const int t = xcd_block(blk, (int)gridDim.x - extra);
    const int4 hdr = Lv.tiles[t];  // uniform
    const int lane = threadIdx.x % kWave;
    if (threadIdx.x < kRunSlots) runs[threadIdx.x] = run_entry(Lv.truns, t, threadIdx.x);
    // (the gate word arrives with them)
    if (STEP && step_stopped(R.g)) return;
    __syncthreads();
    const int a0 = hdr.x, tcnt = hdr.y;
    const int S = hdr.z >= 0 ? hdr.w : 0;
    const PT *pos = static_cast<const PT *>(A.pos_in);
    // the first wavefront updates the tile's atoms at the end (one lane per
    // atom); their inputs are loaded now, to arrive during the pair loop
    AtomIn<D> ain;
    const bool upd = STAGE != kStageSums && threadIdx.x < (unsigned)tcnt;
    if (upd) atom_load<D, STAGE>(A, a0 + (int)threadIdx.x, ain);
    // this thread's atom and lane, and what its pair loop reads from memory
    // (position, membership, entry count, the first chunk of list words),
    // also loaded now: their latency hides behind the staging.  The first
    // chunk is read whatever the lane's count (within the list array's
    // wcap words per lane); words past the count are never used.
    const int li = threadIdx.x / TPA, sub = threadIdx.x % TPA;
    const int i = a0 + li;
    const bool act = li < tcnt;
    Vec<D> xi;
#pragma unroll
    for (int k = 0; k < D; k++) xi.c[k] = 0.0;
    int rk = -1, nlane = 0;
    const uint32_t *wp = Lv.nbr + ((size_t)i * TPA + sub);
    const size_t wstride = (size_t)Lv.npad * TPA;
    uint32_t cur[kChunkWords];
#pragma unroll
    for (int q = 0; q < kChunkWords; q++) cur[q] = 0u;
    if (act) {
        xi = PosStore<D>::load(pos[i]);
        if (hdr.z >= 0) {
            rk = A.rank[i];
            nlane = Lv.lcount[(size_t)i * TPA + sub];
#pragma unroll
            for (int q = 0; q < kChunkWords; q++)
                if (q < Lv.wcap) cur[q] = wp[(size_t)q * wstride];
        }
    }
    if constexpr (LJ) {
        // the stand-in slot: far outside any cutoff (not folded: see `group`)
        if (threadIdx.x < D) stc[(size_t)Lv.smax * D + threadIdx.x] = (Real)(REL32 ? 1e18 : 1e150);
        if constexpr (!SINGLE) {
            if (threadIdx.x == 0) ljtype[Lv.smax] = 0;
            if constexpr (TABLDS)
                for (int q = threadIdx.x; q < P.ntypes * P.ntypes; q += NT)
                    ljtab[q] = LjRow<PREC>::make(P.tab[q]);
        }
    }
    // the tile origin, its middle atom (offsets half as large, and rounded
    // half as far in FP32, as from the first one): loaded now, folded once
    // the stencil's loads are issued
    PT xo_raw{};
    if (!RAW && S > 0) xo_raw = pos[a0 + (tcnt >> 1)];
    Vec<D> xo;
#pragma unroll
    for (int k = 0; k < D; k++) xo.c[k] = 0.0;
    bool xo_ready = false;
    // The largest upper words of the staged offsets' components, as floats
    // (the order of positive doubles is that of their upper words): an offset
    // of L/4 or more anywhere makes pair differences need the fold.
    float wmax[D];
#pragma unroll
    for (int k = 0; k < D; k++) wmax[k] = 0.0f;
    float half = 0.0f;  // upper word of the smallest half edge
    if (!RAW) {
        double h = box.halfL[0];
#pragma unroll
        for (int k = 1; k < D; k++) h = fmin(h, box.halfL[k]);
        half = hi_float(h);
    }
    // kStageBatch slots per thread at a time: their atom indices first (each
    // an independent binary lifting over the runs), then all their position
    // (and type) loads in flight together, then the stores.  A slot is folded
    // only where an atom of its wavefront's 64 lies in another image, and the
    // far and wide tests work on upper words: 179 -> 172 us per launch at 1M
    // atoms.  (The run of a wavefront's first slot from a ballot over runs
    // held in lanes, the others by readlane, in place of the interleaved
    // lifting: 184 us.)
    constexpr int kStageBatch = 5;
    for (int s0 = threadIdx.x; s0 < S; s0 += kStageBatch * NT) {
        int jb[kStageBatch];
        PT pb[kStageBatch];
        int tb[kStageBatch];
        {
            int sb[kStageBatch];
#pragma unroll
            for (int q = 0; q < kStageBatch; q++) sb[q] = s0 + q * NT;
            slot_atoms<kStageBatch>(runs, sb, jb);
        }
#pragma unroll
        for (int q = 0; q < kStageBatch; q++) {
            if (s0 + q * NT < S) {
                pb[q] = pos[jb[q]];
                tb[q] = SINGLE ? 0 : A.type[jb[q]];
            }
        }
        if (!RAW && !xo_ready) {
            xo = fold_image<D>(PosStore<D>::load(xo_raw), box);
            xo_ready = true;
        }
#pragma unroll
        for (int q = 0; q < kStageBatch; q++) {
        const int s = s0 + q * NT;
        if (s >= S) break;
        const int j = jb[q];
        const Vec<D> xj = PosStore<D>::load(pb[q]);
        const int tj = tb[q];
        Vec<D> v = xj;
        if (!RAW) {
            float hm = 0.0f;
#pragma unroll
            for (int k = 0; k < D; k++) {
                v.c[k] = xj.c[k] - xo.c[k];
                hm = fmaxf(hm, fabsf(hi_float(v.c[k])));
            }
            // an atom half an edge away is in another image: one
            // wave-uniform test; several lengths out, rarer still
            if (__ballot(hm >= half) != 0ull) {
                bool far = false;
                v = offset_from<D>(xj, xo, box, far);
                if (far) v = offset_folded<D>(xj, xo, box);
            }
#pragma unroll
            for (int k = 0; k < D; k++) wmax[k] = fmaxf(wmax[k], fabsf(hi_float(v.c[k])));
            if (!COMPACT) stj[s] = j;
        }
        if (COMPACT) {
#pragma unroll
            for (int k = 0; k < D; k++) {
                if (REL32)
                    stc32[s * D + k] = (float)v.c[k];
                else
                    stc64[s * D + k] = v.c[k];
            }
            if constexpr (LJ && !SINGLE) ljtype[s] = (uint8_t)tj;
        } else {
            double4 q;
            q.x = v.c[0];
            q.y = v.c[1];
            if (D == 3) {
                q.z = v.c[2];
                q.w = (double)tj;
            } else {
                q.z = (double)tj;
                q.w = 0.0;
            }
            st64[s] = q;
        }
        }
    }
    // (a thread with no slot to stage still needs the origin)
    if (!RAW && !xo_ready) xo = fold_image<D>(PosStore<D>::load(xo_raw), box);
    bool fold = false;
    if (!RAW) {
        bool wide = false;
#pragma unroll
        for (int k = 0; k < D; k++) wide |= wmax[k] >= hi_float(0.5 * box.halfL[k]);
        const bool any = __ballot(wide) != 0ull;
        if (lane == 0) wides[threadIdx.x / kWave] = any ? 1 : 0;
    }
    __syncthreads();
    if (!RAW) {
#pragma unroll
        for (int q = 0; q < TPA; q++) fold |= wides[q] != 0;
    }

    PairAcc acc;
    double fi[D];
    float f32[D];
#pragma unroll
    for (int k = 0; k < D; k++) {
        fi[k] = 0.0;
        f32[k] = 0.0f;
    }
    const bool member = act && hdr.z >= 0 && rk >= 0;
    if (member) {
        const PairParam *prow = P.tab;
        PairParam p0;
        if (SINGLE)
            p0 = P.p0;
        else
            prow = P.tab + (size_t)A.type[i] * P.ntypes;
        Vec<D> ri64 = xi;
        float ri[D], Lf[D], hLf[D];
#pragma unroll
        for (int k = 0; k < D; k++) ri[k] = Lf[k] = hLf[k] = 0.0f;
        if (!RAW) {
            ri64 = offset_folded<D>(xi, xo, box);
#pragma unroll
            for (int k = 0; k < D; k++) {
                ri[k] = (float)ri64.c[k];
                Lf[k] = (float)box.L[k];
                hLf[k] = (float)box.halfL[k];
            }
        }
        // the reference's d2 (for in/out decisions at the cutoff)
        auto exact_d2 = [&](int s) {
            int j;
            if constexpr (COMPACT) {
                j = slot_atom(runs, s);
            } else {
                j = stj[s];
            }
            const Vec<D> r = diff<D>(xi, PosStore<D>::load(pos[j]), box);
            return sqnorm<D>(r);
        };
        auto pair = [&](int s, auto fold_c) {
            constexpr bool FOLD = decltype(fold_c)::value;
            if constexpr (RAW) {
                const double4 q = st64[s];
                Vec<D> xj;
                xj.c[0] = q.x;
                xj.c[1] = q.y;
                if constexpr (D == 3) xj.c[2] = q.z;
                const int tj = SINGLE ? 0 : (int)(D == 3 ? q.w : q.z);
                const Vec<D> r = diff<D>(xi, xj, box);
                visit<D, KIND, PREC, ENERGY, HARM>(SINGLE ? p0 : prow[tj], r, fi, f32, acc);
            } else if constexpr (REL32) {
                int tj = 0;
                if constexpr (!SINGLE) tj = ljtype[s];
                float rf[D];
#pragma unroll
                for (int k = 0; k < D; k++) {
                    float d = ri[k] - stc32[s * D + k];
                    if (FOLD) d = d > hLf[k] ? d - Lf[k] : (d < -hLf[k] ? d + Lf[k] : d);
                    rf[k] = d;
                }
                lj32f<D, ENERGY>(SINGLE ? p0 : prow[tj], rf, [&]() { return exact_d2(s); },
                                 f32, acc);
            } else {
                double qc[3] = {0.0, 0.0, 0.0};
                int tj = 0;
                if constexpr (COMPACT) {
#pragma unroll
                    for (int k = 0; k < D; k++) qc[k] = stc64[s * D + k];
                    if constexpr (LJ && !SINGLE) tj = ljtype[s];
                } else {
                    const double4 q = st64[s];
                    qc[0] = q.x;
                    qc[1] = q.y;
                    qc[2] = q.z;
                    tj = (int)(D == 3 ? q.w : q.z);
                }
                Vec<D> r;
#pragma unroll
                for (int k = 0; k < D; k++) {
                    double d = ri64.c[k] - qc[k];
                    if (FOLD)
                        d = d > box.halfL[k] ? d - box.L[k]
                                             : (d < -box.halfL[k] ? d + box.L[k] : d);
                    r.c[k] = d;
                }
                const PairParam &pp = SINGLE ? p0 : prow[tj];
                if constexpr (PREC == kFP64) {
                    lj64x<D, ENERGY>(pp, r, [&]() { return exact_d2(s); }, fi, acc);
                } else {
                    float rf[D];
#pragma unroll
                    for (int k = 0; k < D; k++) rf[k] = (float)r.c[k];
                    rep32f<D, ENERGY, HARM>(pp, rf, [&]() { return exact_d2(s); }, f32, acc);
                }
            }
        };
        // kGroup entries (kGroup / 2 words) of the LJ list at once, with no
        // branch but one, uniform over the wavefront, for a pair within a
        // hair of the cutoff.  An entry out of range adds 0 * r.  The words
        // hold valid slots throughout: the stand-in slot smax takes the place
        // of the entries past a lane's count; it lies far outside the cutoff
        // unless the displacement is folded, where it is told by its number.
        //
        // The loop is bound by VALU issue (an FP64 instruction is 4 cycles of
        // a SIMD) and, below four waves a SIMD, by the ~25 cycles of each
        // compare-and-select and of each branch: 25 VALU instructions per
        // entry.  One-type FP64 at 1M atoms 186 -> 179 us per launch against
        // a form that decided each near-cutoff entry in place (four mask
        // merges and a jump per group); two types at 48,611 atoms 25.3 ->
        // 21.7 us against one entry at a time with parameters from memory
        // (untiled: 24.6 us).
        const int ti = SINGLE ? 0 : (int)A.type[i] * P.ntypes;
        auto displacement = [&](auto fold_c, Real (&r)[D]) {  // staged offset -> r
            constexpr bool FOLD = decltype(fold_c)::value;
#pragma unroll
            for (int k = 0; k < D; k++) {
                if constexpr (REL32) {
                    float d = ri[k] - r[k];
                    if (FOLD) d = fmaf(-Lf[k], rintf(d * (float)box.invL[k]), d);
                    r[k] = d;
                } else {
                    double d = ri64.c[k] - r[k];
                    if (FOLD) d = fma(-box.L[k], rint(d * box.invL[k]), d);
                    r[k] = d;
                }
            }
        };
        auto sq = [&](const Real (&r)[D]) {
            Real d2 = r[0] * r[0];
#pragma unroll
            for (int k = 1; k < D; k++) d2 = fma(r[k], r[k], d2);
            return d2;
        };
        auto ljrow = [&](int s) {
            if constexpr (SINGLE)
                return LjRow<PREC>::make(p0);
            else if constexpr (TABLDS)
                return ljtab[ti + ljtype[s]];
            else
                return LjRow<PREC>::make(prow[ljtype[s]]);
        };
        auto ljfs = [&](const LjRow<PREC> &q, Real d2) {
            if constexpr (PREC == kFP64) {
                return lj64_force(q.sig2, q.p6, d2);
            } else {
                const float idsq = __builtin_amdgcn_rcpf(d2);
                const float ir = q.sig2 * idsq;
                const float rsix = ir * ir * ir;
                return q.p6 * rsix * (rsix - 1.0f) * idsq;
            }
        };
        auto addf = [&](Real m, const Real (&r)[D]) {
#pragma unroll
            for (int k = 0; k < D; k++) {
                if constexpr (PREC == kFP64)
                    fi[k] = fma(m, r[k], fi[k]);
                else
                    f32[k] = fmaf(m, r[k], f32[k]);
            }
        };
        auto group = [&](uint32_t wa, uint32_t wb, auto fold_c) {
            constexpr bool FOLD = decltype(fold_c)::value;
            const int sl[kGroup] = {(int)(wa & 0xffffu), (int)(wa >> 16), (int)(wb & 0xffffu),
                                    (int)(wb >> 16)};
            Real r[kGroup][D], fs[kGroup];
            unsigned long long band = 0;
            // the group's slots are read together, before any is used
#pragma unroll
            for (int g = 0; g < kGroup; g++)
#pragma unroll
                for (int k = 0; k < D; k++) r[g][k] = stc[sl[g] * D + k];
#pragma unroll
            for (int g = 0; g < kGroup; g++) {
                displacement(fold_c, r[g]);
                const LjRow<PREC> q = ljrow(sl[g]);
                const Real d2 = sq(r[g]);
                bool in = d2 < q.lo, near = d2 <= q.hi;
                if (FOLD) {
                    in = in && sl[g] != Lv.smax;
                    near = near && sl[g] != Lv.smax;
                }
                band |= __ballot(near) & ~__ballot(in);
                if constexpr (PREC == kFP64) {
                    fs[g] = ljfs(q, far_unless(in, d2));
                } else {
                    const float m = ljfs(q, d2);
                    fs[g] = in ? m : 0.0f;
                }
            }
#pragma unroll
            for (int g = 0; g < kGroup; g++) addf(fs[g], r[g]);
            if (band) {
                // pairs near the cutoff: the reference's decision, on its d2
#pragma unroll 1
                for (int g = 0; g < kGroup; g++) {
                    const uint32_t w = g < 2 ? wa : wb;
                    const int s = (g & 1) ? (int)(w >> 16) : (int)(w & 0xffffu);
                    Real rr[D];
#pragma unroll
                    for (int k = 0; k < D; k++) rr[k] = stc[s * D + k];
                    displacement(fold_c, rr);
                    const LjRow<PREC> q = ljrow(s);
                    const Real d2 = sq(rr);
                    if (s != Lv.smax && !(d2 < q.lo) && d2 <= q.hi) {
                        const int j = slot_atom(runs, s);
                        const PairParam &pp = SINGLE ? p0 : P.tab[ti + (SINGLE ? 0 : ljtype[s])];
                        const double d2x = sqnorm<D>(diff<D>(xi, PosStore<D>::load(pos[j]), box));
                        if (d2x < pp.lim_lo || (!(d2x > pp.lim_hi) && !(d2x / pp.sig2 > pp.cut2)))
                            addf(ljfs(q, d2), rr);
                    }
                }
            }
        };
        // two entries per 32-bit word; for the LJ forms the lane's words
        // stream from memory kChunkWords at a time, each chunk loaded while
        // the one before it is evaluated (the first was loaded before the
        // staging); the loop runs for the wavefront's longest lane
        auto loop = [&](auto fold_c) {
            if constexpr (LJ && !ENERGY) {
                const uint32_t none = (uint32_t)Lv.smax * 0x10001u;
                // word w of the lane with the entries past the count replaced
                auto fix = [&](uint32_t v, int w) {
                    const int left = nlane - 2 * w;
                    v = left == 1 ? (v & 0xffffu) | (none & 0xffff0000u) : v;
                    return left > 0 ? v : none;
                };
                const int nw = (nlane + 1) >> 1;
                for (int w0 = 0; __ballot(w0 < nw) != 0ull; w0 += kChunkWords) {
                    uint32_t nxt[kChunkWords];
#pragma unroll
                    for (int q = 0; q < kChunkWords; q++) {
                        const int w = w0 + kChunkWords + q;
                        nxt[q] = none;
                        if (__ballot(w < nw) != 0ull) nxt[q] = wp[(size_t)w * wstride];
                    }
                    // (wave-uniform: most chunks are full in every lane)
                    if (__ballot(2 * (w0 + kChunkWords) > nlane) != 0ull) {
#pragma unroll
                        for (int q = 0; q < kChunkWords; q++) cur[q] = fix(cur[q], w0 + q);
                    }
#pragma unroll
                    for (int q = 0; q < kChunkWords; q += kGroup / 2)
                        if (__ballot(2 * (w0 + q) < nlane) != 0ull)
                            group(cur[q], cur[q + 1], fold_c);
#pragma unroll
                    for (int q = 0; q < kChunkWords; q++) cur[q] = nxt[q];
                }
            } else {
                // the other forms one entry at a time, the word two ahead
                // loaded while the current one is evaluated
                uint32_t w0 = cur[0], w1 = cur[1];
                for (int m = 0; m < nlane; m += 2) {
                    const uint32_t c = w0;
                    w0 = w1;
                    if (m + 4 < nlane) w1 = wp[(size_t)((m >> 1) + 2) * wstride];
                    pair((int)(c & 0xffffu), fold_c);
                    if (m + 1 < nlane) pair((int)(c >> 16), fold_c);
                }
            }
        };
        if (fold)
            loop(std::integral_constant<bool, true>());
        else
            loop(std::integral_constant<bool, false>());
    }
    if (PREC != kFP64) {
#pragma unroll
        for (int k = 0; k < D; k++) fi[k] += (double)f32[k];
    }
    // the atom's TPA lanes summed (xor butterfly; within a quad by DPP)
    if constexpr (TPA == 2) {
#pragma unroll
        for (int k = 0; k < D; k++) fi[k] += dpp_f64<kDppQuadXor1>(fi[k]);
    } else if constexpr (TPA >= 4) {
#pragma unroll
        for (int k = 0; k < D; k++) fi[k] = quad_sum(fi[k]);
#pragma unroll
        for (int o = 4; o < TPA; o <<= 1) {
#pragma unroll
            for (int k = 0; k < D; k++) fi[k] += __shfl_xor(fi[k], o);
        }
    }
    // The integrator's per-atom memory traffic is done by the first
    // wavefront, one lane per atom (64 consecutive atoms: coalesced), with
    // the summed forces passed through LDS.
    Top2 top;
    double nonfinite = 0.0, dots[4] = {0.0, 0.0, 0.0, 0.0};
    if (STAGE != kStageSums) {
        __shared__ double fsum[D][kTileAtoms];
        if (act && sub == 0) {
#pragma unroll
            for (int k = 0; k < D; k++) fsum[k][li] = fi[k];
        }
        __syncthreads();
        if (upd) {
            double fa[D];
#pragma unroll
            for (int k = 0; k < D; k++) fa[k] = fsum[k][threadIdx.x];
            atom_store<D, STAGE>(A, a0 + (int)threadIdx.x, fa, ain, c, top, nonfinite,
                                 dots);
        }
    }
    group_partials<D, STAGE, ENERGY, TPA, true>(acc, top, nonfinite, dots, R, blk);
}

// ======================================================== host launchers
namespace {

template <int D, int KIND, int PREC, bool SINGLE, bool HARM, int STAGE, int TPA>
hipError_t tiled_tt(const AtomArrays &A, const ListView &Lv, const PairView &P,
                    const Box &box, const StepCoef &c, const ReduceBuf &R, hipStream_t s) {
    constexpr bool DRIFT =
        (STAGE == kStageVerletKickDrift || STAGE == kStageDampedKickDrift);
    constexpr bool ENERGY = STAGE == kStageSums || STAGE == kStageNlcg;
    constexpr bool STEP = DRIFT || STAGE == kStageVerletKick || STAGE == kStageDampedKick;
    const size_t lds = tiled_force_lds(D, PREC, KIND, P.ntypes, Lv.smax);
    const dim3 g(Lv.ntiles + (STEP && R.g.nprev > 0 ? 1 : 0)), b(kWave * TPA);
    bool tab = false;
    if constexpr (KIND == kPairLJ && !SINGLE && !ENERGY) {
        const size_t bytes = (size_t)P.ntypes * P.ntypes * sizeof(LjRow<PREC>);
        tab = lds + bytes <= Lv.lds_max;
        if (tab)
            hipLaunchKernelGGL((k_force_tiled<D, KIND, PREC, SINGLE, HARM, STAGE, TPA, true>), g,
                               b, lds + bytes, s, A, Lv, P, box, c, R);
    }
    if (!tab)
        hipLaunchKernelGGL((k_force_tiled<D, KIND, PREC, SINGLE, HARM, STAGE, TPA, false>), g, b,
                           lds, s, A, Lv, P, box, c, R);
    // (before any other call: the next one's outcome would take its place)
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (R.done) (void)hipEventRecord(R.done, s);
    return ENERGY ? launch_finalize_sums(false, Lv.ntiles, R, s) : hipSuccess;
}

template <int D, int KIND, int PREC, bool SINGLE, bool HARM, int STAGE>
hipError_t tiled_t(const AtomArrays &A, const ListView &Lv, const PairView &P, const Box &box,
                   const StepCoef &c, const ReduceBuf &R, hipStream_t s) {
    switch (Lv.tpa) {
    case 1:
        return tiled_tt<D, KIND, PREC, SINGLE, HARM, STAGE, 1>(A, Lv, P, box, c, R, s);
    case 2:
        return tiled_tt<D, KIND, PREC, SINGLE, HARM, STAGE, 2>(A, Lv, P, box, c, R, s);
    case 8:
        return tiled_tt<D, KIND, PREC, SINGLE, HARM, STAGE, 8>(A, Lv, P, box, c, R, s);
    default:
        return tiled_tt<D, KIND, PREC, SINGLE, HARM, STAGE, 4>(A, Lv, P, box, c, R, s);
    }
}

template <int D, int KIND, int PREC, bool SINGLE, bool HARM>
hipError_t tiled_s(int stage, const AtomArrays &A, const ListView &Lv, const PairView &P,
                   const Box &box, const StepCoef &c, const ReduceBuf &R, hipStream_t s) {
    switch (stage) {
#define PARM_TSTAGE(S) \
    case S:            \
        return tiled_t<D, KIND, PREC, SINGLE, HARM, S>(A, Lv, P, box, c, R, s);
        PARM_TSTAGE(kStageForceOnly)
        PARM_TSTAGE(kStageForceA)
        PARM_TSTAGE(kStageVerletKick)
        PARM_TSTAGE(kStageVerletKickDrift)
        PARM_TSTAGE(kStageDampedKick)
        PARM_TSTAGE(kStageDampedKickDrift)
        PARM_TSTAGE(kStageSums)
        PARM_TSTAGE(kStageForceAdd)
        PARM_TSTAGE(kStageNlcg)
#undef PARM_TSTAGE
    }
    return hipErrorInvalidValue;
}

template <int D, int KIND, int PREC>
hipError_t tiled_k(int stage, const AtomArrays &A, const ListView &Lv, const PairView &P,
                   const Box &box, const StepCoef &c, const ReduceBuf &R, hipStream_t s) {
    if constexpr (KIND == kPairRepulsion) {
        if (P.harmonic) {
            return P.single ? tiled_s<D, KIND, PREC, true, true>(stage, A, Lv, P, box, c, R, s)
                            : tiled_s<D, KIND, PREC, false, true>(stage, A, Lv, P, box, c, R, s);
        }
    }
    return P.single ? tiled_s<D, KIND, PREC, true, false>(stage, A, Lv, P, box, c, R, s)
                    : tiled_s<D, KIND, PREC, false, false>(stage, A, Lv, P, box, c, R, s);
}

}  // namespace

// One dimension, pair kind and precision per object file (PARM_PART, set by
// the Makefile), so that the instantiations compile side by side.
template <int D, int KIND, int PREC>
hipError_t force_tiled_part(int stage, const AtomArrays &A, const ListView &Lv,
                            const PairView &P, const Box &box, const StepCoef &c,
                            const ReduceBuf &R, hipStream_t s) {
    return tiled_k<D, KIND, PREC>(stage, A, Lv, P, box, c, R, s);
}
template hipError_t force_tiled_part<PARM_PART_D, PARM_PART_KIND, PARM_PART_PREC>(
    int, const AtomArrays &, const ListView &, const PairView &, const Box &, const StepCoef &,
    const ReduceBuf &, hipStream_t);

}  // namespace parm
