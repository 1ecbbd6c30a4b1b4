// kernels.hpp -- host-side launchers of the device kernels (internal API of
// libparm_hip.so; the public C ABI is include/parm_hip.h).
#pragma once

#include <hip/hip_runtime.h>

#include <string>

#include <cstdint>

#include "common.hpp"

namespace parm {

// Periodic cell grid used by the list rebuild.
struct CellGrid {
    int nc[3];       // cells per dimension (1 when the box is under 3 list radii)
    int ncell;       // product of nc over the active dimensions
    double invL[3];  // 1 / box edge
};

// ---------------------------------------------------------------- nlist.hip
int radix_blocks(int n);
hipError_t launch_cell_keys(int ndim, int n, const void *pos, const int32_t *rank,
                            const CellGrid &g, uint32_t *keys, int32_t *vals, int *info,
                            hipStream_t s);
hipError_t radix_sort(int n, int bits, uint32_t *&keys, int32_t *&vals,
                      uint32_t *&tmp_keys, int32_t *&tmp_vals, uint32_t *hist,
                      hipStream_t s);
template <typename T>
hipError_t gather(int n, const int32_t *perm, const T *src, T *dst, hipStream_t s);
// One permutation launch over every per-slot column: slot i of each
// destination takes slot perm[i] of its source.
constexpr int kPermD = 11, kPermI = 3;
struct PermuteSet {
    const void *pos_src[2];
    void *pos_dst[2];
    const double *d_src[kPermD];
    double *d_dst[kPermD];
    const int32_t *i_src[kPermI];
    int32_t *i_dst[kPermI];
    int nd, ni;
};
hipError_t launch_permute(int ndim, int n, const int32_t *perm, const PermuteSet &P,
                          hipStream_t s);
// Order by cell of a system whose atoms are all list members: the cells'
// starts (cstart, ncell + 1) and atoms in arrival order (slot), then every
// column into the stable order, the sorted keys, the wrapped positions and,
// with skin, the partials (reduce_blocks(n)) of the skin test of pos_src[1]
// against pos_src[0].  ukeys, arrival: n words of scratch; count: ncell words,
// zero before and after; total: scan_tiles(ncell) words.
int scan_tiles(int ncell);
struct ReduceBuf;
hipError_t launch_cell_order(int ndim, int n, const void *pos, const CellGrid &g,
                             uint32_t *ukeys, int32_t *arrival, uint32_t *count,
                             uint32_t *total, int32_t *cstart, int32_t *slot, int *info,
                             hipStream_t s);
hipError_t launch_cell_permute(int ndim, int n, const int32_t *slot, const uint32_t *ukeys,
                               const int32_t *cstart, const CellGrid &g, const Box &box,
                               uint32_t *keys, void *xw, const PermuteSet &P,
                               const ReduceBuf *skin, hipStream_t s);
hipError_t launch_cell_bounds(int n, int ncell, const uint32_t *keys, int32_t *start,
                              hipStream_t s);
// Outcome of one list build, stored by the build's last launch in pinned
// host memory: the sum and the largest of the per-atom entry counts, the
// flag word of the build (then cleared on the device), and for a
// speculative tiled build the tile plan it ran against.
struct BuildReport {
    unsigned long long sum, max;
    int ntiles, smax, bad;
    uint32_t flag;
    int ok;        // the verdict of a build that a step launch waits for
    uint32_t seq;  // the launch's number, stored last
};

// NeighborList::ignore exclusions (src/trackers.hpp:190-193): excluded
// partners of each atom as a CSR over original atom indices (both directions
// stored, partners sorted); orig maps a device slot to its original index.
// any == 0 disables the test.
struct ExclView {
    const int32_t *orig;
    const int32_t *off;   // natoms + 1
    const int32_t *part;  // off[natoms] partners
    int any;
};

// Builds the full list (and xref = pos); stats[0] = sum of counts, stats[1] =
// max count; part holds 2 * build_blocks(n) scratch words.  wrapped: xw
// already holds the wrapped positions.  report: a device-visible pinned
// BuildReport, or null.
int build_blocks(int n);
hipError_t launch_build_list(int ndim, int n, const void *pos, void *xw,
                             const int32_t *rank, const double *diam, const int32_t *type,
                             const uint32_t *keys, const int32_t *cstart,
                             const CellGrid &g, const Box &box, double skin, double dmax,
                             int type_bits, int tpa, int cap, int npad, uint32_t *nbr,
                             int32_t *ncount, uint16_t *lcount, void *xref,
                             unsigned long long *part, unsigned long long *stats,
                             uint32_t *flag, const ExclView &ex, bool wrapped,
                             BuildReport *report, uint32_t seq, hipStream_t s);

// Tiled layout (tiles.hpp).  launch_tiles fills tiles (cap_tiles records) and,
// info having been cleared by the ordering launches, info[0] = tiles and
// info[2] != 0 when they exceed cap_tiles.
hipError_t launch_tiles(int ndim, int n, const CellGrid &g, const uint32_t *keys,
                        const int32_t *cstart, int cap_tiles, int4 *tiles, int2 *truns,
                        int *info, hipStream_t s);
// info[1] = largest stencil, info[2] |= one does not fit (launch_tiles leaves
// info[1] alone; a speculative build's report carries both by itself).
hipError_t launch_tile_extremes(const int4 *tiles, int *info, hipStream_t s);
size_t tiled_build_lds(int smax);
// spec == null: ntiles and smax are the plan's.  spec == the plan's info
// (launch_tiles, not yet read by the host): ntiles and smax are bounds;
// tiles past info[0] do nothing, and a tile with more than smax staged slots
// (or none that fit) sets kFlagReplan instead of building.  verdict (may be
// null): 0 when the speculative build stands (the plan fits its bounds, the list
// its capacity), else kFlagStopped: the gate of a step launch queued behind it.
// uni: every list
// member has the same diameter.
hipError_t launch_build_tiled(int ndim, int n, int ntiles, int smax, const int4 *tiles,
                              const int2 *truns, const void *pos, void *xw, const int32_t *rank,
                              const double *diam, const int32_t *type, int type_bits,
                              const uint32_t *keys, const int32_t *cstart, const CellGrid &g,
                              const Box &box, double skin, double dmax, int tpa, int cap,
                              int npad, bool out32, void *nbr, int32_t *ncount,
                              uint16_t *lcount, void *xref, unsigned long long *part,
                              unsigned long long *stats, uint32_t *flag, const int *spec,
                              int uni, const ExclView &ex, bool wrapped,
                              BuildReport *report, uint32_t seq, uint32_t *verdict,
                              hipStream_t s);
hipError_t launch_tiled_to_global(int ndim, int ntiles, const int4 *tiles,
                                  const uint32_t *keys, const int32_t *cstart,
                                  const CellGrid &g, const uint16_t *nb16,
                                  const uint16_t *lcount, const int32_t *type, int type_bits,
                                  int tpa, int npad, uint32_t *out, hipStream_t s);

// -------------------------------------------------------------- step.hip
enum PairKind : int { kPairNone = 0, kPairLJ = 1, kPairRepulsion = 2 };
enum Precision : int { kFP64 = 0, kMixed = 1 };

// Per type-pair parameters, precomputed on the host exactly as the
// reference's pair constructors compute them (src/interaction.hpp:1256-1269,
// 1532-1537).  Indexed [t1 * ntypes + t2].
struct PairParam {
    double eps;        // LJ: |eps| ; Repulsion: sqrt(e1 e2)
    double sig;        // (s1 + s2) / 2
    double sig2;       // sig * sig
    double cut2;       // LJ: cut * cut (in sigma units) ; Repulsion: sig * sig
    double lim_lo;     // d2 below: surely inside the cutoff
    double lim_hi;     // d2 above: surely outside
    double p5;         // LJ: cut_energy      ; Repulsion: exponent n
    double p6;         // LJ: 12 * eps        ; Repulsion: n - 1
    float eps_f, sig2_f, p5_f, p6_f;  // single-precision copies (mixed mode)
    float lim_f, sig_f, isig_f, pad_f;
};

// Per-system views handed to the step kernels.
struct AtomArrays {
    int n;                 // slots
    const void *pos_in;    // PosStore<D>::T*
    void *pos_out;         // fused steps write the drifted positions here
    double *v[3], *a[3], *f[3];
    const double *m;
    const int32_t *type;   // pair-table type of each slot
    const int32_t *rank;   // < 0: not a list member (no pair forces, no skin test)
    const void *xref;      // positions at the last rebuild
};

struct ListView {
    const uint32_t *nbr;
    const int32_t *ncount;
    const uint16_t *lcount;  // entries of lane sub of slot i: lcount[i * tpa + sub]
    int npad;
    int type_bits;
    int tpa;               // lanes per atom; entries grouped by tpa (see k_force)
    int built;             // 0: the list was never built -> no pairs
    // tiled layout (tiles.hpp): nbr holds 16-bit staged slots
    int tiled;
    int ntiles;            // tiles = workgroups of a tiled force launch
    int smax;              // largest staged stencil of any tile
    int wcap;              // 32-bit words per lane the list array holds (cap / tpa)
    size_t lds_max;        // dynamic LDS that a tiled launch may take
    const int4 *tiles;
    const int2 *truns;     // kTileRuns runs per tile (tiles.hpp)
    const uint32_t *keys;  // sorted cell keys of the last rebuild
    const int32_t *cstart;
    CellGrid grid;
};

struct PairView {
    int kind;
    int ntypes;
    int single;            // 1: one type pair (parameters uniform)
    int harmonic;          // Repulsion with n == 2 for every type pair
    const PairParam *tab;
    PairParam p0;          // tab[0] by value: a one-type kernel reads it from
                           // its arguments (scalar registers), not from memory
};

// Integrator stage fused into the force kernel.
enum Stage : int {
    kStageForceOnly = 0,   // Collection::set_forces(false): f only
    kStageForceA = 1,      // set_forces(true): f and a = f/m
    kStageVerletKick = 2,  // Verlet second half: a = f/m ; v += a dt/2
    kStageVerletKickDrift = 3,  // ... then the next step's drift + half kick
    kStageDampedKick = 4,  // Damped: a = f/m ; v += a dt c2
    kStageDampedKickDrift = 5,
    kStageSums = 6,        // energy / virial / stress only, nothing written
    kStageForceAdd = 7,    // NListed::set_forces: f += pair forces
    kStageNlcg = 8,        // f, a = 0 for fixed atoms, and the sums of nlcg.hpp
};

struct StepCoef {
    // Verlet: dt, dt*dt/2, dt/2.  Damped: c1*dt, c2*dt*dt, dt*(c1-c2), c0, dt*c2
    double k0, k1, k2, k3, k4;
};

// The skin test of the launch before, reduced inside a step launch (one extra
// workgroup) and the test before that, which may have stopped the run: see
// step_gate / reduce_prev in stepcore.hpp.
struct StepGate {
    const double *prev;           // the previous launch's skin partials (fields as ReduceBuf::part)
    int nprev;                    // their number (0: no reduction in this launch)
    const uint32_t *gate;         // or null: flag word of the test one launch earlier
    uint32_t *flag;               // device flag word of this reduction's test
    uint32_t *hflag;              // device-visible pinned word: (seq << kFlagBits) | flags
    uint32_t seq;
};

// A reduced sum as the host reads it, in pinned memory: the value, then the
// number of the reduction that stored it.
struct SumRec {
    double v;
    unsigned long long seq;
};

// Reduction scratch: one partial per workgroup, reduced by k_finalize_sums (and
// k_finalize, k_finalize_skin for a skin test on demand).
struct ReduceBuf {
    double *part;                 // kRedWidth fields x pstride workgroups
    int pstride;                  // field stride (>= workgroups of any launch)
    double *out;                  // kRedWidth doubles (final sums)
    uint32_t *flag;               // flag word
    double skin;                  // skin test threshold
    uint32_t *hflag;              // device-visible pinned host copy of the flag word
    hipEvent_t done;              // host side, or null: recorded on the launch stream right
                                  // after the force kernel, before its sums' reduction (timing)
    uint32_t *cnt;                // or null: the skin-test reduction over several
    double *gpart;                // workgroups (counter, kFinBlocks x 3 results)
    StepGate g;
    SumRec *rec;                  // or null: device-visible pinned records of the sums
    unsigned long long rseq;      // and their number
};
constexpr int kFinBlocks = 32;    // workgroups of the multi-workgroup skin reduction
constexpr int kRedWidth = 16;     // U, W, S[9], contacts, overlaps, top1, top2, nonfinite

// A kick + drift stage leaves its skin-test partials (force_partials of them)
// to the next step launch, whose ReduceBuf::g names them.
hipError_t launch_force(int ndim, int precision, int stage, bool energy,
                        const AtomArrays &A, const ListView &Lv, const PairView &P,
                        const Box &box, const StepCoef &c, const ReduceBuf &R,
                        hipStream_t s);
// Dynamic LDS that the tiled force kernel cannot do without for a stencil of
// smax staged slots (dimension, precision, pair kind, pair types; no pair kind
// yet gets the largest staging).  A pair table in LDS comes on top where it fits.
size_t tiled_force_lds(int ndim, int prec, int kind, int ntypes, int smax);
// The force launches of one dimension, pair kind and precision: over the
// untiled list (force.hip) and the tiled one (step_tiled.hip).
template <int D, int KIND, int PREC>
hipError_t force_part(int stage, bool energy, const AtomArrays &A, const ListView &Lv,
                      const PairView &P, const Box &box, const StepCoef &c,
                      const ReduceBuf &R, hipStream_t s);
template <int D, int KIND, int PREC>
hipError_t force_tiled_part(int stage, const AtomArrays &A, const ListView &Lv,
                            const PairView &P, const Box &box, const StepCoef &c,
                            const ReduceBuf &R, hipStream_t s);
// The sums over nparts workgroup partials (and with top the top-2 fields).
hipError_t launch_finalize_sums(bool top, int nparts, const ReduceBuf &R, hipStream_t s);
// The drift leaves its skin-test partials (reduce_blocks(n) of them) to the
// next step launch; launch_skin with finalize == false does the same.
hipError_t launch_drift(int ndim, int stage, const AtomArrays &A, const StepCoef &c,
                        const ReduceBuf &R, hipStream_t s);
hipError_t launch_skin(int ndim, const AtomArrays &A, const ReduceBuf &R, bool finalize,
                       hipStream_t s);
// Atom observables: mode 0 -> out[0] = K(originv), out[1..D] = momentum,
// out[4] = mass ; mode 1 -> out[0] = sum |f|, out[13] = max |f|.
hipError_t launch_atom_sums(int ndim, int mode, const AtomArrays &A,
                            const double *originv, const ReduceBuf &R, hipStream_t s);
// Layout conversion between the caller's AoS order and the device slots.
// upload: dst component k of slot s = src[orig[s]*ndim + k]  (what: 0 pos,
// 1 v, 2 a, 3 f);  download: the inverse.
hipError_t launch_upload(int ndim, int what, const AtomArrays &A, const int32_t *orig,
                         const double *src, hipStream_t s);
hipError_t launch_download(int ndim, int what, const AtomArrays &A,
                           const int32_t *orig, double *dst, hipStream_t s);
int reduce_blocks(int n);
// Most lanes per atom of an untiled force launch over n atoms, of which the
// autotuner takes as many as pay: up to 2^18 lanes make at most four wavefronts
// per SIMD, which a launch of few atoms otherwise leaves empty while each lane
// walks its chain of list words, gathers and pair forces.  1000 LJ atoms, 200
// steps with 8 / 16 / 32 lanes: 2.13 / 1.69 / 1.47 ms; 10,007 (mixed), 100 steps
// with 8 / 16: 1.48 / 1.27 ms.
constexpr int kWideLanes = 1 << 18;
constexpr int max_lanes(int n) {
    return n <= kWideLanes / 32 ? 32 : (n <= kWideLanes / 16 ? 16 : 8);
}
int force_blocks(int n, int tpa);  // workgroups of a force launch (also partials)
inline int part_blocks(int n) { return force_blocks(n > 1 ? n : 1, max_lanes(n)); }
int force_partials(int n, const ListView &Lv);  // partials of a launch over this list

// ---------------------------------------------------------------- batch.hip
// Geometry of one system of a batch.
struct BatchGeom {
    Box box;
    CellGrid grid;
    int off;       // first atom of the system in the concatenated arrays
    int n;         // atoms
    int cell_off;  // first cell in the concatenated cell-start array
    int pad;
};

struct BatchArrays {
    int ntot;              // atoms over all systems
    const void *pos_in;    // PosStore<D>::T*
    void *pos_out;
    double *v[3], *a[3], *f[3];
    const double *m;
    const int32_t *type;   // pair-table type
    const int32_t *sys;    // system of each atom
    const double *diam;    // list diameter of each atom
    const void *xref;      // positions at each system's last rebuild
    void *xref_w;          // the same buffer, written by the rebuild
    double *disp;          // |x - xref| per atom (skin test input)
    const BatchGeom *geom; // per system
};

// The batched force launches of one dimension, pair kind and precision
// (batch_force.hip).
template <int D, int KIND, int PREC>
void batch_force_part(int stage, bool energy, const BatchArrays &A, const ListView &Lv,
                      const PairView &P, const StepCoef &c, double *eatom, hipStream_t s);
hipError_t launch_batch_force(int ndim, int precision, int stage, bool energy,
                              const BatchArrays &A, const ListView &Lv, const PairView &P,
                              const StepCoef &c, double *eatom, hipStream_t s);
// A worklist (wl): the number of listed systems (high word) and of their build
// slices (low word).  The drift and disp launches empty it, the skin test
// fills it with the systems to rebuild, launch_batch_all with every system.
hipError_t launch_batch_drift(int ndim, bool damped, const BatchArrays &A,
                              const StepCoef &c, unsigned long long *wl, hipStream_t s);
hipError_t launch_batch_disp(int ndim, const BatchArrays &A, unsigned long long *wl,
                             hipStream_t s);
hipError_t launch_batch_skin(int nsys, const BatchArrays &A, double skin, int lanes,
                             unsigned long long *wl, int32_t *work, int32_t *wslice,
                             uint32_t *gflag, hipStream_t s);
hipError_t launch_batch_all(int nsys, const BatchArrays &A, int lanes, unsigned long long *wl,
                            int32_t *work, int32_t *wslice, hipStream_t s);
// Lanes per atom of the list build for a batch of ntot atoms in `cells` cells.
int batch_build_lanes(int ntot, int cells);
// The batch's lists and what their build works on.
struct BatchLists {
    int type_bits, tpa, cap, npad;
    uint32_t *nbr;
    int32_t *ncount;
    int32_t *keys;        // sorted slots: cell,
    uint32_t *ent;        // list word (index << type_bits | type),
    void *xs;             // position
    double *dsort;        // and diameter
    int32_t *cstart;      // each cell's first sorted slot
    uint32_t *which;      // rebuilds per system
    unsigned long long *nent;  // list entries of its last build (twice its pairs)
    int32_t *work, *wslice;    // nsys each: listed systems, their first build slice
    int sort_grid, build_grid;
    int lanes;            // the build's lanes per atom (batch_build_lanes)
    bool sort_only;       // order the slots, build no list
};
// Rebuilds the systems listed in wl: sort, then the list build spread over
// slices of the listed systems; empties wl_next (may be null).  alt: positions
// one step ahead, whose displacements from the new reference positions are
// stored.
hipError_t launch_batch_rebuild(int ndim, const BatchArrays &A, const BatchLists &B,
                                const void *pos, const void *alt, int count_rebuild,
                                double skin, const unsigned long long *wl,
                                unsigned long long *wl_next, uint32_t *gflag, hipStream_t s);
// Every system's slots in the order of its last sort: pos, v, a, m, diam, type
// and orig (the caller's index of each slot) permuted in place, through
// scratch arrays of the batch (pos_alt, stage: ndim doubles per atom, eatom: 4,
// B.xs).  f and the lists are void afterwards.
hipError_t launch_batch_reorder(int ndim, const BatchArrays &A, const BatchLists &B, void *pos,
                                void *pos_alt, double *m, double *diam, int32_t *type,
                                int32_t *orig, double *stage, double *eatom, hipStream_t s);
hipError_t launch_batch_sys_sums(int nsys, const BatchArrays &A, const double *eatom,
                                 double *out, hipStream_t s);
constexpr int kBatchMaxCellsPerSystem = 4096;

// Sets the calling thread's parm_last_error() message; returns code.
int set_error(int code, const std::string &msg);

}  // namespace parm
