// nlcg.hpp -- launchers of the device passes of the nonlinear
// conjugate-gradient minimiser (nlcg.hip).
#pragma once

#include "kernels.hpp"

namespace parm {

// The assignment a k_nlcg_vec pass applies before its sums.
enum NlcgOp : int {
    kNlcgDots = 0,      // none
    kNlcgAssignAV = 1,  // a = v = f (fixed atoms: 0)
    kNlcgConjugate = 2, // a = f, v = a + v * beta (fixed atoms: 0)
    kNlcgDescend = 3,   // a = v = f for atoms that are not fixed
};

// Output fields (ReduceBuf out[]) of a k_nlcg_vec pass: sums over atoms with a
// finite positive mass.  A kStageNlcg force launch gives the first four and the
// virial.
constexpr int kNlcgFF = 0, kNlcgFA = 1, kNlcgFV = 2, kNlcgVV = 3, kNlcgKin = 4, kNlcgW = 5;

// x <- x * lfac[k] + v * dx (per dimension k), every atom.
hipError_t launch_nlcg_stepx(int ndim, const AtomArrays &A, const double *lfac, double dx,
                             hipStream_t s);
// The assignment `op`, then with sums the fields into R.out and R.rec (lfac
// scales x in field 4).
hipError_t launch_nlcg_vec(int ndim, int op, const AtomArrays &A, double beta,
                           const double *lfac, bool sums, const ReduceBuf &R, hipStream_t s);

}  // namespace parm
