// The sequential sweeps in one launch each (sweep.hip): DIC's and DILU's factorisation, their forward and
// backward substitution, and Gauss-Seidel, on a plan built with the mesh's level schedule. Each sweep returns
// false, having done nothing, where it belongs to the caller's launch-per-level path: a mesh above kFlowMaxCells or
// of few levels, a plan that does not fit, or a first Gauss-Seidel inside a capture (its walk is laid out by the first one).
#pragma once

#include "mfv_internal.hpp"

namespace mfv {

// lays the mesh's plan out, after its level schedule
void sweepPlan(Ctx& c, Mesh& m);

// A factorisation by sweepFactor (0: by the launch-per-level path). On small meshes it also lays the products
// rD*lower and rD*upper out on the mesh, in the order the substitution reads them, in place of those of the mesh's
// last one; a substitution with a factorisation whose products are not there any more is the caller's. (Captured, a
// substitution goes into the same graph as its factorisation.)
using SweepFactor = unsigned;

// rD = 1/d, d = diag - sum over lower faces (ascending) of upper*lower/d[lower neighbour]
SweepFactor sweepFactor(Ctx& c, Mesh& m, const double* diag, const double* upper, const double* lower, double* rD);
// y = rD*r, forward: y -= rD*lower*y[lower neighbour] over lower faces ascending; backward:
// y -= rD*upper*y[upper neighbour] over owned faces descending
bool sweepSubstitute(Ctx& c, Mesh& m, SweepFactor factor, const double* rD, const double* upper, const double* lower,
                     const double* r, double* y, const int* stop);
// nSweeps Gauss-Seidel sweeps of A psi = b (upper == lower); with bPrime each is followed by
// symGaussSeidel's reverse walk
bool sweepGaussSeidel(Ctx& c, Mesh& m, const double* diag, const double* upper, const double* b, double* psi,
                      int nSweeps, double* bPrime);

} // namespace mfv
