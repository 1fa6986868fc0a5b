// The small grids' part of a V-cycle in one launch (cycle_flow.hip).
#pragma once

#include "amg.hpp"
#include "sell_device.hpp"

namespace mfv {

// lays the launch's arrays out for the hierarchy's current precision (after its vectors are allocated)
void flowCycleBuild(Ctx& c, Amg& a);

// whether a cycle's small grids go through it (a.coarseMode aside)
bool flowCycleRuns(const Amg& a, const VcycleControls& vc);

// Runs the cycle from grid a.flowStart to the coarsest and back on that grid's b and x (0 without pre-sweeps). Its
// values go to `up` and, unless null, to `out`, which is not x: rows read their neighbours' x until the end. Needs
// a.flowStart >= 0.
template <typename Tm, typename Tv, typename Ts>
void flowCycle(Ctx& c, Amg& a, const VcycleControls& vc, const Ts* b, const Ts* x, Ts* out, const Scatter<Tv, Ts>& up,
               const int* stop);

} // namespace mfv
