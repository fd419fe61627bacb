// When the host may launch an Arnoldi step before it has read the flags of the one
// before (host only, no HIP).
//
// A step launched ahead keeps the queue full: reading the flags first leaves the GPU
// idle 15-20 us (129 x 129, one RHS: 80 us a step).  Past the last step it is a chain
// of launches that find every flag set: 40 us there, 100 us for a W cycle of six
// levels or a K-cycle.  So the host waits where the step may be the last: when the
// largest residual estimate, carried a step and a half on at the better of the solve's
// mean rate and its last step's, meets the tolerance, and while no step's estimate is
// known.  (Half a step for uneven convergence: a needless wait costs less than a chain.)
// Whole solves on MI355X in us, always ahead / always waiting / this rule (the span of
// two processes each): 1025 x 513 to 0.5 (one step) 631-639 / 525-533 / 511-525, K-cycle
// 257 x 129 x 4 RHS to 0.1 (two steps) 1125-1139 / 1016-1023 / 988-1026, 129 x 129 to
// 1e-6 (104 steps) 6420-6550 / 7360-7380 / 6080-6440.
#pragma once
#include <algorithm>
#include <cmath>

namespace hh {

struct StepAhead {
  double tol;
  double worst = 1.0;  // largest known ||r|| / ||b|| over the RHS still iterating (x = 0 at first)
  double last = 1.0;   // its last change
  int steps = 0;       // steps whose estimates are known

  explicit StepAhead(double tolerance) : tol(tolerance) {}
  // the true residual that a restart cycle begins with
  void restart(double residual) { worst = residual; }
  // the largest estimate of the next step
  void step(double estimate) {
    last = estimate / worst;
    worst = estimate;
    ++steps;
  }
  // whether the step after the last known one may meet the tolerance (NaN: no)
  bool may_end() const {
    if (steps == 0) return true;
    return worst * std::pow(std::min(last, std::pow(worst, 1.0 / steps)), 1.5) <= tol;
  }
};

}  // namespace hh
