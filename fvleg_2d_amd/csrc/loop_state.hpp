// Bookkeeping of the device-resident time loop (main.f90:138-198): the error
// codes, the choice of dt and the step update, run by whichever kernel closes a
// step.
#pragma once

#include "physics.hpp"

namespace cato {

// Error code of error.f90:6-9 from the OR of sanity flags.
__device__ inline int err_code(int flags) {
  if (flags & 1) return 3;  // NANS_FOUND
  if (flags & 2) return 1;  // NEG_DENSITY
  if (flags & 4) return 2;  // NEG_PRESSURE
  return 0;
}

// dt of the next step (main.f90:140-158): the startup period's dt, else a
// constant dt or the given first dt, else the CFL minimum m.
__device__ inline double chosen_dt(const LoopState *L, double m) {
  if (L->startup) return (L->time <= L->startup_period) ? L->startup_dt : m;
  if (L->constant_dt > 0.0) return L->constant_dt;
  if (L->iter0 + L->iteration == 0 && L->initial_dt > 0.0) return L->initial_dt;
  return m;
}

// With exact landing, no step carries the state's time past the next contour
// time or max_time.  The loop moves next_output_time on one step after the
// time reached it, so a time already on it aims at the one after.
__device__ inline double next_dt(const LoopState *L, double m) {
  double d = chosen_dt(L, m);
  if (L->exact) {
    double out = L->next_output_time;
    if (!(out - L->master_time > 0.0)) out = out + L->contour_dt;
    const double to_out = out - L->master_time;
    const double to_end = L->max_time - L->master_time;
    if (to_out > 0.0 && d > to_out) d = to_out;
    if (to_end > 0.0 && d > to_end) d = to_end;
  }
  return d;
}

// Time-loop bookkeeping after a reduction of CFL minimum m and sanity flags e.
// mode 1: initialise (first dt); mode 2: end of a step of main.f90:138-198
// (master%time += dt; contour cadence; dt clip of the driver time).
__device__ inline void loop_update(LoopState *L, double m, int e, int mode) {
  if (mode == 1) {
    L->dt = next_dt(L, m);
    if (!(L->time < L->max_time && L->iteration < L->max_iterations)) L->done = 1;
  } else if (mode == 2) {
    const double EPS = Lim<double>::eps;
    L->master_time = L->master_time + L->dt;
    double new_time = L->master_time;
    if (absd(L->time - L->next_output_time) < EPS) L->next_output_time = L->next_output_time + L->contour_dt;
    if (new_time > L->next_output_time) {
      double delta_t = absd(L->next_output_time - L->time);
      new_time = L->time + delta_t;
    }
    L->time = new_time;
    L->iteration = L->iteration + 1;
    int code = err_code(e);
    if (code) {
      L->error = code;
      L->done = 1;
    }
    L->dt = next_dt(L, m);
    if (!(L->time < L->max_time && L->iteration < L->max_iterations)) L->done = 1;
  }
}

}  // namespace cato
