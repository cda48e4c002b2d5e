// stepctl.h -- what a step's kernels are told about the step, and the part of
// the driver loop they run themselves.
//
// A step needs its dt, and that comes from the CFL minimum of the state the
// previous step left: read on the host, it costs a wait, a copy and the
// launches behind it, about 20 us, more than a small grid's kernel.  In a run
// of several steps (evh_run) the host therefore only launches: the first
// kernel of each step (its head; one of its own where the potential's passes
// come first) forms dt, t and the end of the run as hydrostep, thermalstep and
// updatetime do (timestep.f90:26-57,72-104,147-171), every block from the same
// values and one of them storing the result for the next step.  A step after the end, or after an error, does
// nothing.  128^2 2-D Kelvin-Helmholtz: 31 -> 17 us per step (12 with its
// shorter chunks); 64^3: 62 -> 43 us (30 with them).
//
// Three status blocks take turns: a step reads the limits of the state it
// starts from in one, leaves those of its own new state in the next, and
// clears the third for the step after, so that no launch of its own does.
#pragma once

#include "physics.h"

namespace evh {

// the run at the start of a step; two take turns
struct RunSlot {
  double t, dt;
  double last;  // dt of the last step taken
  int go;    // updatetime's flag: 0 after the step that reaches tend
  int stop;  // no step is taken any more
  int done;  // steps taken
  int why;   // what stopped it (kRun*)
};
enum : int { kRunEnd = 1, kRunCode, kRunNext, kRunDt };

struct StepCtl {
  double dt;           // the step's dt where the host gives it (in == nullptr)
  Status *st;          // takes the step's errors
  Status *lim;         // takes the limits (and next errors) of the new state; nullptr: a later kernel of the step forms them
  const Status *prev;  // the limits and errors of the state the step starts from
  Status *reset;       // cleared for the next step (nullptr: none)
  const RunSlot *in;   // a run on the device: the run so far
  RunSlot *out;        // and after this step
  double tend;
  int head;   // this kernel forms dt; the step's later ones take it from out
  int hydro;  // the step has hydrostep's limit
};

__device__ __forceinline__ void clear_status(Status *s) {
  s->code = 0;
  s->cell = 0;
  s->old_code = 0;
  s->old_cell = 0;
  s->next_code = 0;
  s->next_cell = 0;
  s->vmin_bits = (unsigned long long)__double_as_longlong(1e6);   // timestep.f90:35
  s->tvmin_bits = (unsigned long long)__double_as_longlong(1e99);
}

// The step's dt; false: nothing is to be done.  Called by every lane of every
// block at the start of a step's kernel.
__device__ __forceinline__ bool step_begin(const KParams &P, const StepCtl &C, double &dt) {
  const bool first = blockIdx.x == 0 && threadIdx.x == 0;
  dt = C.dt;
  if (!C.in) {
    if (first && C.reset) clear_status(C.reset);
    if (first && C.prev) {  // errors stay until read, and before those that other blocks report meanwhile
      C.st->old_code = first_code(*C.prev);
      C.st->old_cell = first_cell(*C.prev);
    }
    return true;
  }
  if (!C.head) {
    dt = C.out->dt;
    return !C.out->stop;
  }
  RunSlot s = *C.in;
  if (!s.stop) {
    s.dt = 1e99;  // main.f90:118
    if (!s.go) {
      s.why = kRunEnd;
      s.dt = C.in->dt;
    } else if (first_code(*C.prev)) {
      s.why = kRunCode;
    } else if (C.prev->next_code) {
      s.why = kRunNext;
    } else {
      if (C.hydro) {
        const double c = P.cfl * __longlong_as_double((long long)C.prev->vmin_bits);
        s.dt = c < s.dt ? c : s.dt;
      }
      if (P.conduction && s.dt > 0.0) {
        double v = __longlong_as_double((long long)C.prev->tvmin_bits);
        v = P.c_cond * (P.dx * P.dx) * v / P.temp0;
        s.dt = v < s.dt ? v : s.dt;
      }
      if (s.dt <= 0.0) s.why = kRunDt;
    }
    s.stop = s.why != 0;
  }
  if (s.stop) {
    if (first) *C.out = s;
    return false;
  }
  if (C.tend - s.t <= s.dt) {  // timestep.f90:163-166
    s.dt = C.tend - s.t;
    s.go = 0;
  }
  dt = uniform_value(s.dt);
  if (first) {
    s.t = s.t + s.dt;
    s.last = s.dt;
    s.done += 1;
    *C.out = s;
    clear_status(C.reset);
  }
  return true;
}

}  // namespace evh
