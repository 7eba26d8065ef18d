// mds_clock.h -- the dt policy of one problem's clock, and the clocks of a
// group of folded steps.
//
// A launch of one thread per problem between the steps costs 4 us beside the
// 10 to 20 us a batch of a few columns takes per step.  In a group of
// MDS_FOLD = 4 steps every wavefront of the two-stage column kernels applies
// the policy itself instead: the same operations on the same clock give the
// same dt in all of them, and the wavefront that owns the problem's first
// segment writes the new clock down.  Nothing a launch reads may be written
// by its own wavefronts, so the clocks alternate and the running minima go
// round, step f of the group
//   reads     clock f & 1 (0: DevClock itself, 1: clock2), minimum f
//   writes    clock (f + 1) & 1, folds limits into minimum (f + 1) & 3
//   resets    minimum (f + 2) & 3, whose last readers were step f - 2's
// (minimum 0 is DevClock::mindt).  A group starts and ends with everything in
// DevClock, so whatever else reads a clock finds it there.  The minima start
// at 1e100 and minimum 1 is reset again by a group's last step.
#pragma once
#include "mds_internal.h"
#include "mds_physics.h"

// estimate_dt tail + dt policy (step.c:192-198, main.c:206-251).  The clock
// is advanced here (t += dt, istep++: main.c:263-264) since the stage kernels
// only read dt.  False: the clock stays as it was, but for active and status.
MDS_DEV bool dt_policy(DevClock &c, double md, const RunParams &rp)
{
  if (!c.active) return false;
  if (!(c.t < c.tmax)) { c.active = 0; return false; }
  if (c.istep == 0) md = (md < rp.initial_dt) ? md : rp.initial_dt;
  md = (md < rp.dtmax) ? md : rp.dtmax;
  md *= rp.cfl;
  double dt = md;
  if (dt < rp.dtmin) { c.status = 1; c.active = 0; return false; }
  if (c.istep == 0) dt *= rp.dt_init_safety;
  else { double g = c.dtold * rp.dt_grow_safety; dt = (g < dt) ? g : dt; }
  c.dtold = dt;
  if (c.t + 1 * dt > c.tmax) dt = (1.000000001 * (c.tmax - c.t)) / 1;
  if (dt < rp.dtmin) dt = rp.dtmin;
  c.dt = dt;
  // the reference's second-stage fill adds dt to the global t and takes it
  // off again (bc.c:717-721, 1417), then the main loop adds dt (main.c:263)
  c.t = ((c.t + dt) - dt) + dt;
  c.istep += 1;
  return true;
}

// The clock of problem p in a launch of the two-stage column kernels: dt and
// whether it steps, and the minimum its limits fold into.  first: this
// wavefront owns the problem's first segment.
struct StepClock {
  double dt;
  bool active;
  unsigned long long *mindt;
};
template <bool FOLD>
MDS_DEV StepClock step_clock(const Sweep1DArgs &a, int p, bool first)
{
  StepClock s;
  DevClock *ck = &a.clock[p];
  if constexpr (!FOLD) {
    s.dt = ck->dt;
    s.active = ck->active != 0;
    s.mindt = &ck->mindt;
    return s;
  } else {
    const int f = a.fold;
    unsigned long long *mind = a.mind + (size_t)p * MDS_FOLD;
    auto minimum = [&](int k) { return (k & (MDS_FOLD - 1)) == 0 ? &ck->mindt : mind + (k & (MDS_FOLD - 1)); };
    DevClock c = (f & 1) ? a.clock2[p] : *ck;
    const unsigned long long key = *minimum(f);
    dt_policy(c, __longlong_as_double((long long)key), a.rp);
    s.dt = c.dt;
    s.active = c.active != 0;
    s.mindt = minimum(f + 1);
    if (first && (threadIdx.x & 63) == 0) {
      DevClock *o = (f & 1) ? ck : &a.clock2[p];
      o->t = c.t;
      o->dt = c.dt;
      o->dtold = c.dtold;
      o->tmax = c.tmax;
      o->istep = c.istep;
      o->active = c.active;
      o->status = c.status;
      *minimum(f + 2) = dt_key(1.0e100);
    }
    return s;
  }
}
