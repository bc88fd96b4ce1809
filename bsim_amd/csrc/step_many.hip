/*
 * step_many.hip -- the step kernel (step.hip) in workgroups of eight wavefronts,
 * four per compute unit, for networks of very many units.
 *
 * With twelve wavefronts a unit ends sooner and two of them fit a compute unit;
 * with eight, four of event and four of owner wavefronts, four units overlap
 * their waits.  The first is better while the launch is as long as its longest
 * units, the second when it is the sum of all units' work.  us per cycle with
 * twelve / with eight, units: sweeps of 180 and 300 chains (2,194 and 3,638
 * units of 192) 34.6 / 24.1 and 53.3 / 34.5, 300 chains (2,730 of 256) 44.4 /
 * 30.1, networks at ~100 Hz of 210,000 neurons (1,094 of 192) 39.1 / 48.5, 330,000
 * (1,719) 54.9 / 63.9, 490,000 (2,553) 77.4 / 78.1, 650,000 (3,386) 97.2 / 86.2;
 * units of 384 (two targets per owner thread), 1,693 at ~100 Hz 98 / 113; rows
 * two at a time need more registers than eight wavefronts per SIMD leave (164 /
 * 482 for 18,000 neurons with delays up to 30 steps).  So: units of at most 256,
 * rows one at a time, from BSIM_MANY_UNITS on.
 *
 * Eight wavefronts per SIMD leave 64 vector registers, all of which are used, and
 * some 80 scalar ones, of which 30 more go to lanes of a vector register.  (The
 * twelve-wavefront kernels need 52, or 68 with two rows, and spill nothing.)  One
 * vector register more went to private memory: 650,000 neurons 86.6 us per cycle
 * so, 86.0 without, 300 chains in units of 192 34.4 / 33.6.
 */
#define NEV 4
#define STEP_EU 8
#define STEP_MANY
#define bsim_step_kernel bsim_step_kernel_many
#include "step.hip"
