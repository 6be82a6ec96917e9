// mdk_internal.h -- device data layout shared by the HIP translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mdk_pot.h"

// 3x3 tensors are Fortran column-major: T(i,j) == t[(j-1)*3 + (i-1)].
#define TT(a, i, j) (a)[((j)-1) * 3 + ((i)-1)]

// Box and thermodynamic state of one system, resident on the device, in four
// copies used in turn (mdk_ctx::cur).  A kernel in which every workgroup reads the
// current copy writes its results into later ones: a drift, a predictor and a kick
// with the next drift the advanced box into cur + 1; a kick that also finishes the
// forces the finished box into cur + 1 and the advanced one into cur + 2, which no
// workgroup of that launch reads.  The step's own sums follow in the next density
// pass, into the finished copy and the advanced one: before any later kernel writes
// either again.  Steps in a fixed box between two others of a call stay on one copy.
struct BoxState {
  double b0[9], b1[9], b2[9], b3[9];  // b3: box jolt of the predictor-corrector
  double tk[9], tc[9], tg[9], tp[9], tginv[9], tgdot[9], tgid[9], fb[9];
  double tgid_lag[9];   // tgid seen by the velocity half-kick (quench_m.F90:595)
  double binv[9];       // cofactor(b0)/vol used by update_therm_avs (dynamics_m.F90:692-700)
  double bref[9];       // b0 when the current neighbour list was built (skin bound)
  double vol, pe, pe_emb, ke, s1, s2, s3, te, h, th, boxke;
  double maxdisp2;      // max |B0 (s - s_ref)|^2 since the last full-list build
  double maxstep2;      // max |B0 (x1 + x2)|^2 of the last step (next drift)
  int status;           // MDK_ERR_* raised on the device (singular box)
  int pad_;
};

// Kernel classes for the HIP-event timing accumulators.
enum { TC_DRIFT = 0, TC_DENSITY, TC_FORCE, TC_KICK, TC_REBUILD, TC_NCLASS };

// Per-block partial sums of force() (value-major, one column of a value per
// block): [0] pair energy and [1..6] virial W (xx yy zz xy xz yz) from the
// force pass; the embedding energy from the density pass; kinten's tk
// (column-major, [0..8]) from the kernel that last set the velocities.  In the
// order of their sums: force pass, embedding, kinten.
#define NPART_FORCE 7
#define PART_EMB 7
#define PART_KIN 8
#define NPART_KIN 9
#define NSUM_FORCE (NPART_FORCE + 1 + NPART_KIN)
// Partials of the force pass fused with the kick (fixed boxes): pair energy,
// s3, maxdisp2, maxstep2
#define NPART_FIXED 4
// Partials of the half-kick kernel: s1, s2, s3, maxdisp2, maxstep2
#define NPART_KICK 5

#define MDK_BLOCK 256
