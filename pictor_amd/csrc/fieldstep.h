// fieldstep.h -- types and launchers of the fused field step (kernels_fieldstep.hip).
#pragma once
#include "pictor_common.h"

namespace pictor {

// Lehe coefficients in the field precision (em_update_lehe.F90:8-25), launch_update_b_half_lehe's order
template <typename R>
struct LeheP {
    R ax, ay, az, bxy, bxz, byx, byz, bzx, bzy, dx, dy, dz;
};

template <typename R>
struct FieldC {
    R hc, fc, idx, idy, idz;
    double dfc, dix, diy, diz, jscale;   // the split form updates its E pair in FP64
    LeheP<R> L;
};

// one step's field work; E, B (and the split form's low part L of E) with their ghosts filled
template <typename R>
struct FieldStepP {
    const R *E[3], *B[3];
    const float *L[3];
    const double *J[3];
    R *En[3], *Bn[3];
    float *Ln[3];
    double *Jz[3];     // current to clear (null: none)
    int fold;          // 1: J is as deposited, its ghost layers are added as it is read
    int next;          // 1: B goes on by the next step's first half step
    Gate gate;
    int *host;         // pinned {spill count, error bits, stop step}, written when set
    const int *spill, *err;
};

// E' and B' from E, B and J (kernels_fieldstep.hip): 2-D, and 3-D with the Yee update
template <typename R>
void launch_field_step(const GridP &g, const PhysP &ph, double jscale, const FieldStepP<R> &P, hipStream_t s);
// a B half step B -> Bn (the same array or another), clearing Jz; and E, J -> En in place
template <typename R>
void launch_field_b(const GridP &g, const PhysP &ph, const FieldStepP<R> &P, hipStream_t s);
template <typename R>
void launch_field_e(const GridP &g, const PhysP &ph, double jscale, const FieldStepP<R> &P, hipStream_t s);

}  // namespace pictor
