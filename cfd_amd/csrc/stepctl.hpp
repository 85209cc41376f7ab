// Step control (ns2DComp.ALE.f90:142-166, meshMove.f90:55-70): DTMIN from the
// minimum of deltat's element values, the 1 % hysteresis against DTMIN1, the
// clock, the local-time-step blend factor and the body's rotation increment for
// TRANSF.  BANDERA's increment after fluidStructure (ns2DComp.ALE.f90:250) is
// applied here too: nothing in between reads it.
#pragma once

#include "cfd_internal.hpp"

namespace cfd {

struct StepLaw {
    int itlocal, motion;
    double amp, omega;
};

// The hysteresis alone: dtmin (in: the elements' minimum) and the next
// DTMIN1 and BANDERA (in: the last ones)
__device__ __forceinline__ void step_dtmin(double& dtmin, double& dtmin1, double& bandera) {
    if ((int)bandera == 1) {
        dtmin1 = dtmin;
        bandera = 2.0;
    }
    const double porc = fabs((dtmin - dtmin1) / dtmin);
    if (100.0 * porc <= 1.0) {
        dtmin = dtmin1;
    } else {
        dtmin1 = dtmin;
        bandera = 2.0;
    }
}

// One thread: the step's scalars from the minimum m and the last DTMIN1, BANDERA
__device__ __forceinline__ void step_control(double* ctl, double m, double dtmin1, double bandera,
                                             const StepLaw& law) {
    double dtmin = m;
    ctl[X_RAW] = dtmin;
    const double iter = ctl[CFD_S_ITER] + 1.0;
    ctl[CFD_S_ITER] = iter;
    step_dtmin(dtmin, dtmin1, bandera);
    ctl[CFD_S_DTMIN1] = dtmin1;
    ctl[CFD_S_BANDERA] = bandera + 1.0;
    ctl[CFD_S_DTMIN] = dtmin;
    ctl[X_FDTL] = law.itlocal != 0 ? 1.0 - exp(-iter * 4.6 / law.itlocal) : 1.0;
    const double time = ctl[CFD_S_TIME] + dtmin;
    ctl[CFD_S_TIME] = time;
    // meshMove.f90:55-57,70: ampli*sin(10 t), ampli = pi/8 (motion 0)
    const double pi = 3.141592653589793;
    const double ang = law.motion == 1 ? law.amp * sin(law.omega * time) : pi / 8.0 * sin(10.0 * time);
    const double alpha = ang - ctl[CFD_S_DISN2];
    ctl[CFD_S_DISN2] = ang;
    ctl[X_CA] = cos(alpha);
    ctl[X_SA] = sin(alpha);
}

}  // namespace cfd
