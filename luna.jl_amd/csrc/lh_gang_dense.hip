// lh_gang_dense.hip -- the gang solvers for large batches: two workgroups per CU.
// Field grids and envelope grids whose member leaves the LDS for it; the Raman
// response of a field grid and the largest grids do not.
#include "lh_gang.h"

bool lg_has_dense(int cls, bool raman) {
    if (raman) return false;
    return cls == LH_CLASS_16384 || cls == LH_CLASS_8192 || cls == LH_CLASS_4096 || cls == LH_CLASS_ENV8192 ||
           cls == LH_CLASS_ENV4096;
}

bool lg_dense_solve(const GangLaunch& l) {
    switch (l.cls) {
        case LH_CLASS_16384: return lg_launch_dense<0, 8192>(l);
        case LH_CLASS_8192: return lg_launch_dense<0, 4096>(l);
        case LH_CLASS_4096: return lg_launch_dense<0, 2048>(l);
        case LH_CLASS_ENV8192: return lg_launch_dense<1, 8192>(l);
        case LH_CLASS_ENV4096: return lg_launch_dense<1, 4096>(l);
        default: return false;
    }
}
