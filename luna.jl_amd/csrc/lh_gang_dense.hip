// lh_gang_dense.hip -- the gang solvers for large batches: two workgroups per CU.
// Field grids whose member leaves the LDS for it.  Not the Raman response of a
// field grid, whose longer transform does not, and not the envelope grids: 256
// propagations of 0.15 m at 8192 points with Raman took 2.42 s on such kernels
// and 2.15 s at one workgroup per CU.
#include "lh_gang.h"

bool lg_has_dense(int cls, bool raman) {
    return !raman && (cls == LH_CLASS_16384 || cls == LH_CLASS_8192 || cls == LH_CLASS_4096);
}

bool lg_dense_solve(const GangLaunch& l) {
    switch (l.cls) {
        case LH_CLASS_16384: return lg_launch_dense<8192>(l);
        case LH_CLASS_8192: return lg_launch_dense<4096>(l);
        case LH_CLASS_4096: return lg_launch_dense<2048>(l);
        default: return false;
    }
}
