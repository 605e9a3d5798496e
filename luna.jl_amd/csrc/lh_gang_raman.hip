// lh_gang_raman.hip -- the gang kernels of the field grids with RamanPolarField,
// kernels of their own: the convolution's transforms are twice as long, and the
// others keep their registers and LDS.
#include "lh_gang.h"

bool lg_raman_solve(const GangLaunch& l, bool stream) {
    switch (l.cls) {
        case LH_CLASS_16384: return lg_launch_solve<0, 8192, true>(l, stream);
        case LH_CLASS_8192: return lg_launch_solve<0, 4096, true>(l, stream);
        case LH_CLASS_4096: return lg_launch_solve<0, 2048, true>(l, stream);
        default: return false;
    }
}

bool lg_raman_rhs(const GangLaunch& l, int* status) {
    switch (l.cls) {
        case LH_CLASS_16384: return lg_launch_rhs<0, 8192, true>(l, status);
        case LH_CLASS_8192: return lg_launch_rhs<0, 4096, true>(l, status);
        case LH_CLASS_4096: return lg_launch_rhs<0, 2048, true>(l, status);
        default: return false;
    }
}
