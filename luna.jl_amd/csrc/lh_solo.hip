// lh_solo.hip -- the one-workgroup solvers, built without the hoisting of loop
// constants (see build.py), and the choice of one; lh_solo_8192.hip has the one
// that is faster with it.
#include "lh_solo_kernel.h"

bool launch_solo(int cls, int n, const DInst* d, const double2* tw, hipStream_t s, bool zdep, bool raman) {
    if (cls == LH_CLASS_ENV4096) {
        solo_launch<1, 4096, 4096, false, false>(n, d, tw, s);
        return true;
    }
    if (raman) {
        if (cls == LH_CLASS_8192)
            solo_launch<0, 4096, 2048, false, true>(n, d, tw, s);
        else if (cls == LH_CLASS_4096)
            solo_launch<0, 2048, 1024, false, true>(n, d, tw, s);
        else
            return false;
        return true;
    }
    switch (cls) {
        case LH_CLASS_16384: zdep ? solo_launch<0, 8192, 4096, true, false>(n, d, tw, s) : solo_launch<0, 8192, 4096, false, false>(n, d, tw, s); break;
        case LH_CLASS_8192: zdep ? solo_launch<0, 4096, 2048, true, false>(n, d, tw, s) : launch_solo_8192(n, d, tw, s); break;
        case LH_CLASS_4096: zdep ? solo_launch<0, 2048, 1024, true, false>(n, d, tw, s) : solo_launch<0, 2048, 1024, false, false>(n, d, tw, s); break;
        default: return false;
    }
    return true;
}
