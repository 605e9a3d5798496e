// lh_gang_field.hip -- the gang kernels of the field grids (Kerr, PPT plasma).
#include "lh_gang.h"

bool lg_field_solve(const GangLaunch& l, bool stream) {
    switch (l.cls) {
        case LH_CLASS_32768: return lg_launch_solve<0, 16384, false>(l, stream);
        case LH_CLASS_16384: return lg_launch_solve<0, 8192, false>(l, stream);
        case LH_CLASS_8192: return lg_launch_solve<0, 4096, false>(l, stream);
        case LH_CLASS_4096: return lg_launch_solve<0, 2048, false>(l, stream);
        default: return false;
    }
}

bool lg_field_rhs(const GangLaunch& l, int* status) {
    switch (l.cls) {
        case LH_CLASS_32768: return lg_launch_rhs<0, 16384, false>(l, status);
        case LH_CLASS_16384: return lg_launch_rhs<0, 8192, false>(l, status);
        case LH_CLASS_8192: return lg_launch_rhs<0, 4096, false>(l, status);
        case LH_CLASS_4096: return lg_launch_rhs<0, 2048, false>(l, status);
        default: return false;
    }
}

bool lg_field_stats(const GangLaunch& l, double z, double dz, int* status) {
    switch (l.cls) {
        case LH_CLASS_16384: return lg_launch_stats<0, 8192>(l, z, dz, status);
        case LH_CLASS_8192: return lg_launch_stats<0, 4096>(l, z, dz, status);
        case LH_CLASS_4096: return lg_launch_stats<0, 2048>(l, z, dz, status);
        default: return false;
    }
}
