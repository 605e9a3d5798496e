// lh_gang_env.hip -- the gang kernels of the envelope grids (Kerr, Raman).
#include "lh_gang.h"

bool lg_env_solve(const GangLaunch& l, bool stream) {
    switch (l.cls) {
        case LH_CLASS_ENV16384: return lg_launch_solve<1, 16384, false>(l, stream);
        case LH_CLASS_ENV8192: return lg_launch_solve<1, 8192, false>(l, stream);
        case LH_CLASS_ENV4096: return lg_launch_solve<1, 4096, false>(l, stream);
        default: return false;
    }
}

bool lg_env_rhs(const GangLaunch& l, int* status) {
    switch (l.cls) {
        case LH_CLASS_ENV16384: return lg_launch_rhs<1, 16384, false>(l, status);
        case LH_CLASS_ENV8192: return lg_launch_rhs<1, 8192, false>(l, status);
        case LH_CLASS_ENV4096: return lg_launch_rhs<1, 4096, false>(l, status);
        default: return false;
    }
}

bool lg_env_stats(const GangLaunch& l, double z, double dz, int* status) {
    switch (l.cls) {
        case LH_CLASS_ENV8192: return lg_launch_stats<1, 8192>(l, z, dz, status);
        case LH_CLASS_ENV4096: return lg_launch_stats<1, 4096>(l, z, dz, status);
        default: return false;
    }
}
