// lh_gang_launch.h -- launches of the gang kernels (lh_gang.h) and the memory
// they need.
#pragma once
#include <hip/hip_runtime.h>
#include <string.h>

#include "../../include/luna_hip.h"
#include "lh_gang_proto.h"

struct DInst;

static constexpr int LG_TWN = 32768;         // twiddle table: exp(-2πi m/LG_TWN)
static constexpr int LG_MIN_WG = 32;         // workgroups of the smallest launch
static constexpr int LG_SLOTS = 14;          // vectors of an instance's work block, see LgVec

// Complex points of a transform and the work block of a mode-averaged class.
static inline int lg_points(const lh_desc& d) { return d.grid_kind == LH_GRID_REAL ? d.n_to / 2 : d.n_to; }
static inline size_t lg_stride(const lh_desc& d) {  // one vector of the work block
    const int M = lg_points(d);
    return (size_t)LG_G * ((d.grid_kind == LH_GRID_REAL ? M / 8 : M / 4) + 8);
}
static inline size_t lg_exchange_len(const lh_desc& d) {  // one exchange series
    return (size_t)lg_points(d) * ((d.grid_kind == LH_GRID_REAL && d.raman) ? 2 : 1);
}
static inline size_t lg_area_len(const lh_desc& d) {  // complex points of the exchange area
    return 2 * lg_exchange_len(d) + 256 + (size_t)lg_points(d) / 2;
}

// Workgroups of a launch over n jobs: whole gangs in equal numbers on the eight
// XCDs, at most one workgroup per CU, two of a dense kernel.
static constexpr int LG_MAX_WG = 256;        // one workgroup per CU
static inline int lg_workgroups(int n, bool dense) {
    const int want = (LG_G * n + LG_MIN_WG - 1) / LG_MIN_WG * LG_MIN_WG, most = (dense ? 2 : 1) * LG_MAX_WG;
    return want < most ? want : most;
}
// Instances in a batch above which it runs on dense kernels, where a class has
// one.  A gang on half the registers and half a CU per member takes 1.6 times as
// long for a step, two of them do 1.25 times as much: better once there are two
// to three instances for each of the 64 gangs, before that the longest instance
// decides.  ms for n propagations of 0.4 m (half Nto = 8192, half 16384), one
// workgroup per CU / two: 128 23.2/29.0, 160 27.7/29.7, 192 34.4/30.3, 224
// 38.8/33.2, 256 44.6/40.0; 384 of 0.2 m 35.3/34.0.
static constexpr int LG_DENSE_ABOVE = 176;
static inline void lg_ctl_init(void* p, int njobs, int nwg, const unsigned* beat) {
    memset(p, 0, lg_ctl_bytes(njobs, nwg));
    GangCtl* c = (GangCtl*)p;
    c->njobs = (unsigned)njobs;
    c->n_wg = (unsigned)nwg;
    c->beat = beat;
}

// Launches of a class over the instances d (job i is d[i]; device memory for a
// solve, host memory for a single right-hand side or record, whose instance
// travels with the launch), control block ctl (lg_ctl_init) and the gangs'
// twiddle table tw.  False: no such kernel.
struct GangLaunch {
    int cls, nwg;
    GangCtl* ctl;
    const DInst* d;
    const double2* tw;
    hipStream_t s;
};
bool lg_field_solve(const GangLaunch& l, bool stream);
bool lg_has_dense(int cls, bool raman);
bool lg_dense_solve(const GangLaunch& l);
bool lg_field_rhs(const GangLaunch& l, int* status);
bool lg_field_stats(const GangLaunch& l, double z, double dz, int* status);
bool lg_raman_solve(const GangLaunch& l, bool stream);  // field grids with a Raman response
bool lg_raman_rhs(const GangLaunch& l, int* status);
bool lg_env_solve(const GangLaunch& l, bool stream);
bool lg_env_rhs(const GangLaunch& l, int* status);
bool lg_env_stats(const GangLaunch& l, double z, double dz, int* status);
