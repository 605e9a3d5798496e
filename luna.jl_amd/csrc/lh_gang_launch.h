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
// Instances of the classes that have one above which a batch runs on dense
// kernels.  A gang on half the registers and half a CU per member takes 1.6
// times as long for a step, two of them do 1.25 times as much: better once 64
// gangs would take a third round, before that the longest instance decides.  ms,
// one workgroup per CU / two, energies and pressures at random, Nto = 8192: 96
// 7.6/8.3, 128 9.2/8.7, 144 11.0/9.2, 160 11.5/10.0, 192 12.8/12.4, 256 16.8/14.8;
// 16384: 96 10.0/11.7, 128 12.3/12.8, 144 15.2/13.7, 160 16.0/15.0, 192 17.5/17.1,
// 256 23.0/20.3; both: 128 11.0/12.2, 160 13.9/13.3, 192 15.7/13.9, 256 18.9/17.2.
static constexpr int LG_DENSE_ABOVE = 128;
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
