// lh_solo.h -- the launches of lh_solo.hip and lh_solo_8192.hip.
#pragma once
#include <hip/hip_runtime.h>

struct DInst;

// Solves the n instances d (device memory) of a class, one workgroup each: field
// grids of Nto = 4096, 8192 and 16384 (zdep: all have a z-dependent fill, else
// none), of 4096 and 8192 with a Raman response (raman), the envelope grid of
// 4096 points.  tw: the twiddle table of the single-workgroup transforms.  False:
// no such kernel.
bool launch_solo(int cls, int n, const DInst* d, const double2* tw, hipStream_t s, bool zdep, bool raman);
void launch_solo_8192(int n, const DInst* d, const double2* tw, hipStream_t s);  // constant fill, Nto = 8192
