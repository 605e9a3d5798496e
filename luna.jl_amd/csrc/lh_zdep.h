// lh_zdep.h -- the launch of lh_zdep.hip.
#pragma once
#include <hip/hip_runtime.h>

struct DInst;

// Solves the n instances d (device memory) of a size class, one workgroup each;
// tw: the twiddle table of the single-workgroup transforms.
void launch_zdep(int cls, int n, const DInst* d, const double2* tw, hipStream_t s);
