// lh_solo.h -- the launch of lh_solo.hip.
#pragma once
#include <hip/hip_runtime.h>

struct DInst;

// Solves the n instances d (device memory) of a field-grid class (Nto = 4096, 8192
// or 16384, no Raman response), one workgroup each; zdep: all have a z-dependent
// fill (else none).  tw: the twiddle table of the single-workgroup transforms.
void launch_solo(int cls, int n, const DInst* d, const double2* tw, hipStream_t s, bool zdep);
