// lh_solo_8192.hip -- the one-workgroup solver of the constant fill at Nto = 8192,
// a file of its own because it is built with the hoisting of loop constants: it
// fills the 256 registers and spills, and is faster all the same (256 equal
// propagations of 0.2 m 4.61 → 4.27 ms, 512 9.18 → 8.49).  The
// others are not: Nto = 16384 10.8 ms without, 11.0 with; 4096 3.65 both; with a
// Raman response 4096 13.9 without, 14.2 with, 8192 27.5 both; envelope 4096 11.4
// both.
#include "lh_solo_kernel.h"

void launch_solo_8192(int n, const DInst* d, const double2* tw, hipStream_t s) {
    solo_launch<0, 4096, 2048, false, false>(n, d, tw, s);
}
