// lh_gang_proto.h -- how the workgroups of a gang launch find and wait for each
// other: tickets, the mailbox of a gang, the flags of its barrier.  The memory
// operations are a parameter (Mem: ld, st, add, cas, drain, pause), so the same
// source runs on the host under threads (tests/test_gang_protocol.py).
#pragma once
#include <stddef.h>

static constexpr int LG_G = 4;               // members of a gang
static constexpr int LG_XCC = 16;            // values of HW_REG_XCC_ID
static constexpr int LG_FLAG_STRIDE = 32;    // unsigneds between two members' flags (one cache line)

// A member's flag: the barrier it has reached and its error status.
__device__ __forceinline__ unsigned lg_flag(unsigned ep, int status) { return ep << 4 | (unsigned)(status & 15); }
// Whether a member whose flag is v has yet to reach barrier ep.  A flag has 28
// bits of the epoch, so the difference is taken modulo 2^28 (modulo 2^32 above
// the status): right for any number of barriers while two members are less
// than 2^27 apart, and a barrier lets them be one apart.
__device__ __forceinline__ bool lg_behind(unsigned v, unsigned ep) { return (int)((v & ~15u) - (ep << 4)) < 0; }
