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

static constexpr int LG_LOST = 2;  // LH_E_HIP: a member that others wait for has not come

// The status of one member at barrier ep: what its flag carries once it has
// arrived; LG_LOST where it has not within the polls, or has given up itself
// (its flag may then stay behind).  One test and one branch per poll: the loop
// lies on every wait (with a branch per condition a right-hand side at
// Nto = 4096 takes 7.1 µs instead of 6.2).
template <class Mem>
__device__ __forceinline__ int lg_await(const unsigned* flag, unsigned ep, int polls) {
    unsigned v;
    bool again;
    do {
        v = Mem::ld(flag);
        again = lg_behind(v, ep) & ((v & 15u) != (unsigned)LG_LOST) & (--polls > 0);
    } while (again);
    return lg_behind(v, ep) ? LG_LOST : (int)(v & 15u);
}

// Control block of one launch.
struct GangCtl {
    unsigned next_job, njobs, n_wg, left;
    const unsigned* beat;  // a word that every solver on the device changes as it gets on, or null
    unsigned pad[10];
    unsigned ticket[LG_XCC];
    // then per job LG_G flags (LG_FLAG_STRIDE apart), then mail[LG_XCC][n_wg / LG_G] (64-bit)
};
__host__ __device__ constexpr size_t lg_flags_off() { return sizeof(GangCtl); }
__host__ __device__ constexpr size_t lg_mail_off(size_t njobs) {
    return sizeof(GangCtl) + njobs * LG_G * LG_FLAG_STRIDE * sizeof(unsigned);
}
__host__ __device__ constexpr size_t lg_ctl_bytes(size_t njobs, size_t n_wg) {
    return lg_mail_off(njobs) + LG_XCC * (n_wg / LG_G) * sizeof(unsigned long long);
}

// A gang's mailbox holds sequence << 32 | job: 0 until the gang is complete,
// then sequence 1, then one message per job with sequences 2, 3, ...
static constexpr unsigned LG_NONE = 0xffffffffu;             // as a job: no more
static constexpr unsigned long long LG_FORMED = 1ull << 32 | 0xfffffffeull;
static constexpr unsigned long long LG_GONE = ~0ull;         // a member has left before the gang was complete

// The next job of a workgroup (LG_NONE: leave), after seq − 1 jobs.  The last
// member to arrive completes the gang and leads it: it takes jobs from the
// launch's counter and posts them.  lost: the last job ended with LG_LOST; such
// a gang takes no more.
//
// No wait here is without an end.  A workgroup whose gang is never completed
// leaves once every job has been taken (it reads the counter first and the
// mailbox after it, and the leader forms the gang before it takes a job), or
// after max_poll polls during which nothing on the device got on: the places on
// its XCD may be held by other work, which is worth waiting for, or may not
// exist (a stream restricted to few CUs; launches that hold each other's
// places).  It then marks the mailbox, so that no gang counts on it.  Jobs that
// nobody takes keep the status the host gave them.
template <class Mem>
__device__ __forceinline__ unsigned lg_next_job(GangCtl* ctl, unsigned long long* mail, int member, unsigned seq,
                                                bool lost, unsigned njobs, int max_poll) {
    if (member == LG_G - 1) {
        if (seq == 1 && Mem::cas(mail, 0ull, LG_FORMED) != 0ull) return LG_NONE;
        unsigned job = lost ? LG_NONE : Mem::add(&ctl->next_job, 1u);
        if (job >= njobs) job = LG_NONE;
        Mem::st(mail, (unsigned long long)(seq + 1) << 32 | job);
        return job;
    }
    if (lost) return LG_NONE;
    const unsigned* beat = ctl->beat;
    unsigned last = 0;
    for (int it = 0;;) {
        const unsigned taken = Mem::ld(&ctl->next_job), now = beat ? Mem::ld(beat) : 0u;
        Mem::drain();
        const unsigned long long m = Mem::ld(mail);
        const unsigned s = (unsigned)(m >> 32);
        if (s > seq) return s == seq + 1 ? (unsigned)m : LG_NONE;  // a later one: the gang went on without this member
        if (m == 0ull) {
            if (taken >= njobs) return LG_NONE;
            if (now != last) it = 0;
            last = now;
        }
        if (++it >= max_poll) {
            if (m != 0ull || Mem::cas(mail, 0ull, LG_GONE) == 0ull) return LG_NONE;
            it = 0;
        }
        Mem::pause();
    }
}

// What a workgroup adds to GangCtl::left as it leaves a launch of one job: one,
// its status, and whether the job was taken.  The status of the launch follows
// from the sum of all: LG_LOST if the job was not taken or any member lost
// another, else member 0's.
__device__ __forceinline__ unsigned lg_leave(int member, unsigned jobs, int status) {
    return 1u | (jobs ? (unsigned)(status & 15) << (8 + 4 * member) : 0u) |
           (jobs && member == LG_G - 1 ? 1u << 24 : 0u);
}
__device__ __forceinline__ int lg_left(unsigned sum) {
    int status = (int)(sum >> 8 & 15u);
    for (int m = 1; m < LG_G; m++)
        if ((int)(sum >> (8 + 4 * m) & 15u) == LG_LOST) status = LG_LOST;
    return sum >> 24 & 1u ? status : LG_LOST;
}
