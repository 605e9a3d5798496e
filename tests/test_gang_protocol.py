"""The protocol of the gangs' workgroups (lh_gang_proto.h), compiled for the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "luna.jl_amd", "csrc")


def build(tmp_path, body):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text("#define __device__\n#define __host__\n#define __forceinline__ inline\n#include <stdio.h>\n"
                   "#include \"lh_gang_proto.h\"\n" + body)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-pthread", "-I" + CSRC, str(src), "-o", str(exe)], check=True)
    return str(exe)


EPOCHS = r"""
int main() {
    // epochs counted in 64 bits around every point where a flag or the 32-bit
    // count wraps, members up to 3 apart, every status
    const unsigned long long at[] = {4, 1ull << 27, 1ull << 28, 3ull << 28, 1ull << 32, 5ull << 32};
    int bad = 0;
    for (unsigned long long a : at)
        for (unsigned long long mine = a - 4; mine <= a + 4; mine++)
            for (unsigned long long other = mine < 3 ? 0 : mine - 3; other <= mine + 3; other++)
                for (int st = 0; st < 16; st++)
                    if (lg_behind(lg_flag((unsigned)other, st), (unsigned)mine) != (other < mine)) {
                        if (bad++ == 0) printf("mine %llu other %llu status %d\n", mine, other, st);
                    } else if ((lg_flag((unsigned)other, st) & 15) != (unsigned)st)
                        bad++;
    return bad != 0;
}
"""


def test_barrier_epochs_wrap(tmp_path):
    r = subprocess.run([build(tmp_path, EPOCHS)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


# A launch on the host: a workgroup is a thread, its members' work a series that
# every barrier exchanges.  wait(h, job, barrier) lets a member come late.
MODEL = r"""

#include "lh_gang_proto.h"
#include <algorithm>
#include <atomic>
#include <chrono>
#include <functional>
#include <thread>
#include <vector>

struct HostMem {
    template <class T> static T ld(const T* p) {  // polls give way, so that a limit in polls is one in time
        thread_local unsigned n = 0;
        if (++n % 32 == 0) std::this_thread::sleep_for(std::chrono::microseconds(50));
        return __atomic_load_n(p, __ATOMIC_SEQ_CST);
    }
    static void st(unsigned long long* p, unsigned long long v) { __atomic_store_n(p, v, __ATOMIC_SEQ_CST); }
    static void st(unsigned* p, unsigned v) { __atomic_store_n(p, v, __ATOMIC_SEQ_CST); }
    static unsigned add(unsigned* p, unsigned v) { return __atomic_fetch_add(p, v, __ATOMIC_SEQ_CST); }
    static unsigned long long cas(unsigned long long* p, unsigned long long old, unsigned long long v) {
        __atomic_compare_exchange_n(p, &old, v, false, __ATOMIC_SEQ_CST, __ATOMIC_SEQ_CST);
        return old;
    }
    static void drain() {}
    static void pause() { std::this_thread::yield(); }
};

static const int POLLS = 64000, BARRIERS = 40;  // 2000 naps of 50 µs or more
struct Launch {
    std::vector<unsigned long long> block;
    GangCtl* ctl;
    std::vector<std::vector<long>> x;  // [job][member]: the series
    std::vector<int> status, lost_in, wrong, runs;
    int launch_status = -1;
    unsigned beat = 0;
    std::atomic<int> lost{0};          // members that count another one as lost
    std::function<void(int, int, int)> wait = [](int, int, int) {};
    std::function<void(int)> arrive = [](int) {};  // before workgroup i takes a ticket
    Launch(int njobs, int nwg) : block(lg_ctl_bytes(njobs, nwg) / 8 + 1), x(njobs, std::vector<long>(LG_G)),
                                 status(njobs, LG_LOST), lost_in(njobs), wrong(njobs), runs(njobs) {
        ctl = (GangCtl*)block.data();
        ctl->njobs = njobs;
        ctl->n_wg = nwg;
        ctl->beat = &beat;
    }
    bool sync(unsigned* flags, int h, unsigned& ep, int& flag, int& gflag) {
        ep++;
        HostMem::st(flags + LG_FLAG_STRIDE * h, lg_flag(ep, flag));
        int st[LG_G];
        for (int t = 0; t < LG_G; t++) st[t] = lg_await<HostMem>(flags + LG_FLAG_STRIDE * t, ep, gflag == LG_LOST ? 1 : POLLS);
        for (int t = 0; t < LG_G; t++)
            if (st[t] == LG_LOST) {
                if (gflag != LG_LOST) lost++;
                flag = gflag = LG_LOST;
            }
        if (gflag == LG_LOST) HostMem::st(flags + LG_FLAG_STRIDE * h, lg_flag(ep, LG_LOST));
        return gflag == 0;
    }
    void group(int i, int xcc) {  // as gang_loop and g_solve
        arrive(i);
        const unsigned tk = HostMem::add(&ctl->ticket[xcc], 1u);
        const int h = tk % LG_G;
        unsigned long long* mail = (unsigned long long*)((char*)ctl + lg_mail_off(ctl->njobs)) + xcc * (ctl->n_wg / LG_G) + tk / LG_G;
        unsigned seq = 1;
        int gflag = 0;
        for (;;) {
            const int job = (int)lg_next_job<HostMem>(ctl, mail, h, seq, gflag == LG_LOST, ctl->njobs, POLLS);
            if (job < 0) break;
            seq++;
            unsigned* flags = (unsigned*)((char*)ctl + lg_flags_off()) + (size_t)job * LG_G * LG_FLAG_STRIDE;
            unsigned ep = 0;
            int flag = gflag = 0;
            __atomic_fetch_add(&runs[job], 1, __ATOMIC_SEQ_CST);
            for (int b = 1; b <= BARRIERS && gflag == 0; b++) {
                wait(h, job, b);
                __atomic_store_n(&x[job][h], (long)b, __ATOMIC_SEQ_CST);
                if (!sync(flags, h, ep, flag, gflag)) break;
                for (int m = 0; m < LG_G; m++) {
                    const long v = __atomic_load_n(&x[job][m], __ATOMIC_SEQ_CST);
                    if (v < b || v > b + 1) wrong[job] = 1;
                }
                __atomic_fetch_add(&beat, 1, __ATOMIC_SEQ_CST);
            }
            if (gflag == LG_LOST) __atomic_store_n(&lost_in[job], 1, __ATOMIC_SEQ_CST);
            if (h == 0) status[job] = gflag;
        }
        if (ctl->njobs == 1) {
            const unsigned mine = lg_leave(h, seq - 1, gflag), sum = HostMem::add(&ctl->left, mine) + mine;
            if ((sum & 255u) == ctl->n_wg) launch_status = lg_left(sum);
        }
    }
    void run(const std::vector<int>& xcc) {
        std::vector<std::thread> th;
        for (size_t i = 0; i < xcc.size(); i++) th.emplace_back([this, i, &xcc] { group((int)i, xcc[i]); });
        for (auto& t : th) t.join();
        for (size_t j = 0; j < status.size(); j++)
            if (lost_in[j]) status[j] = LG_LOST;
    }
};
static std::vector<int> spread(int nwg, int nx) {
    std::vector<int> v;
    for (int i = 0; i < nwg; i++) v.push_back(i % nx);
    return v;
}
static void ms(int n) { std::this_thread::sleep_for(std::chrono::milliseconds(n)); }
static int failures = 0;
#define CHECK(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); failures++; } } while (0)

int main() {
    {   // every job once, by four members, in order
        Launch l(20, 32);
        l.run(spread(32, 8));
        for (int j = 0; j < 20; j++) CHECK(l.status[j] == 0 && !l.wrong[j] && l.runs[j] == LG_G);
    }
    {   // one job: status of the launch
        Launch l(1, 32);
        l.run(spread(32, 8));
        CHECK(l.launch_status == 0 && l.runs[0] == LG_G);
    }
    {   // places for three of each four: nobody waits for ever, the job keeps its status
        Launch l(1, 32);
        l.run(spread(24, 8));
        CHECK(l.runs[0] == 0 && l.status[0] == LG_LOST && (l.ctl->left & 255) == 24);
        for (int i = 0; i < 8; i++) l.group(24 + i, i);  // the rest arrives when the first have gone: no gang counts on those
        CHECK(l.runs[0] == 0 && l.launch_status == LG_LOST);
    }
    {   // the places are held by something that gets on: worth waiting for
        Launch l(3, 32);
        std::atomic<bool> stop{false};
        std::thread other([&] { while (!stop) { __atomic_fetch_add(&l.beat, 1, __ATOMIC_SEQ_CST); std::this_thread::yield(); } });
        l.arrive = [](int i) { if (i >= 24) ms(1500); };  // far longer than the poll limit
        l.run(spread(32, 8));
        stop = true;
        other.join();
        for (int j = 0; j < 3; j++) CHECK(l.status[j] == 0 && l.runs[j] == LG_G);
    }
    for (int late = 0; late < LG_G; late++)
        for (int at : {1, BARRIERS / 2, BARRIERS}) {  // a member comes far too late to a barrier of job 1
            Launch l(40, 32);
            l.wait = [&, late, at](int h, int job, int b) { if (job == 1 && h == late && b == at) while (l.lost < LG_G - 1) ms(1); };
            l.run(spread(32, 8));
            CHECK(l.status[1] == LG_LOST);
            for (int j = 0; j < 40; j++)
                if (j != 1) CHECK(l.status[j] == 0 && !l.wrong[j] && l.runs[j] == LG_G);
        }
    for (int late = 0; late < LG_G; late++) {  // the only job of a launch: its status says so
        Launch l(1, 32);
        l.wait = [&, late](int h, int, int b) { if (h == late && b == BARRIERS) while (l.lost < LG_G - 1) ms(1); };
        l.run(spread(32, 8));
        CHECK(l.launch_status == LG_LOST);
    }
    return failures != 0;
}
"""


def test_waits_end(tmp_path):
    """Jobs run once by whole gangs; where a gang cannot form, or a member comes
    too late, every workgroup leaves and the job's status says so."""
    r = subprocess.run([build(tmp_path, MODEL)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
