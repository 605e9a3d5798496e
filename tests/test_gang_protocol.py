"""The protocol of the gangs' workgroups (lh_gang_proto.h), compiled for the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "luna.jl_amd", "csrc")


def build(tmp_path, body):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text("#define __device__\n#define __forceinline__ inline\n#include <stdio.h>\n"
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
