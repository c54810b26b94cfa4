"""The waits of the LU-SGS sweeps (csrc/lusgs_plan.h, the code that the kernel
runs), compiled for the CPU with a made-up clock and memory: a wait ends when its
terms arrive, however long ago an earlier sweep was given up; it is given up at
the limit; and it ends early only for the abort word of its own sweep."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "combustioncodegpu_amd", "csrc")

HARNESS = r"""
#include <cstdio>
#include "lusgs_plan.h"

struct Gpu {  // what the kernel keeps: the context's error flags, the sweep's abort word
  int flags = 0, word = 0;
  long long time = 0;
  // a wait whose terms arrive at the poll `arrive`; another patch raises the word at the poll `other`
  bool wait(long long arrive, long long limit, long long other = -1) {
    long long polls = 0;
    const bool ok = cfx::lu_wait([&] { return polls < arrive; },
                                 [&] {
                                   ++polls, ++time;
                                   if (polls == other) word = 1;
                                 },
                                 [&] { return time; }, limit, [&] { flags |= 2, word = 1; }, [&] { return word != 0; });
    std::printf("%d %lld %d %d\n", ok ? 1 : 0, polls, flags, word);
    return ok;
  }
  void reset() { word = 0; }  // before every sweep
};

int main() {
  Gpu g;
  g.wait(0, 1000);            // there already
  g.wait(700, 1000);          // late, in time
  g.wait(1 << 20, 1000);      // never: given up
  g.wait(1 << 20, 1000000);   // the same sweep's next wait
  g.wait(0, 1000);            // ... of which the terms are there
  g.reset();
  g.wait(700, 1000);          // the next sweep: its patches are running
  g.wait(1 << 20, 1000000, 300);  // ended by another patch of its own sweep
  return 0;
}
"""


def test_waits(tmp_path):
    src = tmp_path / "wait.cpp"
    src.write_text(HARNESS)
    exe = str(tmp_path / "wait")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", exe], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split("\n")
    rows = [tuple(map(int, r.split())) for r in out if r]
    # (terms there, polls, error flags, abort word)
    assert rows == [(1, 0, 0, 0), (1, 700, 0, 0), (0, 1024, 2, 1), (0, 256, 2, 1), (1, 0, 2, 1),
                    (1, 700, 2, 0), (0, 512, 2, 1)]
    # the kernel's waits have no other end: its one look at the flags is the report
    with open(os.path.join(CSRC, "kernels_ns.hip")) as f:
        code = f.read()
    sweep = code[code.index("lusgs_sweep_kernel(const BlockView"):code.index("int launch_lusgs_coef")]
    assert sweep.count("lu_wait(") == 1 and sweep.count("atomicOr(flags, kLuFlag)") == 1
    assert sweep.count("flags") == 2  # the parameter and the report
