"""The order in which the batched prefill attention fills, reads and refills
its LDS stages (gg_pf_schedule.h, the same code as the kernel runs), followed
on the CPU: a stage is read only after the copy of the wanted tile has arrived
for all waves, and refilled only after a barrier that follows its last reads."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "webgpu-gemma_amd", "csrc")
PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "gg_pf_schedule.h"
int main(int, char** argv) {
  const int tb = atoi(argv[1]), te = atoi(argv[2]);
  auto copy = [](int t, int part, int stage) { printf("copy %d %d %d\n", t, part, stage); };
  gg::pf_schedule_fill(tb, te, copy);
  gg::pf_schedule_run(tb, te, copy, [] { puts("arrive"); }, [] { puts("barrier"); },
                      [](int t, int ks) { printf("read %d 0 %d\n", t, ks); },
                      [](int t, int ks, int vs) { printf("read %d 0 %d\nread %d 1 %d\n", t + 1, ks, t, vs); },
                      [](int t, int vs) { printf("read %d 1 %d\n", t, vs); });
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("schedule")
    (d / "main.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(d / "main.cpp"), "-o", str(d / "main")], check=True)
    return str(d / "main")


@pytest.mark.parametrize("tb,tiles", [(0, 1), (0, 2), (3, 2), (0, 3), (5, 3), (1, 4), (0, 5), (7, 6), (2, 17)])
def test_stages_are_read_filled_and_refilled_only_after_a_barrier(program, tb, tiles):
    te = tb + tiles
    log = subprocess.run([program, str(tb), str(te)], check=True, capture_output=True, text=True).stdout.split("\n")
    holds, state = {}, {}   # (part, stage): tile, and copying -> arrived -> ready -> read
    used = {0: [], 1: []}
    for line in filter(None, log):
        op, *args = line.split()
        if op == "arrive":
            state = {k: "arrived" if v == "copying" else v for k, v in state.items()}
        elif op == "barrier":
            state = {k: {"arrived": "ready", "read": "ready"}.get(v, v) for k, v in state.items()}
        else:
            t, part, stage = map(int, args)
            if op == "copy":
                assert state.get((part, stage)) in (None, "ready"), f"{line}: the stage may still be read or filled"
                assert tb <= t < te, line
                holds[part, stage], state[part, stage] = t, "copying"
            else:
                assert state[part, stage] in ("ready", "read"), f"{line}: the copy is not known to have arrived"
                assert holds[part, stage] == t, f"{line}: the stage holds tile {holds[part, stage]}"
                state[part, stage] = "read"
                used[part].append(t)
    assert used[0] == used[1] == list(range(tb, te))
    assert "copying" not in state.values(), "a copy in flight at the end"
