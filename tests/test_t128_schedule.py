"""The counted waits of the 128 x 128 kernel against a model of its request queue, on the host: csrc/mx_t128_schedule.h is
what the kernel takes its order and its counts from."""
import pathlib
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parent.parent / "cutile-python_amd" / "csrc"
# pipeline depth, stages per K-quad, loads per wave and stage: 8-bit pairs, 8-bit x FP4, FP4 x FP4 (two K-steps a stage)
INSTANCES = [(ns, spq, tl) for ns in (2, 4) for spq, tl in ((4, 8), (4, 6), (2, 8))]
PROGRAM = """
#include <cstdio>
#include "mx_t128_schedule.h"
template <class S> void show() {
  for (int stages = 1; stages <= 40; ++stages)
    std::printf("%d %d %d %d %d %d\\n", S::NS, S::SPQ, S::TL, stages, mx::t128_uncovered<S>(stages),
                mx::t128_uncovered<S>(stages, true, (S::NS - 1) * S::TL));
}
int main() { SHOW }
"""


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    d = tmp_path_factory.mktemp("t128_schedule")
    show = " ".join(f"show<mx::T128Schedule<{ns}, {spq}, {tl}>>();" for ns, spq, tl in INSTANCES)
    (d / "p.cpp").write_text(PROGRAM.replace("SHOW", show))
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{CSRC}", "-o", str(d / "p"), str(d / "p.cpp")], check=True)
    rows = [tuple(map(int, line.split())) for line in subprocess.run([str(d / "p")], check=True, capture_output=True,
                                                                     text=True).stdout.splitlines()]
    assert len(rows) == 40 * len(INSTANCES)
    return rows


def test_everything_read_is_covered_by_a_wait(model):
    assert [r for r in model if r[4] != -1] == []


def test_the_model_finds_scales_requested_ahead_of_all_stages(model):
    """With every scale load in front of the stages, the first iteration of the four-deep FP4 x FP4 instance waits for all
    but 17 loads where stage 1 is followed by 16 only; every other instance has one scale load in flight or waits for
    everything, and is not affected."""
    assert {r[:3] for r in model if r[5] != -1} == {(4, 2, 8)}
    assert {r[5] for r in model if r[:3] == (4, 2, 8)} == {0}


def test_kernel_takes_order_and_waits_from_the_schedule():
    """The kernel states no count of its own: its waits between the prologue and the epilogue are the schedule's."""
    body = (CSRC / "mx_gemm_t128.hip").read_text().split("// ---- prologue")[1].split("// ---- epilogue")[0]
    waits = [line.strip() for line in body.splitlines() if "s_waitcnt" in line and "vmcnt" in line]
    assert len(waits) == 2 and "Sched::prologue_wait()" in waits[0] and "Sched::stage_wait(t)" in waits[1]
    assert "Sched::prologue_scales(k)" in body
