"""The counted waits of the 128 x 128 kernel against a model of its request queue, on the host: csrc/mx_t128_schedule.h is
what the kernel takes its order and its counts from."""
import pathlib
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parent.parent / "cutile-python_amd" / "csrc"
# pipeline depth, stages per K-quad, loads per wave and stage: 8-bit pairs, 8-bit x FP4, FP4 x FP4 (two K-steps a stage), on tiles
# of 128 x 128 and of 64 x 64
INSTANCES = [(ns, spq, tl) for ns in (2, 4) for spq, tl in ((4, 8), (4, 6), (2, 8))] + \
            [(ns, spq, tl) for ns in (4, 8) for spq, tl in ((4, 4), (4, 3), (2, 4))]
PROGRAM = """
#include <cstdio>
#include "mx_t128_schedule.h"
template <class S> void show() {
  for (int stages = 1; stages <= 40; ++stages) {
    int any = -1, shorter = 0;
    for (int loads = 0; loads <= S::kAnyLoads; ++loads)
      for (int ahead = 0; ahead <= loads; ++ahead) {
        const int u = mx::t128_any_uncovered<S>(stages, loads, ahead);
        if (u != -1) any = u;
        // one load more left open than there may be: found where nothing but the stages' own loads is in the queue
        if (loads == 0)
          shorter = (mx::t128_any_uncovered<S>(stages, 0, 0, S::any_prologue_wait() + 1) == -2) +
                    2 * (mx::t128_any_uncovered<S>(stages, 0, 0, S::any_prologue_wait(), S::any_stage_wait() + 1) == 0);
      }
    std::printf("%d %d %d %d %d %d %d %d\\n", S::NS, S::SPQ, S::TL, stages, mx::t128_uncovered<S>(stages),
                mx::t128_uncovered<S>(stages, true, (S::NS - 1) * S::TL), any, shorter);
  }
}
int main() {
  SHOW
  std::printf("%d\\n", mx::t128_any_uncovered<mx::T128Schedule<4, 1, 8>>(8));
}
"""


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    d = tmp_path_factory.mktemp("t128_schedule")
    show = " ".join(f"show<mx::T128Schedule<{ns}, {spq}, {tl}>>();" for ns, spq, tl in INSTANCES)
    (d / "p.cpp").write_text(PROGRAM.replace("SHOW", show))
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{CSRC}", "-o", str(d / "p"), str(d / "p.cpp")], check=True)
    rows = [tuple(map(int, line.split())) for line in subprocess.run([str(d / "p")], check=True, capture_output=True,
                                                                     text=True).stdout.splitlines()]
    assert len(rows) == 40 * len(INSTANCES) + 1
    return rows


def test_everything_read_is_covered_by_a_wait(model):
    assert [r for r in model[:-1] if r[4] != -1] == []


def test_the_model_finds_scales_requested_ahead_of_all_stages(model):
    """With every scale load in front of the stages, an instance that has several of them in flight waits for too little: the first
    iteration of the four-deep FP4 x FP4 instance for all but 17 loads where stage 1 is followed by 16 only.  The others have one scale
    load in flight or wait for everything, and are not affected."""
    deep = {(4, 2, 8), (4, 2, 4), (8, 4, 4), (8, 4, 3), (8, 2, 4)}
    assert {r[:3] for r in model[:-1] if r[5] != -1} == deep
    assert {r[5] for r in model if r[:3] == (4, 2, 8)} == {0}


def test_scales_at_any_byte_are_covered_too(model):
    """However many of a quad's register loads are still in the queue, and wherever the first quad's lie."""
    assert [r for r in model[:-1] if r[6] != -1] == []


def test_the_model_finds_a_wait_for_too_little_and_scales_read_in_the_stage_that_writes_them(model):
    assert {r[7] for r in model[:-1]} == {3}
    assert model[-1] == (-4,)   # one stage a quad


def test_kernel_takes_order_and_waits_from_the_schedule():
    """The kernel states no count of its own: its waits between the prologue and the epilogue are the schedule's, each scale form
    its own."""
    body = (CSRC / "mx_gemm_t128.hip").read_text().split("// ---- prologue")[1].split("// ---- epilogue")[0]
    waits = [line.strip() for line in body.splitlines() if "s_waitcnt" in line and "vmcnt" in line]
    assert len(waits) == 2
    assert "vmcnt_imm(ANY ? Sched::any_prologue_wait() : Sched::prologue_wait())" in waits[0]
    assert "vmcnt_imm(ANY ? Sched::any_stage_wait() : Sched::stage_wait(t))" in waits[1]
    assert "!ANY && Sched::prologue_scales(k)" in body
    # scales at any byte: written behind the barrier of a quad's first stage, read at its last
    first, last = body.split("if constexpr (t == 0)")[1], body.split("if constexpr (t == SPQ - 1)")
    assert "store_any(Q + 1);" in first.split("issue(s + NS, buf)")[0] and "read_scales(Q + 1);" in last[1].splitlines()[0]
    assert "s_barrier" in body.split("store_any(q0);")[1].split("read_scales(q0);")[0]


def test_scales_at_any_byte_keep_the_requests_together_for_long_k(tmp_path):
    cases = [(992, 1, 1), (4096, 1, 1), (4097, 1, 1), (8192, 2, 1), (8193, 2, 1), (5120, 0, 2), (5121, 1, 2), (14336, 3, 2)]
    body = "".join('std::printf("%%d\\n", (int)mx::t128_any_spread(%d, %d, %d));' % c for c in cases)
    (tmp_path / "p.cpp").write_text('#include <cstdio>\n#include "mx_t128_schedule.h"\nint main() { %s }\n' % body)
    subprocess.run(["g++", "-std=c++17", f"-I{CSRC}", "-o", str(tmp_path / "p"), str(tmp_path / "p.cpp")], check=True)
    got = subprocess.run([str(tmp_path / "p")], check=True, capture_output=True, text=True).stdout.split()
    assert got == ["1", "1", "0", "1", "0", "1", "0", "1"]
