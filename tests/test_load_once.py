"""The sizes from which a kernel reads an operand past the caches (csrc/mx_load_once.h), on the host."""
import pathlib
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parent.parent / "cutile-python_amd" / "csrc"


@pytest.fixture(scope="module")
def evaluate(tmp_path_factory):
    """Values of C++ expressions over the header."""
    d = tmp_path_factory.mktemp("load_once")

    def run(*expressions):
        body = "".join(f'std::printf("%d\\n", (int)({e}));' for e in expressions)
        (d / "p.cpp").write_text('#include <cstdio>\n#include "mx_load_once.h"\nusing namespace mx;\nint main() { %s }\n' % body)
        subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", "-o", str(d / "p"), str(d / "p.cpp")], check=True)
        return [int(v) for v in subprocess.run([str(d / "p")], check=True, capture_output=True, text=True).stdout.split()]
    return run


def test_quantiser_input(evaluate):
    """The line is a number of elements: 32-bit input between 96 and 192 MB is slower that way, with a product behind and
    without one."""
    mi = 1 << 20
    assert evaluate(f"quantize_loads_once({48 * mi})", f"quantize_loads_once({48 * mi} - 8)", "quantize_loads_once(3072LL * 8192)",
                    "quantize_loads_once(8192LL * 8192)") == [1, 0, 0, 1]


def test_quantiser_stores_its_codes_for_whoever_reads_next():
    """A product reads the codes behind the quantiser: no store of theirs is non-temporal."""
    assert "nontemporal_store" not in (CSRC / "mx_aux.hip").read_text()


def test_streamed_weights(evaluate):
    """Whole lines that one workgroup alone reads, 96 MB of them: not behind several row tiles, not from inside a line, not a view
    or a broadcast that spans as much and reads less."""
    big = 12288, 8192, 8192   # rows, bytes read of a row, pitch: 96 MB
    call = lambda rows, row, pitch, at=0, tiles=1: f"stream_loads_once({rows}, {row}, {pitch}, {at}, {tiles})"
    assert evaluate(call(*big), call(*big, 128), call(12288, 8192, 8192 + 128), call(25000, 4096, 4096)) == [1] * 4
    assert evaluate(call(12287, 8192, 8192), call(*big, 0, 2), call(*big, 16), call(*big, 64), call(*big, 0x1000 | 8192 + 16),
                    call(12288, 8192, 8192 + 64), call(14336, 4096, 8192), call(1 << 20, 8192, 0)) == [0] * 8


def test_shapes_of_the_gpu_tests_reach_the_non_temporal_instances(evaluate):
    import test_gpu_load_once as g
    byte = lambda fmt, k: k // 2 if fmt == "e2m1" else k
    assert evaluate(*[f"stream_loads_once({n}, {byte(f, g.STREAM_K)}, {byte(f, g.STREAM_K)}, 0, 1)" for f, n in g.STREAM_N.items()],
                    *[f"weights_load_once({n}, {k // 2}, {k // 2})" for n, k in g.DECODE_NK],
                    *[f"stream_loads_once({min(t * g.MOE_TOPK, e) * rows}LL, {byte(f, k)}, {byte(f, k)}, 0, 1)"
                      for f, e in g.MOE_E.items() for t in g.MOE_T for rows, k in ((2 * g.MOE_F, g.MOE_H), (g.MOE_OUT, g.MOE_F))]
                    ) == [1] * (len(g.STREAM_N) + len(g.DECODE_NK) + 4 * len(g.MOE_T))
