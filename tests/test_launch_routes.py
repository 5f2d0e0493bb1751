"""CPU: which kernels a call launches, read from liblsmx.so itself with the HIP
runtime answered by tests/launch_trace.cpp (a 256-CU gfx950 that runs nothing)."""

import json
import shutil
import subprocess
from pathlib import Path

import pytest

from lockstep_amd import _capi as C

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def trace(tmp_path_factory):
    """trace([command, ...]) -> one answer per command."""
    rocm = Path("/opt/rocm/include")
    if not shutil.which("g++") or not rocm.exists():
        pytest.skip("needs g++ and the HIP headers")
    exe = tmp_path_factory.mktemp("trace") / "launch_trace"
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{rocm}", "-rdynamic",
                    str(ROOT / "tests" / "launch_trace.cpp"), "-o", str(exe), "-ldl", "-pthread"], check=True)

    def run(cmds):
        res = subprocess.run([str(exe), str(C.LIB_PATH)], input="\n".join(cmds) + "\n", capture_output=True, text=True,
                             timeout=120)
        assert res.returncode == 0, res.stderr
        return [json.loads(x) for x in res.stdout.splitlines()]
    return run


def test_calls_of_several_threads_on_one_stream_keep_their_launches_together(trace):
    """The K slices and their reduction are two launches through one workspace
    per stream: no other thread's call may come between them."""
    r, = trace(["threads 20 4096 14336 3 20"])
    assert r["rc"] == 0 and r["launches"] == 2 * r["calls"], "this shape must be sliced"
    assert r["split"] == 0


@pytest.mark.parametrize("lda,ldb", [(1 << 19, 0), (0, 1 << 19), ((1 << 24) - 16, (1 << 24) - 16)])
def test_quantizing_gemm_takes_long_rows_on_its_long_row_form(trace, lda, ldb):
    """32 rows of 2^19 bytes do not fit the plain form's 24-bit load offsets."""
    short, long_ = trace(["f4q 512 512 512 524272 524272", f"f4q 512 512 512 {lda} {ldb}"])
    assert [x[0] for x in short["launches"]] == ["gemm_f4f4_mx16_kernel<4, 1, true, false>"]
    assert [x[0] for x in long_["launches"]] == ["gemm_f4f4_mx16_kernel<4, 1, true, true>"]
