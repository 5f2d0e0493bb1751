"""CPU: which kernels a call launches, read from liblsmx.so itself with the HIP
runtime answered by tests/launch_trace.cpp (a 256-CU gfx950 that runs nothing)."""

import json
import math
import random
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


def test_slices_query_is_the_plan_that_runs(trace):
    """lsmx_gemm_bf16f4_slices says how many slices a call with a workspace runs;
    their partial tiles stay within the bytes asked for, those within the fixed
    64 MiB of lsmx_gemm_bf16f4_noalloc; without slices or a workspace the call
    launches the same kernels."""
    rng = random.Random(5)
    shapes = [(20, 4096, 14336), (128, 14336, 4096), (64, 2304, 4096), (200, 1024, 4096), (32, 2048, 2048)]
    for _ in range(4000):
        m = rng.choice((rng.randint(1, 64), int(math.exp(rng.uniform(4, 8)))))
        shapes.append((m, int(math.exp(rng.uniform(0, 10.5))), 128 * int(math.exp(rng.uniform(0, 5.5)))))
    cmds = [(s, dual) for s in shapes for dual in (0, 1)]
    with_ws, without = (trace([f"w4 {M} {N} {K} {d} {ws} 0" for (M, N, K), d in cmds]) for ws in (1, 0))
    sliced = 0
    for ((M, N, K), dual), r, r0 in zip(cmds, with_ws, without):
        names = [x[0] for x in r["launches"]]
        assert r["rc"] == 0 and r["workspace"] <= 64 << 20
        assert (r["slices"] > 1) == any("splitk_reduce" in n for n in names), (M, N, K, dual, r)
        if r["slices"] == 1:
            assert r["launches"] == r0["launches"]
            continue
        # gemm_bf16f4_tile_kernel<CT, SPLITK, WM, WN, TM, TN, ...>: tiles of 32 WM TM x 32 WN TN
        _, split, wm, wn, tm, tn = names[0].split("<")[1].split(", ")[:6]
        bm, bn = 32 * int(wm) * int(tm), 32 * int(wn) * int(tn)
        grid = r["launches"][0][1]
        assert split == "true" and grid == -(-M // bm) * -(-N // bn) * (1 + dual) * r["slices"]
        assert grid * bm * bn * 4 <= r["workspace"]
        sliced += 1
    assert sliced > 100
