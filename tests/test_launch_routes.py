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


KMAJOR = C.SCALE_E8M0_KMAJOR


def _launched(answers):
    assert all(r["rc"] == 0 for r in answers)
    return {name for r in answers for name, _ in r["launches"]}


def _args(name):
    return name[name.index("<") + 1:-1].split(", ")


def test_gpu_tile_tests_reach_every_tile(trace):
    """The shapes of the GPU tile tests launch every tile kernel of the library
    (with fp32 outputs; bf16 operands for the dense ones) and the large-tile
    kernel beside them."""
    from tests import test_gpu_dense_tiles, test_gpu_f4_tiles, test_gpu_fp8_tiles, test_gpu_weight_tiles
    kernels, = trace(["kernels 0 0 0"])

    def instances(kernel, **fixed):
        pos = {int(k[1:]): v for k, v in fixed.items()}
        return {n for n in kernels if n.startswith(kernel + "<") and all(_args(n)[i] == v for i, v in pos.items())}

    got = _launched(trace([f"f4 {m} {n} {k} {KMAJOR}" for m, n, k, _ in test_gpu_f4_tiles.SHAPES]))
    want = instances("gemm_f4f4_tile_kernel", a3="0")
    assert len(want) == 10 and got == want | {"gemm_f4f4_mx16_kernel<4, 0, false, false>"}

    got = _launched(trace([f"f8 {m} {n} {k} {nc}" for m, n, k in test_gpu_fp8_tiles.SHAPES
                           for nc in (0, 1) if not nc or n % 16 == 0]))
    want = instances("gemm_f8f8_tile_kernel", a0="0")
    assert len(want) == 10 and got == want | {"gemm_f8f8_kernel<0, true>", "gemm_f8f8_kernel<0, false>"}

    got = _launched(trace([f"dense {m} {n} {k} 1 {mode} {nc}" for m, n, k in test_gpu_dense_tiles.SHAPES
                           for mode in (0, 1, 2) for nc in (0, 1)]))
    want = instances("gemm_dense_tile_kernel", a0="1") | instances("gemm_dense_ring_kernel", a0="1")
    assert len(want) == 36 and got == want

    got = _launched(trace([f"w4 {m} {n} {k} {dual} 1 0" for m, n, k in test_gpu_weight_tiles.SHAPES for dual in (0, 1)]))
    whole = instances("gemm_bf16f4_tile_kernel", a0="0", a1="false")
    sliced = instances("gemm_bf16f4_tile_kernel", a1="true")
    assert len(whole) == 10 and len(sliced) == 5
    assert got >= whole | sliced | {n for n in kernels if n.startswith("gemm_bf16f4_ring_kernel<") and _args(n)[1] == "0"}


def test_decode_tests_run_the_decode_kernel(trace):
    """More than 4096 K and more than 16 weight rows per CU: two passes of the
    decode kernel; few weight rows: K slices."""
    from tests import test_gpu_gemm
    for shapes, kernel in ((test_gpu_gemm.DECODE, "gemm_bf16f4_decode_kernel"),
                           (test_gpu_gemm.DECODE_SLICED, "gemm_bf16f4_tile_kernel")):
        for r in trace([f"w4 {m} {n} {k} {dual} 1 0" for m, n, k in shapes for dual in (0, 1)]):
            assert r["launches"][0][0].startswith(kernel + "<")
    assert any(k > 4096 for _, _, k in test_gpu_gemm.DECODE)


def test_long_rows_keep_off_the_24_bit_offsets(trace):
    """K-major scales with rows of 2^19 bytes run the 32 x 32 x 64 kernel."""
    for ld in ("524288 0", "0 524288"):
        for k in (256, 384):
            r, = trace([f"f4 70 50 {k} {KMAJOR} {ld}"])
            assert r["launches"][0][0] == "gemm_f4f4_kernel<2, 4, 0>"


# us on the kernel named, and on the one that took the shape in between
@pytest.mark.parametrize("M,N,K,dual", [
    (1, 320, 21888, 0),     # 13.4, 55.5
    (2, 64, 2944, 0),       # 4.3, 10.4
    (12, 2752, 3328, 0),    # 6.5, 11.8
    (2, 9152, 14208, 0),    # 25.8, 38.5
    (6, 512, 2816, 1),      # 5.9, 10.2
])
def test_few_rows_of_any_depth_run_the_skinny_kernel(trace, M, N, K, dual):
    """Up to 16 rows that the decode kernel does not take (K % 512 != 0)."""
    r, r1 = trace([f"w4 {M} {N} {K} {dual} 1 0", f"w4 {M} {N} {K} {1 - dual} 1 0"])
    for x in (r, r1):   # the single and the dual form alike
        assert x["slices"] == 1 and x["launches"][0][0].startswith("gemm_bf16f4_skinny_kernel<")
    wide, = trace(["w4 10 59200 6784 0 1 0"])   # 60 us on the skinny kernel, 40 here
    assert wide["launches"][0][0].startswith("gemm_bf16f4_tile_kernel<")


@pytest.mark.parametrize("M,N,K,dual,kernel", [
    # us on the kernel named, and on the one that took the shape in between
    (12189, 29056, 512, 0, "gemm_bf16f4_ring_kernel<1, 0>"),                               # 419, 504
    (4829, 12864, 512, 1, "gemm_bf16f4_ring_kernel<2, 0>"),                                # 156, 197
    (30508, 384, 256, 0, "gemm_bf16f4_tile_kernel<0, false, 1, 4, 2, 1, 3, 2, true>"),     # 18.4, 24.0
    (252, 33771, 384, 0, "gemm_bf16f4_tile_kernel<0, false, 1, 4, 2, 1, 3, 2, false>"),    # 18.3, 27.8
])
def test_short_k_has_tiles_of_its_own(trace, M, N, K, dual, kernel):
    r, = trace([f"w4 {M} {N} {K} {dual} 1 0"])
    assert [x[0] for x in r["launches"]] == [kernel]


@pytest.mark.parametrize("M,N,K,kernel", [
    # us on the kernel named, and before (other tile or stores)
    (34898, 133, 1152, "gemm_f4f4_mx16_kernel<4, 0, false, false>"),     # 16.9, 31.4
    (520, 8185, 640, "gemm_f4f4_tile_kernel<6, 4, 3, 0, false>"),        # the stores of odd rows
    (15781, 28450, 384, "gemm_f4f4_mx16_kernel<4, 0, false, false>"),    # 362, 740
    (4443, 5184, 128, "gemm_f4f4_mx16_kernel<4, 0, false, false>"),      # 18.2, 28.1
    (4892, 4660, 896, "gemm_f4f4_mx16_kernel<4, 0, false, false>"),      # 26.4, 59.9
])
def test_f4_tiles_of_ragged_outputs(trace, M, N, K, kernel):
    r, = trace([f"f4 {M} {N} {K} {KMAJOR}"])
    assert [x[0] for x in r["launches"]] == [kernel]


@pytest.mark.parametrize("cmd,kernel", [
    # us on the kernel named, and on the one that took the shape in between
    ("dense 940 4256 960 1 2 1", "gemm_dense_tile_kernel<1, 2, true, 3, 2, 4>"),   # 32.3, 39.3
    ("dense 22565 1312 448 1 2 1", "gemm_dense_ring_kernel<1, 2, true>"),          # 96.8, 110
    ("f8 290 25088 4096 1", "gemm_f8f8_tile_kernel<0, true, 3, 2, 3>"),            # 46.2, 79.2
    ("f8 3618 14688 768 1", "gemm_f8f8_kernel<0, true>"),                          # 80.2, 92.4
])
def test_dense_and_e4m3_tiles_past_one_round(trace, cmd, kernel):
    r, = trace([cmd])
    assert [x[0] for x in r["launches"]] == [kernel]
