"""GPU: mxfp4_gemm_fp8 (mxfp4_gemm.py:74-87) at sizes that run each output tile
of csrc/gemm_f8f8.hip, ragged edges and the shortest K included, B N-contiguous
(read in place) and K-contiguous: bit-exact on the E2M1 grid with scales of
2^-1 .. 2^1, where every fp32 sum is exact (multiples of 2^-4 below 2^18 for
K <= 1536)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


SHAPES = [
    (1, 16, 128), (64, 64, 256), (65, 80, 384), (300, 528, 1024), (131, 77, 256),   # 64 x 64
    (256, 8176, 512), (700, 2064, 1024), (2048, 2032, 512),                         # 64 x 128
    (700, 5008, 1024),                                                              # 128 x 128
    (1500, 4096, 640),                                                              # 192 x 128
    (1537, 4097, 256), (1000, 8192, 1024), (4095, 2048, 512),                       # 256 x 128
    (4096, 4080, 384),                                                              # 256 x 256
]


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_fp8_tiles_bit_exact(M, N, K, out_dtype):
    from lockstep_amd import fp4, mxfp4_gemm
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(M + 3 * N + 5 * K)
    ac, bc = (torch.randint(0, 16, (r, K), device=dev, generator=g).to(torch.uint8) for r in (M, N))
    ac[ac == 8], bc[bc == 8] = 0, 0
    sa, sb = (torch.exp2(torch.randint(-1, 2, (r, K // 32), device=dev, generator=g).float()) for r in (M, N))
    vals = fp4.E2M1_VALUES.to(dev)
    a = vals[ac.long()].double() * sa.double().repeat_interleave(32, 1)
    b = vals[bc.long()].double() * sb.double().repeat_interleave(32, 1)
    want = (a @ b.t()).to(out_dtype)
    a8 = fp4.codes_to_e4m3(ac)
    for nc in (True, False):
        b8 = fp4.codes_to_e4m3(bc.t().contiguous()) if nc else fp4.codes_to_e4m3(bc).t()
        c = mxfp4_gemm.mxfp4_gemm_fp8(a8, b8, sa, sb.t().contiguous(), out_dtype=out_dtype)
        assert torch.equal(c, want)
