"""GPU: the f4 x f4 GEMM at sizes that run each of its output tiles
(csrc/gemm_f4f4.hip, pick_tile), with ragged edges, K % 256 == 128 and rows
padded with codes that must not count, against the float64 product of the
dequantized operands (mxfp4_gemm.py:116-174)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# tolerance: exact products, fp32 accumulation of K <= 2176 terms; the
# repository's bound for fp32 outputs is 1e-5 of the largest value, and a
# 16-bit output adds its unit roundoff times the value: rounding to p
# significant bits is within 2^-p of the value (bf16 p = 8, fp16 p = 11)
TOL = {torch.float32: 1e-5, torch.bfloat16: 2 ** -8 + 1e-5, torch.float16: 2 ** -11 + 1e-5}


# N % 4 != 0 runs the form for rows at any alignment
SHAPES = [
    (1, 1, 128, 0), (64, 64, 256, 0), (65, 63, 384, 16), (200, 520, 640, 0),        # 64 x 64
    (250, 8185, 1152, 0), (700, 2060, 512, 48), (900, 4104, 896, 0),                # 64 x 128
    (1111, 3000, 2176, 0), (1110, 2999, 1152, 0),                                   # 128 x 128
    (520, 8185, 640, 16), (1500, 4096, 1408, 0), (2050, 8192, 1024, 0),             # 192 x 128
    (1537, 4099, 640, 16), (1000, 8190, 1024, 0), (8189, 1024, 1152, 0),            # 256 x 128
    (4096, 4090, 384, 16),                                                          # 256 x 256
]


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K,pad", SHAPES)
def test_every_tile_against_float64(M, N, K, pad, out_dtype):
    from lockstep_amd import fp4, mxfp4_gemm
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(M + 7 * N + 13 * K)
    ops, vals = [], []
    for rows, std in ((M, 1.0), (N, 0.02)):
        x = torch.randn((rows, K), device=dev, generator=g) * std
        # block magnitudes over a few binades
        x *= torch.exp2(torch.randint(-3, 4, (rows, K // 32), device=dev, generator=g).float()).repeat_interleave(32, 1)
        pk, sc = fp4.quantize_pack_mxfp4(x, scale_layout="kmajor")
        vals.append(fp4.dequantize_packed(*fp4.quantize_pack_mxfp4(x)).double())
        if pad:  # rows followed by the largest codes: a read past K would show
            wide = torch.full((rows, K // 2 + pad), 0x77, dtype=torch.uint8, device=dev)
            wide[:, :K // 2] = pk
            pk = wide[:, :K // 2]
        ops.append((pk, sc))
    (ap, asc), (bp, bsc) = ops
    c = mxfp4_gemm.mxfp4_gemm_packed(ap, bp, asc, bsc, out_dtype=out_dtype)
    ref = vals[0] @ vals[1].t()
    assert c.shape == (M, N) and c.dtype == out_dtype
    err = (c.double() - ref).abs().max() / ref.abs().max()
    assert err.item() <= TOL[out_dtype]


def test_nan_scales_reach_exactly_their_outputs():
    """A NaN scale in the last half stage of K = 640 poisons its row only."""
    from lockstep_amd import fp4, mxfp4_gemm
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(5)
    a, b = (torch.randn((r, 640), device=dev, generator=g) for r in (100, 130))
    ap, asc = fp4.quantize_pack_mxfp4(a, scale_layout="kmajor")
    bp, bsc = fp4.quantize_pack_mxfp4(b, scale_layout="kmajor")
    asc[4, 37, 3] = 255
    c = mxfp4_gemm.mxfp4_gemm_packed(ap, bp, asc, bsc)
    assert torch.isnan(c[37]).all() and torch.isnan(c).sum().item() == 130
