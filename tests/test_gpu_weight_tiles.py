"""GPU: the weight-only GEMM (mxfp4_gemm_bf16, dual_mxfp4) at sizes that run each
tile of csrc/gemm_bf16f4.hip with and without K slices: K % 512 != 0, ragged
edges, M from 2, E8M0 bytes 0 and 255 -- against the float64 product of the
dequantized weight; the dual form gives the single form's bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# the tile of the single form; the dual form counts twice the tiles
SHAPES = [
    (4, 4096, 14336), (16, 1000, 8192), (20, 4096, 14336), (32, 130, 8192), (64, 4096, 8320),  # 32 x 128, sliced
    (20, 14330, 1024), (17, 5000, 640), (33, 515, 1408), (100, 4104, 4096),                                     # 32 x 128
    (15, 520, 1152), (2, 200, 4224), (12, 2752, 3328), (1, 320, 17536),                                         # skinny
    (162, 5000, 8192), (100, 5000, 6144),                          # 64 x 128, sliced (dual of 100: 128 x 128, sliced)
    (117, 8255, 8832), (267, 3601, 12160),                         # dual: 128 x 256 and 192 x 256, sliced
    (128, 14336, 512), (1000, 2048, 2048),                         # 64 x 128
    (200, 14336, 640), (600, 4090, 1152),                          # 128 x 128
    (300, 14336, 1152), (1500, 4096, 640), (4096, 4096, 640), (2048, 4090, 1536),   # 128 x 256
    (600, 14336, 896), (577, 14330, 512),                          # 192 x 256
    (1000, 14336, 512),                                            # 256 x 256 ring
]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_weight_tiles(M, N, K):
    from lockstep_amd import dual_gemm, fp4, mxfp4_gemm
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(M + 3 * N + 7 * K)
    a0, a1 = (torch.randn((M, K), device=dev, generator=g).to(torch.bfloat16) for _ in range(2))
    w = torch.randn((N, K), device=dev, generator=g) * 0.02
    pk, sc = fp4.quantize_pack_mxfp4(w)
    v = fp4.dequantize_packed(pk, sc).double().t()
    ref = a0.double() @ v
    c = mxfp4_gemm.mxfp4_gemm_bf16(a0, pk, sc, out_dtype=torch.float32)
    # exact products, fp32 accumulation: the repository's 1e-5 of the largest value
    assert ((c.double() - ref).abs().max() / ref.abs().max()).item() <= 1e-5
    # a 16-bit output is the fp32 one rounded
    assert torch.equal(mxfp4_gemm.mxfp4_gemm_bf16(a0, pk, sc), c.to(torch.bfloat16))
    # rows of a wider matrix, the same bits
    wide = torch.zeros((M, K + 40), device=dev, dtype=torch.bfloat16)
    wide[:, :K] = a0
    assert torch.equal(mxfp4_gemm.mxfp4_gemm_bf16(wide[:, :K], pk, sc, out_dtype=torch.float32), c)
    c0, c1 = dual_gemm.dual_mxfp4(a0, a1, pk, sc, out_dtype=torch.float32)
    assert torch.equal(c0, c)
    assert torch.equal(c1, mxfp4_gemm.mxfp4_gemm_bf16(a1, pk, sc, out_dtype=torch.float32))


@pytest.mark.parametrize("M,N,K", [(20, 4096, 14336), (100, 1000, 1152), (600, 4096, 640)])
def test_special_scale_bytes(M, N, K):
    """Byte 255 makes its column NaN, byte 0 is 2^-127; nothing else changes."""
    from lockstep_amd import fp4, mxfp4_gemm
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(K)
    a = torch.randn((M, K), device=dev, generator=g).to(torch.bfloat16)
    pk, sc = fp4.quantize_pack_mxfp4(torch.randn((N, K), device=dev, generator=g))
    c = mxfp4_gemm.mxfp4_gemm_bf16(a, pk, sc, out_dtype=torch.float32)
    s2 = sc.clone()
    s2[7, K // 32 - 1] = 255
    s2[9, :] = 0
    d = mxfp4_gemm.mxfp4_gemm_bf16(a, pk, s2, out_dtype=torch.float32)
    assert torch.isnan(d[:, 7]).all()
    assert (d[:, 9].abs() < 1e-30).all()
    keep = torch.ones(N, dtype=torch.bool, device=dev)
    keep[7] = keep[9] = False
    assert torch.equal(d[:, keep], c[:, keep])


def test_sliced_calls_of_two_threads_on_one_stream():
    """Both threads use the default stream and so one workspace; each gets its own result."""
    import threading

    from lockstep_amd import fp4, mxfp4_gemm
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(3)
    pk, sc = fp4.quantize_pack_mxfp4(torch.randn((4096, 14336), device=dev, generator=g) * 0.02)
    acts = [torch.randn((m, 14336), device=dev, generator=g).to(torch.bfloat16) for m in (20, 4)]
    want = [mxfp4_gemm.mxfp4_gemm_bf16(a, pk, sc) for a in acts]
    got = [[], []]

    def work(i):
        for _ in range(50):
            got[i].append(mxfp4_gemm.mxfp4_gemm_bf16(acts[i], pk, sc))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for g_, w_ in zip(got, want):
        assert len(g_) == 50 and all(torch.equal(c, w_) for c in g_)
