"""GPU: the bf16 / fp16 dense GEMMs (dual_gemm.py:188-255) at sizes that run
each output tile of csrc/gemm_dense_ring.hip, ragged edges and the shortest K
included: bit-exact on the integer grid, where every order of summation is
exact (|sum| <= 144 * 2 * K < 2^24), with B N-contiguous (read in place) and
K-contiguous."""

import pytest
import torch

pytestmark = pytest.mark.gpu

Q = [0, 1, 2, 3, 4, 6, 8, 12, -1, -2, -3, -4, -6, -8, -12]


# the tile of one product (gemm, packed); two products count twice the tiles
SHAPES = [
    (1, 8, 64), (64, 64, 128), (65, 72, 192), (500, 520, 640), (511, 2040, 320),     # 64 x 64
    (1000, 1032, 1024),                                                              # 64 x 128
    (2048, 2040, 512), (1500, 2000, 1024), (3000, 1000, 512),                        # 128 x 128
    (2000, 2056, 256), (4095, 1032, 512), (4096, 4104, 192),                         # 192 x 128
    (2048, 4096, 512),                                                               # 256 x 128
    (4095, 4088, 320),                                                               # 256 x 256
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("form", ["gemm", "packed", "separate"])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_dense_tiles_bit_exact(M, N, K, form, dtype):
    from lockstep_amd import dual_gemm as D
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(M + 3 * N + 5 * K)
    q = torch.tensor(Q, device=dev, dtype=dtype)
    a1, a2 = (q[torch.randint(0, 15, (M, K), device=dev, generator=g)] for _ in range(2))
    b1, b2 = (q[torch.randint(0, 15, (K, N), device=dev, generator=g)] for _ in range(2))
    want1, want2 = a1.float() @ b1.float(), a2.float() @ b2.float()
    for nc in (True, False):
        x1, x2 = (b1, b2) if nc else (b1.t().contiguous().t(), b2.t().contiguous().t())
        if form == "gemm":
            assert torch.equal(D.gemm(a1, x1), want1)
        elif form == "packed":
            assert torch.equal(D.dual_packed(a1, a2, x1, x2), want1 + want2)
        else:
            c1, c2 = D.dual_separate(a1, a2, x1, x2)
            assert torch.equal(c1, want1) and torch.equal(c2, want2)
