"""The many-token kernels against plain 64-bit references at the edges of their tiles: the
dense bf16 GEMM, the prompts of the core layers, and the grouped MoE kernels over I8 rows."""
import numpy as np
import pytest
import torch

from npu_amd import ops
from npu_amd.gguf_types import GGMLQuantizationType as QT

pytestmark = pytest.mark.gpu


# (M, K, T): 128 x 64 tiles with an odd M (scalar stores) and a last half step; K split in
# two with a K of one step; K split in four with a last part that is short, and parts that
# hold no step at all; one token past a tile; the first size the tiles take; the few-token
# kernel's last size below them
@pytest.mark.parametrize("M,K,T", [(4099, 96, 700), (4096, 32, 300), (2050, 1056, 260), (3072, 160, 65),
                                   (3072, 2048, 17), (3072, 2048, 16)])
def test_gemm_bf16_tiles(gpu, M, K, T):
    g = torch.Generator().manual_seed(M + K + T)
    w = (torch.randn(M, K, generator=g) * 0.05).to(torch.bfloat16)
    x = torch.randn(T, K, generator=g) * torch.exp(torch.randn(T, 1, generator=g))
    print(f"gemm case M={M} K={K} T={T}", flush=True)
    y = ops.matvec(QT.BF16, w.to(gpu), M, K, x.to(gpu)).cpu().double()
    ref = x.double() @ w.double().T
    # every product is exact; a value is a chain of at most 24 + K / 256 additions of 32-product
    # sums, each rounding at most 2^-24 of the sum of magnitudes (twice that for the inner sums)
    bound = (2 * 24 + K / 256 + 4) * 2.0 ** -24 * (x.abs().double() @ w.abs().double().T)
    assert bool(((y - ref).abs() <= bound).all())
    assert float((y - ref).norm() / ref.norm()) <= 1e-6
