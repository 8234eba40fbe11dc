"""dW over token splits of 256 x 256 tiles (csrc/lora_prefill.hip, product_tn_splits): sizes off the
tile on both sides, token counts off the 64-token tile, splits that do not divide the tokens, and the
padded rows' leading dimension, against float64.

|error| <= 2^-8 |dW| (one bf16 rounding) + the fp32 sums' n 2^-24 worst case, taken over the sum of
absolute products.
"""
import pytest
import torch

from weightshared_torchtitan_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,pad", [
    (12001, 1088, 960, 0),   # 12 splits of 16 token tiles, the last short; 64 and 192 columns past whole tiles
    (3001, 1536, 1536, 8),   # 6 splits, whole tiles, rows in wider buffers
    (1601, 2112, 2112, 0),   # 3 splits, 64 columns past whole tiles both ways
    (1001, 5120, 3328, 0),   # 260 large tiles, past one wave: product_splits' choice, 4 splits of 128 x 128 tiles
    (8192, 1024, 3072, 0),   # 5 splits of 26 token tiles, the last 24
])
def test_dw_over_large_tile_splits(gpu, M, N, K, pad):
    print(f"[dW splits] M={M} N={N} K={K} pad={pad}", flush=True)
    gen = torch.Generator().manual_seed(M)
    mk = lambda n: torch.randn(M, n + pad, generator=gen).bfloat16().to(gpu)[:, :n]  # noqa: E731
    x, gy = mk(K), mk(N)
    dw = ops.weight_grads(x, gy, None, None, 1.0, True, False, False)[0]
    xd, gd = x.double(), gy.double()
    want, mag = gd.t() @ xd, gd.abs().t() @ xd.abs()
    err = (dw.double() - want).abs()
    tol = 2.0 ** -8 * want.abs() + M * 2.0 ** -24 * mag
    assert bool((err <= tol).all()), float((err / tol).max())
    assert torch.equal(dw, ops.weight_grads(x, gy, None, None, 1.0, True, False, False)[0])
