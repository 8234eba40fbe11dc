"""fp8 base weights decoded onto the bf16 matrix cores, on the tiles the planner takes."""
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 1e-2  # one rounding of T and one of y to bf16


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def rel(x, ref):
    return ((x.double() - ref).abs().max() / ref.abs().max()).item()


def inputs(gpu, M, N, K, r, seed, groups=1):
    from weightshared_torchtitan_amd import quantize_fp8_per_channel
    g = torch.Generator(device="cuda").manual_seed(seed)
    mk = lambda *s, std=1.0: (torch.randn(*s, device=gpu, generator=g) * std).bfloat16()  # noqa: E731
    q, sc = quantize_fp8_per_channel(mk(N, K, std=0.02))
    return mk(M, K), q, sc, (mk(groups * r, K, std=0.02) if r else None), (mk(N, r, std=0.02) if r else None)


CASES = [
    # M, N, K, r, the planner's tile
    (2700, 3072, 128, 16, (256, 192)),   # 768 chunks of codes a K tile for 512 threads
    (1024, 12288, 256, 128, (256, 192)),
]


@pytest.mark.parametrize("M,N,K,r,tile", CASES)
def test_fp8_tiles(gpu, wsl_opts, M, N, K, r, tile):
    from weightshared_torchtitan_amd import ops
    wsl_opts(fp8_prefill=1)
    _say(f"[fp8 tiles] M={M} N={N} K={K} r={r}")
    pl = ops.plan(M, K, r, [N], fp8=True)
    assert (pl["tile_m"], pl["tile_n"]) == tile
    x, q, sc, a, b = inputs(gpu, M, N, K, r, M + N + r)
    y = ops.lora_linear_op(x, q, sc, a, b, 1.0)
    ref = x.double() @ (q.double() * sc.double()[:, None]).t()
    if r:
        ref += (x.double() @ a.double().t()) @ b.double().t()
    assert rel(y, ref) <= TOL
    assert torch.equal(y, ops.lora_linear_op(x, q, sc, a, b, 1.0))
