"""fp8 base weights decoded onto the bf16 matrix cores, on every tile the planner takes (two-buffer
rings of 128 x 128, 128 x 256, 256 x 192 and 256 x 256 tiles, and the split-K form, whose deep ring
holds the codes), with ragged M and N, T in the K loop and from the pre-pass, grouped and shared-base
rows, splits from one K tile on; and every code decodes exactly, by either decoder."""
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
    (65, 512, 64, 0, (128, 128)),       # one K tile
    (300, 1500, 128, 40, (128, 128)),   # two K tiles
    (70, 1000, 1088, 0, (128, 128)),    # 17 K tiles: no even split
    (130, 1000, 256, 16, (128, 128)),   # an N tail
    (333, 1536, 320, 64, (128, 128)),   # two rank blocks
    (333, 6144, 448, 128, (128, 128)),  # T from the pre-pass
    (2700, 2900, 128, 8, (128, 128)),   # more tiles than CUs
    (4096, 2048, 192, 32, (128, 256)),
    (3900, 2040, 448, 128, (128, 256)),
    (2700, 3072, 128, 16, (256, 192)),   # 768 chunks of codes a K tile for 512 threads
    (1024, 12288, 256, 128, (256, 192)),
    (8192, 2048, 192, 16, (256, 256)),
    (8100, 2040, 256, 128, (256, 256)),
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


SPLITS = [
    # M, N, K, r, splits
    (65, 512, 1024, 0, 2),
    (100, 1000, 4096, 16, 8),           # an N tail
    (333, 4096, 4096, 64, 2),           # two rank blocks
    (129, 1024, 8192, 128, 16),         # T from the pre-pass, applied by the first split
    (80, 4096, 12288, 256, 8),
]


@pytest.mark.parametrize("M,N,K,r,splits", SPLITS)
def test_fp8_splits_of_k(gpu, wsl_opts, M, N, K, r, splits):
    """The in-launch split-K form on codes: the planner's split count, equal to the unsplit launch
    within the bar, repeatable, its counters back at zero under graph replays."""
    from weightshared_torchtitan_amd import ops
    _say(f"[fp8 split-K] M={M} N={N} K={K} r={r}")
    pl = ops.plan(M, K, r, [N], fp8=True)
    assert pl["path"] == "prefill_splitk" and pl["k_splits"] == splits
    x, q, sc, a, b = inputs(gpu, M, N, K, r, M + N + r)
    y = ops.lora_linear_op(x, q, sc, a, b, 1.0)
    ref = x.double() @ (q.double() * sc.double()[:, None]).t()
    if r:
        ref += (x.double() @ a.double().t()) @ b.double().t()
    assert rel(y, ref) <= TOL
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        ops.lora_linear_op(x, q, sc, a, b, 1.0)
    s.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        out = ops.lora_linear_op(x, q, sc, a, b, 1.0)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, y) and torch.equal(ops.lora_linear_op(x, q, sc, a, b, 1.0), y)
    wsl_opts(prefill_split=-1, fp8_prefill=1)
    assert ops.plan(M, K, r, [N], fp8=True)["path"] == "prefill"
    assert rel(ops.lora_linear_op(x, q, sc, a, b, 1.0), ref) <= TOL


@pytest.mark.parametrize("r", [0, 32, 64, 128])
@pytest.mark.parametrize("tiles", [1, 2, 3, 4, 5])
def test_fp8_splits_of_few_k_tiles(gpu, wsl_opts, tiles, r):
    """Two splits of as many K tiles as the deep ring's four buffers, of fewer and of one more: the ring's
    start and end overlap."""
    from weightshared_torchtitan_amd import ops
    M, N, K = 130, 520, 128 * tiles
    wsl_opts(prefill_split=2, fp8_prefill=1)
    _say(f"[fp8 split-K] {tiles} K tiles a split, r={r}")
    pl = ops.plan(M, K, r, [N], fp8=True)
    assert pl["path"] == "prefill_splitk" and pl["k_splits"] == 2
    x, q, sc, a, b = inputs(gpu, M, N, K, r, tiles + r)
    y = ops.lora_linear_op(x, q, sc, a, b, 1.0)
    ref = x.double() @ (q.double() * sc.double()[:, None]).t()
    if r:
        ref += (x.double() @ a.double().t()) @ b.double().t()
    assert rel(y, ref) <= TOL
    assert torch.equal(y, ops.lora_linear_op(x, q, sc, a, b, 1.0))


@pytest.mark.parametrize("M,N,K,r", [(65, 512, 1024, 16), (100, 1000, 4096, 8), (333, 4096, 4096, 64),
                                     (200, 1024, 4096, 40)])
def test_fp8_splits_keep_parts_of_t_that_cancel(gpu, wsl_opts, M, N, K, r):
    """T = x . A^T whose halves of K, in different splits, nearly cancel. The operands are small
    multiples of powers of two, so every sum is exact in fp32 in any order, and the error is T's
    rounding (at most one, u = 2^-8 of |T|) and y's: u |y| + u (1 + u) sum |T| |B|."""
    from weightshared_torchtitan_amd import ops
    _say(f"[fp8 split-K, cancelling T] M={M} N={N} K={K} r={r}")
    pl = ops.plan(M, K, r, [N], fp8=True)
    assert pl["path"] == "prefill_splitk" and pl["k_splits"] % 2 == 0 and not pl["rank_prepass"]
    g = torch.Generator(device="cuda").manual_seed(r)
    ints = lambda n, *s: torch.randint(-n, n + 1, s, device=gpu, generator=g)  # noqa: E731
    v, e = ints(16, M, K // 2), ints(1, M, K // 2) * (ints(8, M, K // 2) == 0)
    x = (torch.cat([v, e - v], 1) / 8).bfloat16()
    a = (ints(16, r, K // 2) / 64).repeat(1, 2).bfloat16()
    b = (ints(16, N, r) / 64).bfloat16()
    W = torch.zeros(N, K, device=gpu).to(torch.float8_e4m3fn)
    y = ops.lora_linear_op(x, W, torch.ones(N, device=gpu), a, b, 2.0).double()
    t = 2.0 * x.double() @ a.double().t()
    want = t @ b.double().t()
    parts = 2.0 * x[:, :K // 2].double() @ a[:, :K // 2].double().t()
    assert float(parts.abs().mean()) > 16 * float(t.abs().mean())
    u = 2.0 ** -8
    tol = u * want.abs() + u * (1 + u) * t.abs() @ b.double().abs().t()
    assert bool(((y - want).abs() <= tol).all()), float(((y - want).abs() / tol.clamp_min(1e-30)).max())
    x[3, 5] = float("inf")  # the terms of an infinite part of T are itself and zeros
    W = torch.ones(N, K, device=gpu).to(torch.float8_e4m3fn)
    got = ops.lora_linear_op(x, W, torch.ones(N, device=gpu), a, b, 2.0)
    ref = (2.0 * x.double() @ a.double().t()) @ b.double().t() + x.double() @ W.double().t()
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())


def test_fp8_grouped_and_shared_base_rows(gpu, wsl_opts):
    from weightshared_torchtitan_amd import ops
    wsl_opts(fp8_prefill=1)
    M, K, r, gn = 300, 1024, 128, [512, 256, 256]
    assert ops.plan(M, K, r, gn, fp8=True)["path"] == "prefill_splitk"
    x, q, sc, a, b = inputs(gpu, M, sum(gn), K, r, 3, groups=3)
    y = ops.lora_linear_grouped_op(x, q, sc, a, b, 1.0, gn)
    n0 = 0
    for j, n in enumerate(gn):
        ref = x.double() @ (q[n0:n0 + n].double() * sc[n0:n0 + n].double()[:, None]).t() \
            + (x.double() @ a[j * r:(j + 1) * r].double().t()) @ b[n0:n0 + n].double().t()
        assert rel(y[:, n0:n0 + n], ref) <= TOL
        n0 += n
    base_n, g = 128, 2  # 256 wide projections on a base of 128 rows, two templates
    y = ops.lora_linear_bcast_op(x, q[:base_n], sc[:base_n], a, b[:768], 1.0, g, 3)
    c, d = torch.arange(256, device=gpu), base_n // g
    rows = c // (2 * d) * d + c % d
    for j in range(3):
        ref = x.double() @ (q[rows].double() * sc[rows].double()[:, None]).t() \
            + (x.double() @ a[j * r:(j + 1) * r].double().t()) @ b[j * 256:(j + 1) * 256].double().t()
        assert rel(y[:, j * 256:(j + 1) * 256], ref) <= TOL


@pytest.mark.parametrize("M,K,path", [(80, 128, "prefill"), (130, 128, "prefill"), (4096, 128, "prefill"),
                                      (128, 1024, "prefill_splitk"), (130, 4096, "prefill_splitk")])
def test_every_code_decodes_exactly(gpu, wsl_opts, M, K, path):
    """Row n of W holds code n in column n % 128 of the last 128 alone, and x's row m a one in column
    m % 128 of these: y picks the codes out (the first M of each half)."""
    from weightshared_torchtitan_amd import ops
    wsl_opts(fp8_prefill=1)
    assert ops.plan(M, K, 0, [256], fp8=True)["path"] == path
    codes = torch.arange(256, dtype=torch.uint8, device=gpu)
    W = torch.zeros(256, K, dtype=torch.uint8, device=gpu)
    W[torch.arange(256), K - 128 + torch.arange(256) % 128] = codes
    W = W.view(torch.float8_e4m3fn)
    x = torch.zeros(M, K, device=gpu, dtype=torch.bfloat16)
    m = torch.arange(M, device=gpu)
    x[m, K - 128 + m % 128] = 1.0
    y = ops.lora_linear_op(x, W, torch.ones(256, device=gpu), None, None, 0.0)
    want = codes.view(torch.float8_e4m3fn).float()
    for half in (0, 1):
        got = y[:128 if M >= 128 else M].float()
        k = torch.arange(got.shape[0], device=gpu)
        v, w = got[k, k + 128 * half], want[k + 128 * half]
        assert torch.equal(v.isnan(), w.isnan()) and torch.equal(v[~w.isnan()], w[~w.isnan()])
