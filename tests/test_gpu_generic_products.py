"""The products for layouts off the tiled kernels (csrc/lora_generic.hip) at the edges of their
tiles (64 x 64 over k steps of 128; 128 x 128 over 64 where those fill the chip), with odd
strides and unaligned pointers, forward and every gradient against plain torch in float64; and
ranks off 8 on grid shapes, which the ops bring to the next multiple of 8 for the tiled kernels."""
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 1e-2  # one rounding of T or U and one of the result to bf16, of the largest value


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def rel(x, ref):
    return ((x.double() - ref).abs().max() / ref.abs().max().clamp_min(1e-30)).item()


def view(t, odd):
    """t as it is, or a view of odd stride and odd element offset into a wider buffer of NaN."""
    if not odd:
        return t
    big = torch.full((t.shape[0], t.shape[1] + 5), float("nan"), dtype=t.dtype, device=t.device)
    v = big[:, 1:1 + t.shape[1]]
    v.copy_(t)
    return v


def inputs(gpu, M, N, K, r, seed, odd=False):
    g = torch.Generator(device="cuda").manual_seed(seed)
    mk = lambda *s, std=1.0: view((torch.randn(*s, device=gpu, generator=g) * std).bfloat16(), odd)  # noqa: E731
    return mk(M, K), mk(N, K, std=0.05), mk(r, K, std=0.05), mk(N, r, std=0.05), mk(M, N)


def check_all(gpu, M, N, K, r, odd=False, seed=0, s=2.0):
    from weightshared_torchtitan_amd import ops
    x, w, a, b, gy = inputs(gpu, M, N, K, r, seed + M + 3 * N + 7 * K, odd)
    X, W, A, B, G = (t.double() for t in (x, w, a, b, gy))
    y = ops.lora_linear_op(x, w, None, a, b, s)
    assert rel(y, X @ W.t() + s * (X @ A.t()) @ B.t()) <= TOL
    assert rel(ops.lora_linear_op(x, None, None, a, b, s), s * (X @ A.t()) @ B.t()) <= TOL
    assert rel(ops.lora_linear_op(x, w, None, None, None, s), X @ W.t()) <= TOL
    assert rel(ops.lora_linear_bwd_input_op(gy, w, None, a, b, s), G @ W + s * (G @ B) @ A) <= TOL
    assert rel(ops.lora_linear_bwd_input_op(gy, w, None, None, None, s), G @ W) <= TOL
    for need_w in (False, True):
        got = ops.lora_linear_weight_grads_op(x, gy, a, b, s, need_w, True, True)
        again = ops.lora_linear_weight_grads_op(x, gy, a, b, s, need_w, True, True)
        assert all(torch.equal(p, q) for p, q in zip(got, again))
        assert rel(got[1], s * (G @ B).t() @ X) <= TOL and rel(got[2], s * G.t() @ (X @ A.t())) <= TOL
        if need_w:
            assert rel(got[0], G.t() @ X) <= TOL


CASES = [
    # M, N, K, r, odd strides and offsets
    (1, 1, 1, 1, False),
    (1, 100, 72, 3, True),
    (5, 63, 127, 7, False),
    (64, 64, 129, 9, False),       # one k past a step
    (65, 65, 128, 8, True),        # one row and column past a tile, rows unaligned
    (127, 129, 256, 16, True),     # grid sizes on unaligned rows
    (200, 333, 77, 31, False),
    (777, 150, 1000, 12, False),
    (130, 260, 136, 256, False),   # the largest rank
    (2100, 2090, 100, 5, False),   # 128-wide tiles
    (2049, 2177, 65, 33, True),
]


@pytest.mark.parametrize("M,N,K,r,odd", CASES)
def test_generic_layouts(gpu, M, N, K, r, odd):
    _say(f"[generic products] M={M} N={N} K={K} r={r} odd={odd}")
    check_all(gpu, M, N, K, r, odd)


@pytest.mark.parametrize("M,N,K,r", [(1, 512, 1024, 4), (64, 256, 512, 1), (200, 384, 256, 12), (300, 520, 192, 20),
                                     (130, 128, 64, 63), (600, 1024, 1024, 4), (100, 192, 256, 250)])
def test_ranks_off_8_on_grid_shapes(gpu, M, N, K, r):
    """Decode, prefill, split-K and rank pre-pass forms on padded factors."""
    _say(f"[rank off 8] M={M} N={N} K={K} r={r}")
    check_all(gpu, M, N, K, r)


@pytest.mark.parametrize("M,K,r,gn", [(8, 1024, 4, (256, 128)), (200, 256, 12, (256, 256, 128)), (96, 200, 12, (60, 33))])
def test_grouped_and_shared_base_ranks_off_8(gpu, M, K, r, gn):
    from weightshared_torchtitan_amd import ops
    _say(f"[grouped, rank off 8] M={M} K={K} r={r} groups={gn}")
    G = len(gn)
    x, w, _, b, _ = inputs(gpu, M, sum(gn), K, r, 5)
    a = inputs(gpu, M, 8, K, G * r, 6)[2]
    y = ops.lora_linear_grouped_op(x, w, None, a, b, 2.0, list(gn)).double()
    n0 = 0
    for j, n in enumerate(gn):
        ref = x.double() @ w[n0:n0 + n].double().t() + 2.0 * (x.double() @ a[j * r:(j + 1) * r].double().t()) @ b[n0:n0 + n].double().t()
        assert rel(y[:, n0:n0 + n], ref) <= TOL
        n0 += n
    n = gn[0]
    bs = torch.cat([inputs(gpu, 1, n, K, r, 9 + j)[3] for j in range(G)])
    y = ops.lora_linear_bcast_op(x, w[:n // 2], None, a, bs, 2.0, 1, G).double()
    rows = torch.arange(n, device=gpu) % (n // 2)
    for j in range(G):
        ref = x.double() @ w[rows].double().t() + 2.0 * (x.double() @ a[j * r:(j + 1) * r].double().t()) @ bs[j * n:(j + 1) * n].double().t()
        assert rel(y[:, j * n:(j + 1) * n], ref) <= TOL


@pytest.mark.parametrize("M,N,K,r", [(3, 50, 100, 5), (130, 200, 129, 8)])
def test_generic_fp8_base(gpu, M, N, K, r):
    from weightshared_torchtitan_amd import ops, quantize_fp8_per_channel
    _say(f"[generic fp8] M={M} N={N} K={K} r={r}")
    x, w, a, b, _ = inputs(gpu, M, N, K, r, 3)
    q, sc = quantize_fp8_per_channel(w)
    y = ops.lora_linear_op(x, q, sc, a, b, 1.0)
    ref = x.double() @ (q.double() * sc.double()[:, None]).t() + (x.double() @ a.double().t()) @ b.double().t()
    assert rel(y, ref) <= TOL


@pytest.mark.parametrize("r", [1, 2, 3, 5, 7, 12, 63])
@pytest.mark.parametrize("M,N,K", [(4, 256, 512), (70, 512, 1024), (200, 384, 256), (2050, 512, 128), (70, 100, 104)])
def test_infinities_stay_infinities_at_ranks_off_8(gpu, M, N, K, r):
    """A row of x (or grad_y) with an infinity: each output is the infinity or NaN that its own terms
    sum to (the decode, split-K, tiled, pre-pass and generic forms). Positive factors at the
    infinity's column, so that the low-rank term is +Inf and half of the base products agree."""
    from weightshared_torchtitan_amd import ops
    _say(f"[infinities, rank off 8] M={M} N={N} K={K} r={r}")
    x, w, a, b, gy = inputs(gpu, M, N, K, r, 11 + r)
    a, b = a.abs() + 2.0 ** -6, b.abs() + 2.0 ** -6
    x[2, 7] = gy[1, 5] = float("inf")
    X, W, A, B, G = (t.double().cpu() for t in (x, w, a, b, gy))
    wide = torch.cat([b, b.flip(0)])  # two groups: their own factors, one base twice
    got = [(ops.lora_linear_op(x, w, None, a, b, 2.0), X @ W.t() + 2.0 * (X @ A.t()) @ B.t()),
           (ops.lora_linear_op(x, None, None, a, b, 2.0), 2.0 * (X @ A.t()) @ B.t()),
           (ops.lora_linear_bwd_input_op(gy, w, None, a, b, 2.0), G @ W + 2.0 * (G @ B) @ A),
           (ops.lora_linear_grouped_op(x, torch.cat([w, w]), None, torch.cat([a, a]), wide, 2.0, [N, N]),
            torch.cat([X @ W.t() + 2.0 * (X @ A.t()) @ f.t() for f in (B, B.flip(0))], 1)),
           (ops.lora_linear_bcast_op(x, w, None, torch.cat([a, a]), wide, 2.0, 1, 2),
            torch.cat([X @ W.t() + 2.0 * (X @ A.t()) @ f.t() for f in (B, B.flip(0))], 1))]
    for y, ref in got:
        y = y.double().cpu()
        assert bool(ref.isinf().any()) and torch.equal(y.isnan(), ref.isnan())
        assert torch.equal(y == float("inf"), ref == float("inf")) and torch.equal(y.isfinite(), ref.isfinite())
        ok = ref.isfinite()
        assert rel(y[ok], ref[ok]) <= TOL


@pytest.mark.parametrize("form", ["linear", "grouped", "shared base"])
@pytest.mark.parametrize("M,N,K,r", [(65, 512, 1024, 4), (200, 1024, 4096, 12), (333, 2048, 4096, 63)])
def test_ranks_off_8_keep_parts_of_t_that_cancel(gpu, M, N, K, r, form):
    """T = x . A^T whose halves of K, in different splits of the launch, nearly cancel. The operands are
    small multiples of powers of two, so every sum is exact in fp32 in any order, and the error is T's
    rounding (at most one, u = 2^-8 of |T|) and y's: u |y| + u (1 + u) sum |T| |B|."""
    from weightshared_torchtitan_amd import ops
    _say(f"[rank off 8, cancelling T] M={M} N={N} K={K} r={r} {form}")
    G = 1 if form == "linear" else 2
    pl = ops.plan(M, K, (r + 7) // 8 * 8, [N] * G)
    assert pl["path"] == "prefill_splitk" and pl["k_splits"] % 2 == 0 and not pl["rank_prepass"]
    g = torch.Generator(device="cuda").manual_seed(r)
    ints = lambda n, *s: torch.randint(-n, n + 1, s, device=gpu, generator=g)  # noqa: E731
    v, e = ints(16, M, K // 2), ints(1, M, K // 2) * (ints(8, M, K // 2) == 0)
    x = (torch.cat([v, e - v], 1) / 8).bfloat16()
    a = (ints(16, G * r, K // 2) / 64).repeat(1, 2).bfloat16()
    b = (ints(16, G * N, r) / 64).bfloat16()
    w = torch.zeros(N if form == "shared base" else G * N, K, device=gpu).bfloat16()
    if form == "linear":
        y = ops.lora_linear_op(x, w, None, a, b, 2.0)
    elif form == "grouped":
        y = ops.lora_linear_grouped_op(x, w, None, a, b, 2.0, [N, N])
    else:
        y = ops.lora_linear_bcast_op(x, w, None, a, b, 2.0, 1, 2)
    u = 2.0 ** -8
    for j in range(G):
        t, bj = 2.0 * x.double() @ a[j * r:(j + 1) * r].double().t(), b[j * N:(j + 1) * N].double()
        want = t @ bj.t()
        tol = u * want.abs() + u * (1 + u) * t.abs() @ bj.abs().t()
        err = (y[:, j * N:(j + 1) * N].double() - want).abs()
        assert bool((err <= tol).all()), float((err / tol.clamp_min(1e-30)).max())


@pytest.mark.parametrize("N,K", [(100, 104), (128, 64), (64, 36)])
@pytest.mark.parametrize("which", [2, 3])
def test_input_gradient_refuses_factors_of_other_types(gpu, N, K, which):
    """On every route: the generic products, the tiled kernel and the transposed copy."""
    from weightshared_torchtitan_amd import ops
    x, w, a, b, gy = inputs(gpu, 70, N, K, 8, 4)
    args = [gy, w, None, a, b, 2.0]
    args[1 + which] = args[1 + which].float()
    with pytest.raises(TypeError):
        ops.lora_linear_bwd_input_op(*args)


def test_nan_stays_in_its_rows_and_columns(gpu):
    """A NaN or infinity of one row meets only that row's outputs, in products whose tiles are padded."""
    from weightshared_torchtitan_amd import ops
    x, w, a, b, gy = inputs(gpu, 70, 100, 100, 5, 4)
    x[3, 99] = float("nan")
    w[7, 2] = float("inf")
    y = ops.lora_linear_op(x, w, None, a, b, 2.0)
    bad = ~y.isfinite()
    assert bool(bad[3].all()) and bool(bad[:, 7].all())
    bad[3] = False
    bad[:, 7] = False
    assert not bad.any()
