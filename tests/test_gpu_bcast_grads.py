"""Every gradient of the shared-base linear in one call (wsl::lora_linear_bcast_grads,
csrc/lora_backward.hip) against float64 gradients of the reference's composition: base rows shared over
heads and groups, token counts around the 64-token tiles and their splits, ranks whose groups' sum is
below and off 16, each output alone, strided operands; and the layouts it leaves to the composed route.

Rounding of the outputs, with u = 2^-8 (half a unit of bf16's eighth significant bit): gy's fold over the
base rows and U, T are rounded to bf16 once before the second product, the result once, so
|error| <= u |exact| + u (1 + u) sum |folded or U| |other|; both products accumulate in fp32, whose 2^-24
terms the factor 1.01 and the absolute 1e-6 cover.
"""
import pytest
import torch

from weightshared_torchtitan_amd import ops

U = 2.0 ** -8


def _operands(M, N, K, r, base_n, G, seed):
    gen = torch.Generator().manual_seed(seed)
    mk = lambda *s, std=1.0: (torch.randn(*s, generator=gen) * std).bfloat16()  # noqa: E731
    return (mk(M, K), mk(M, G * N), mk(base_n, K, std=K ** -0.5), mk(G * r, K, std=K ** -0.5),
            mk(G * N, r, std=0.1))


def _oracle(x, gy, w, a, b, scale, g, G):
    """float64 gradients and their error bounds."""
    x, gy, w, a, b = (t.double() for t in (x, gy, w, a, b))
    M, base_n, r = x.shape[0], w.shape[0], b.shape[1]
    N, D = gy.shape[1] // G, base_n // g
    fold = lambda t: t.view(M, G, g, N // base_n, D).sum(dim=(1, 3)).reshape(M, base_n)  # noqa: E731
    gyb = fold(gy)
    bg, ag = b.view(G, N, r), a.view(G, r, -1)
    gj = gy.view(M, G, N).transpose(0, 1)
    u = torch.cat([scale * gj[j] @ bg[j] for j in range(G)], 1)
    t = [scale * x @ ag[j].t() for j in range(G)]
    dx, bx = gyb @ w + u @ a, gyb.abs() @ w.abs() + u.abs() @ a.abs()
    dw, bw = gyb.t() @ x, gyb.abs().t() @ x.abs()
    da, ba = u.t() @ x, u.abs().t() @ x.abs()
    db = torch.cat([gj[j].t() @ t[j] for j in range(G)])
    bb = torch.cat([gj[j].abs().t() @ t[j].abs() for j in range(G)])
    return [(v, 1.01 * (U * v.abs() + U * (1 + U) * bnd) + 1e-6) for v, bnd in ((dx, bx), (dw, bw), (da, ba), (db, bb))]


def _check(got, want, names="dx dw da db".split()):
    for name, t, (v, tol) in zip(names, got, want):
        if t is None or (t.numel() == 0 and v.numel() != 0):
            continue
        err = (t.double().cpu() - v).abs()
        assert bool((err <= tol).all()), (name, float((err / tol).max()))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,r,base_n,g,G", [
    (1, 128, 64, 8, 64, 1, 1),         # one row, one group
    (63, 64, 128, 16, 64, 2, 3),       # N = base_n, below one token tile
    (65, 256, 192, 8, 64, 4, 2),       # four heads a template, one row over a tile
    (200, 192, 320, 24, 64, 8, 3),     # template width 8; group rank sum 72
    (513, 512, 256, 32, 256, 2, 4),    # token splits, group rank sum 128
    (300, 128, 576, 56, 128, 1, 4),    # the most groups, rank sum 224, no head sharing
    (257, 256, 128, 128, 128, 1, 2),   # the rank limit
])
def test_bcast_grads(gpu, M, N, K, r, base_n, g, G):
    print(f"[bcast grads] M={M} N={N} K={K} r={r} base_n={base_n} g={g} groups={G}", flush=True)
    host = _operands(M, N, K, r, base_n, G, seed=M + N)
    want = _oracle(*host, 2.0, g, G)
    x, gy, w, a, b = (t.to(gpu) for t in host)
    assert ops.bcast_grads_supported(x, gy, w, a, b, g, G)
    full = ops.lora_linear_bcast_grads_op(x, gy, w, a, b, 2.0, g, G, True, True, True, True)
    _check(full, want)
    for i in range(4):  # each output alone: the same bits
        only = ops.lora_linear_bcast_grads_op(x, gy, w, a, b, 2.0, g, G, *(j == i for j in range(4)))
        assert torch.equal(only[i], full[i]) and all(only[j].numel() == 0 for j in range(4) if j != i)
    no_lora = ops.lora_linear_bcast_grads_op(x, gy, w, None, None, 2.0, g, G, True, True, False, False)
    zero = (torch.zeros(G * 8, K).bfloat16(), torch.zeros(G * N, 8).bfloat16())
    _check(no_lora[:2], _oracle(*host[:3], *zero, 2.0, g, G)[:2])


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["strided", "offset", "template 4", "rank 12", "K off", "K off rank"])
def test_bcast_backward_routes(gpu, case):
    """The op's backward over layouts: rows 16 bytes apart in wider buffers, storage off 16 bytes, and
    those the one call does not take give gradients within the same bounds through the public op."""
    M, N, K, r, base_n, g, G = 130, 128, 128, 16, 64, 2, 3
    if case == "template 4":
        g = 16
    elif case == "rank 12":
        r = 12
    elif case.startswith("K off"):
        K, r = 136, 12 if case.endswith("rank") else 16
    print(f"[bcast backward] {case}", flush=True)
    host = _operands(M, N, K, r, base_n, G, seed=7)
    dev = [t.to(gpu) for t in host]
    if case in ("strided", "offset"):
        wide = []
        for t in dev:
            off = 8 if case == "strided" else 1
            buf = torch.zeros(t.shape[0], t.shape[1] + 16, dtype=t.dtype, device=gpu)
            buf[:, off:off + t.shape[1]] = t
            wide.append(buf[:, off:off + t.shape[1]])
        dev = wide
    x, gy, w, a, b = (t.detach().requires_grad_() for t in dev)
    taken = ops.bcast_grads_supported(x, gy, w, a, b, g, G)
    assert taken == (case == "strided")
    y = ops.lora_linear_bcast_op(x, w, None, a, b, 2.0, g, G)
    got = torch.autograd.grad(y, (x, w, a, b), gy.detach())
    want = _oracle(*host, 2.0, g, G)
    if not taken:  # the composed route rounds the base part and the delta of dx apart
        v, tol = want[0]
        want[0] = (v, 3 * tol)
    _check(got, want)


def _wrong():
    """Name -> operands that do not belong together, and whether the factors' gradients are asked for."""
    M, N, K, r, base_n, G = 24, 128, 64, 8, 64, 2
    good = dict(zip(("x", "gy", "w", "a", "b"), _operands(M, N, K, r, base_n, G, seed=1)), g=2, n_groups=G)
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16)  # noqa: E731
    for name, change in {
        "gy rows": {"gy": z(M - 1, G * N)}, "gy columns": {"gy": z(M, G * N - 1)}, "N": {"gy": z(M, G * 96)},
        "w columns": {"w": z(base_n, K - 8)}, "a rows": {"a": z(r, K)}, "a columns": {"a": z(G * r, K - 8)},
        "b rows": {"b": z(N, r)}, "a alone": {"b": None}, "b alone": {"a": None}, "no factors": {"a": None, "b": None},
        "rank 0": {"a": z(0, K), "b": z(G * N, 0)}, "template": {"g": 3}, "no template": {"g": 0},
        "no group": {"n_groups": 0}, "groups": {"n_groups": 5}, "3-d": {"x": z(2, M // 2, K)},
        **{f"{n} type": {n: good[n].float()} for n in ("x", "gy", "w", "a", "b")},
    }.items():
        yield name, {**good, **change}


@pytest.mark.parametrize("name,args", _wrong(), ids=lambda v: v if isinstance(v, str) else "")
def test_operands_that_do_not_match_are_refused(name, args):
    with pytest.raises((TypeError, ValueError)):
        ops._bcast_grads_operands(**args, need_ab=True)


@pytest.mark.gpu
def test_bcast_grads_op_checks_its_operands(gpu):
    for name, args in _wrong():
        print(f"[bcast grads] refused: {name}", flush=True)
        x, gy, w, a, b = (args[n].to(gpu) if args[n] is not None else None for n in ("x", "gy", "w", "a", "b"))
        for op in (ops.lora_linear_bcast_grads_op, torch.ops.wsl.lora_linear_bcast_grads):
            with pytest.raises((TypeError, ValueError)):
                op(x, gy, w, a, b, 2.0, args["g"], args["n_groups"], True, True, True, True)


@pytest.mark.gpu
@pytest.mark.parametrize("which", range(5))
@pytest.mark.parametrize("layout", ["columns apart", "transposed", "overlapping"])
def test_bcast_grads_takes_any_strides(gpu, which, layout):
    """An operand with columns apart, transposed, or with rows that overlap gives the gradients of its values."""
    M, N, K, r, base_n, g, G = 65, 128, 128, 16, 64, 2, 2
    print(f"[bcast grads] operand {which} {layout}", flush=True)
    host = list(_operands(M, N, K, r, base_n, G, seed=3))
    dev = [t.to(gpu) for t in host]
    t = dev[which]
    if layout == "columns apart":
        buf = torch.full((t.shape[0], 2 * t.shape[1]), float("nan"), dtype=t.dtype, device=gpu)
        buf[:, ::2] = t
        dev[which] = buf[:, ::2]
    elif layout == "transposed":
        dev[which] = t.t().contiguous().t()
    else:  # row i + 1 starts 8 elements after row i
        line = t.flatten()[:8 * (t.shape[0] - 1) + t.shape[1]].contiguous()
        dev[which] = line.as_strided(t.shape, (8, 1))
        host[which] = dev[which].cpu()
    _check(ops.lora_linear_bcast_grads_op(*dev, 2.0, g, G, True, True, True, True), _oracle(*host, 2.0, g, G))
