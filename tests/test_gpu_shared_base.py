"""The shared-base linear with its base computed once per tile (csrc/lora_prefill.hip, the SHARE form):
token counts and base rows off the tiles, templates 8 wide, every rank chunk count, one and several
groups, heads per template, unaligned output rows, and a workspace that only has room for the form
over the output columns, against float64.

T is rounded to bf16 once and the sum once (u = 2^-8): |error| <= u |y| + u (1 + u) sum |T| |B|, the
fp32 accumulation covered by the factor 1.01 and 2^-16 of the absolute products.
"""
import ctypes

import pytest
import torch

from weightshared_torchtitan_amd import _native, ops

pytestmark = pytest.mark.gpu
U = 2.0 ** -8


def _case(dev, M, N, K, r, base_n, g, G, seed=0):
    gen = torch.Generator().manual_seed(seed)
    mk = lambda *s, std=1.0: (torch.randn(*s, generator=gen) * std).bfloat16().to(dev)  # noqa: E731
    x, w, a, b = mk(M, K), mk(base_n, K, std=K ** -0.5), mk(G * r, K, std=K ** -0.5), mk(G * N, r, std=0.1)
    c = torch.arange(N, device=dev)
    rows = c // (N // g) * (base_n // g) + c % (base_n // g)
    xd, wd = x.double(), w.double()
    yb, mag = (xd @ wd.t())[:, rows], (xd.abs() @ wd.abs().t())[:, rows]
    want, tol = [], []
    for j in range(G):
        t = 2.0 * xd @ a[j * r:(j + 1) * r].double().t()
        bj = b[j * N:(j + 1) * N].double()
        y = yb + t @ bj.t()
        lora = t.abs() @ bj.abs().t()
        want.append(y)
        tol.append(1.01 * (U * y.abs() + U * (1 + U) * lora) + 2.0 ** -16 * (mag + lora))
    return x, w, a, b, torch.cat(want, 1), torch.cat(tol, 1)


def _check(y, want, tol):
    err = (y.double() - want).abs()
    assert bool((err <= tol).all()), float((err / tol).max())


@pytest.mark.parametrize("M,N,K,r,base_n,g,G", [
    (4097, 1096, 1024, 32, 1096, 1, 3),   # one row and 8 (72) columns past whole tiles of either width
    (2049, 4096, 1088, 80, 1024, 128, 2), # templates 8 wide, four heads each; ranks 64 + 16; one wave of tiles
    (4200, 2176, 1024, 16, 1088, 2, 2),   # two heads a template, the smallest rank
    (2048, 8192, 1024, 128, 1024, 4, 1),  # one group, eight heads, two whole rank chunks
    (8192, 1024, 1024, 48, 1024, 1, 2),   # on the line: the fewest multiply-adds saved
])
def test_shared_base_once(gpu, M, N, K, r, base_n, g, G):
    print(f"[shared base] M={M} N={N} K={K} r={r} base_n={base_n} g={g} groups={G}", flush=True)
    assert (G * N // base_n - 1) * M * base_n * K >= 1 << 33
    x, w, a, b, want, tol = _case(gpu, M, N, K, r, base_n, g, G, seed=M)
    y = ops.lora_linear_bcast_op(x, w, None, a, b, 2.0, g, G)
    _check(y, want, tol)
    assert torch.equal(y, ops.lora_linear_bcast_op(x, w, None, a, b, 2.0, g, G))


def _call(x, w, a, b, y, M, N, K, r, base_n, g, G, ws, nbytes):
    rc = _native.lib().wsl_lora_linear_bcast_fwd(
        x.data_ptr(), K, w.data_ptr(), K, 0, None, a.data_ptr(), K, b.data_ptr(), r, ctypes.c_float(2.0),
        y.data_ptr(), y.stride(0), M, N, K, r, base_n, g, G, ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream)
    assert rc == _native.WSL_OK, _native.last_error()


def test_shared_base_rows(gpu):
    """Output rows 8 bytes apart from 16-byte steps, nothing written past them."""
    M, N, K, r, base_n, g, G = 4097, 1096, 1024, 16, 1096, 1, 3
    print("[shared base] C entry, rows off 16 bytes", flush=True)
    x, w, a, b, want, tol = _case(gpu, M, N, K, r, base_n, g, G, seed=3)
    nbytes = _native.bcast_workspace_bytes(M, N, K, r, G, 0)
    y = torch.full((M, G * N + 4), 7.0, dtype=torch.bfloat16, device=gpu)
    _call(x, w, a, b, y, M, N, K, r, base_n, g, G, torch.zeros(nbytes, dtype=torch.uint8, device=gpu), nbytes)
    _check(y[:, :G * N], want, tol)
    assert bool((y[:, G * N:] == 7.0).all())


@pytest.mark.parametrize("M,N,K,r,base_n,g,G", [(4200, 2176, 1024, 16, 1088, 2, 2), (8192, 4096, 1024, 32, 1024, 1, 1)])
def test_shared_base_without_room_for_t(gpu, M, N, K, r, base_n, g, G):
    """In the grouped query's workspace T of all groups does not fit (at G r <= 32 no other form wants it
    there): the launch over the output columns runs, whose T stays in its tiles and leaves the scratch alone."""
    print(f"[shared base] M={M} N={N} r={r} groups={G}: the grouped query's workspace", flush=True)
    x, w, a, b, want, tol = _case(gpu, M, N, K, r, base_n, g, G, seed=M)
    assert (G * N // base_n - 1) * M * base_n * K >= 1 << 33
    full, small = _native.bcast_workspace_bytes(M, N, K, r, G, 0), _native.grouped_workspace_bytes(M, K, r, [N] * G, 0)
    assert small < full
    for nbytes, once in ((full, True), (small, False)):
        y = torch.zeros(M, G * N, dtype=torch.bfloat16, device=gpu)
        ws = torch.zeros(full, dtype=torch.uint8, device=gpu)
        _call(x, w, a, b, y, M, N, K, r, base_n, g, G, ws, nbytes)
        _check(y, want, tol)
        assert bool(ws[65536:].any()) is once
