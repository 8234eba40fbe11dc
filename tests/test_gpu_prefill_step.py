"""The prompt kernels between the fused projections (wsl::kv_norm_rope, wsl::prefill_attention,
wsl::swiglu_pair) against plain fp32 torch, at the edges of their tiles: 32 query rows a wave, 64
keys a tile, one to four heads of a kv group per workgroup, two or four waves; and the model's
inference forward on them against its torch-op forward and the oracle."""
import sys

import pytest
import torch

from oracle import qwen3_ref as Q

pytestmark = pytest.mark.gpu

# bf16 rounding (2^-9 relative) of the rotated q and k, of the probabilities and of the output
TOL = 1e-2


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def rel(x, ref):
    return ((x.float() - ref).abs().max() / ref.abs().max()).item()


def norm_rope(x, w, eps, rope):
    """x [b, s, heads, hd] fp32 normed over hd and rotated by rope rows 0..s-1."""
    s, hd = x.shape[1], x.shape[3]
    n = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w
    rot = torch.cat((-n[..., hd // 2:], n[..., :hd // 2]), -1)
    return n * rope[:s, None, :hd] + rot * rope[:s, None, hd:]


def inputs(gpu, b, s, nh, nkv, hd, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *sh: torch.randn(*sh, device=gpu, generator=g)  # noqa: E731
    q, k, v = r(b * s, nh * hd).bfloat16(), r(b * s, nkv * hd).bfloat16(), r(b * s, nkv * hd).bfloat16()
    qw, kw = (1 + 0.2 * r(hd)).bfloat16(), (1 + 0.2 * r(hd)).bfloat16()
    ang = r(s + 3, hd) * 3  # every element of a row its own angle
    return q, k, v, qw, kw, torch.cat((ang.cos(), ang.sin()), -1).contiguous()


CASES = [
    # b, seq, heads, kv heads, head_dim, cache positions past seq
    (1, 1, 2, 1, 128, 0),
    (2, 2, 4, 2, 64, 5),
    (3, 31, 4, 4, 128, 1),     # one head per workgroup
    (1, 33, 8, 2, 64, 0),      # one row past a wave
    (2, 63, 4, 2, 128, 9),
    (2, 64, 6, 2, 64, 0),      # three heads per kv head
    (1, 65, 8, 1, 128, 3),     # one key past a tile, eight heads per kv head
    (4, 129, 16, 4, 64, 0),    # four heads per workgroup
    (5, 200, 16, 4, 128, 24),
    (8, 257, 16, 8, 128, 0),   # the benchmark model's heads, four waves
    (2, 700, 5, 5, 128, 1),
    (1, 1000, 16, 8, 128, 0),
]


@pytest.mark.parametrize("b,s,nh,nkv,hd,extra", CASES)
def test_prompt_attention(gpu, b, s, nh, nkv, hd, extra):
    from weightshared_torchtitan_amd import ops
    _say(f"[prompt attention] b={b} s={s} heads={nh}/{nkv} hd={hd}")
    q, k, v, qw, kw, rope = inputs(gpu, b, s, nh, nkv, hd, 31 * s + nh)
    kc = torch.full((b, nkv, s + extra, hd), float("nan"), device=gpu, dtype=torch.bfloat16)
    vc = torch.full_like(kc, float("nan"))  # past the prompt: neither read nor written
    ops.kv_norm_rope_op(k, v, kw, 1e-6, rope, kc, vc)
    kr = norm_rope(k.float().view(b, s, nkv, hd), kw.float(), 1e-6, rope).transpose(1, 2)
    assert rel(kc[:, :, :s], kr) <= 2 ** -8  # one rounding to bf16, and fp32 sums in another order
    assert torch.equal(vc[:, :, :s], v.view(b, s, nkv, hd).transpose(1, 2))
    assert bool(kc[:, :, s:].isnan().all()) and bool(vc[:, :, s:].isnan().all())
    out = ops.prefill_attention_op(q, qw, 1e-6, rope, kc, vc, nh, hd ** -0.5)
    assert torch.equal(out, ops.prefill_attention_op(q, qw, 1e-6, rope, kc, vc, nh, hd ** -0.5))
    qr = norm_rope(q.float().view(b, s, nh, hd), qw.float(), 1e-6, rope).transpose(1, 2)
    rep = nh // nkv
    kk = kr.repeat_interleave(rep, 1).transpose(2, 3).contiguous()
    vv = v.float().view(b, s, nkv, hd).transpose(1, 2).repeat_interleave(rep, 1).contiguous()
    sc = torch.matmul(qr.contiguous(), kk) * hd ** -0.5
    sc = sc.masked_fill(~torch.ones(s, s, dtype=torch.bool, device=gpu).tril(), float("-inf"))
    ref = torch.matmul(sc.softmax(-1), vv).transpose(1, 2).reshape(b * s, nh * hd)
    assert rel(out, ref) <= TOL


def test_prompt_attention_strided_rows_and_large_scores(gpu):
    """q, k and v as column blocks of one grouped projection; norm weights that make the softmax
    peaked (scores of some hundreds), so a wrong running maximum overflows."""
    from weightshared_torchtitan_amd import ops
    b, s, nh, nkv, hd = 2, 150, 4, 2, 128
    _say("[prompt attention] strided, large scores")
    q, k, v, qw, kw, rope = inputs(gpu, b, s, nh, nkv, hd, 77)
    qkv = torch.cat((q, k, v), 1)
    q2, k2, v2 = qkv.split([nh * hd, nkv * hd, nkv * hd], -1)
    res = []
    for w in (1.0, 8.0):
        for qq, k_, v_ in ((q, k, v), (q2, k2, v2)):
            kc = torch.empty(b, nkv, s, hd, device=gpu, dtype=torch.bfloat16)
            vc = torch.empty_like(kc)
            ops.kv_norm_rope_op(k_, v_, kw * w, 1e-6, rope, kc, vc)
            res.append(ops.prefill_attention_op(qq, qw * w, 1e-6, rope, kc, vc, nh, hd ** -0.5))
    assert torch.equal(res[0], res[1]) and torch.equal(res[2], res[3])
    assert bool(res[2].isfinite().all())


@pytest.mark.parametrize("rows,ffn", [(1, 8), (3, 64), (300, 3072)])
def test_swiglu_pair_equals_swiglu(gpu, rows, ffn):
    from weightshared_torchtitan_amd import ops
    _say(f"[swiglu pair] rows={rows} ffn={ffn}")
    g = torch.Generator(device="cuda").manual_seed(ffn)
    gu = torch.randn(rows, 2 * ffn, device=gpu, generator=g).bfloat16()
    want = ops.swiglu_op(gu)
    assert torch.equal(ops.swiglu_pair_op(gu[:, :ffn], gu[:, ffn:]), want)
    assert torch.equal(ops.swiglu_pair_op(gu[:, :ffn].contiguous(), gu[:, ffn:].contiguous()), want)


def test_prompt_ops_refuse_bad_operands(gpu):
    from weightshared_torchtitan_amd import ops
    q, k, v, qw, kw, rope = inputs(gpu, 2, 4, 4, 2, 64, 5)
    kc = torch.zeros(2, 2, 8, 64, device=gpu, dtype=torch.bfloat16)
    args = (k, v, kw, 1e-6, rope, kc, kc.clone())
    for i, bad in ((0, k[:, :64]), (2, kw[:32]), (4, rope[:3]), (4, rope.bfloat16()), (5, kc.transpose(0, 1)), (5, kc.float()),
                   (5, kc[:, :, :3].contiguous()), (6, kc[:1])):
        with pytest.raises((ValueError, TypeError)):
            ops.kv_norm_rope_op(*[bad if j == i else t for j, t in enumerate(args)])
    for n_heads, scale in ((3, 0.1), (4, 0.0)):
        with pytest.raises(ValueError):
            ops.prefill_attention_op(q, qw, 1e-6, rope, kc, kc, n_heads, scale)


@pytest.mark.parametrize("b,s,grouped,cached", [(2, 12, False, True), (3, 70, True, True), (2, 65, False, False)])
def test_model_forward_fused_matches_torch_ops_and_oracle(gpu, b, s, grouped, cached):
    from weightshared_torchtitan_amd.qwen3_shared import KVCache, SharedQwen3, SharedQwen3Args
    _say(f"[model forward] b={b} s={s} grouped={grouped} cached={cached}")
    a = SharedQwen3Args(dim=256, n_layers=4, n_unique_blocks=2, n_heads=4, n_kv_heads=2, head_dim=64, hidden_dim=512,
                        vocab_size=1000, embed_rank=64, lora_rank=16, max_seq_len=128)
    m = SharedQwen3(a)
    m.init_random(seed=9, std=0.05)
    m = m.to(gpu).to(torch.bfloat16)
    m.prefill_grouped = grouped
    p = {k: v.detach().float().cpu() for k, v in m.named_parameters()}
    toks = torch.randint(0, a.vocab_size, (b, s), generator=torch.Generator().manual_seed(s))
    ref = Q.reference_forward(p, a, toks)
    got = {}
    with torch.no_grad():
        for fused in (True, False):
            m.prefill_fusion = fused
            cache = KVCache(a, b, s + 4, gpu) if cached else None
            assert m._prefill_fused_ok(toks.to(gpu), cache) is fused
            got[fused] = (m(toks.to(gpu), cache), cache)
        m.prefill_fusion = True
        assert not m._prefill_fused_ok(toks.to(gpu), KVCache(a, b, s - 1, gpu))
        h = m.norm.register_forward_hook(lambda *_: None)
        assert not m._prefill_fused_ok(toks.to(gpu), None)
        h.remove()
    assert not m._prefill_fused_ok(toks.to(gpu), None)  # gradients are recorded
    err = {f: rel(got[f][0].cpu(), ref) for f in got}
    _say(f"  max rel err fused {err[True]:.2e} torch ops {err[False]:.2e}")
    assert err[True] <= 3e-2
    if cached:
        for x, y in ((got[True][1].k, got[False][1].k), (got[True][1].v, got[False][1].v)):
            assert rel(x, y.float()) <= 3e-2
            assert not x[:, :, :, s:].any()


@pytest.mark.parametrize("compiled", [False, True])
@pytest.mark.parametrize("what", ["norm", "q norm", "k norm", "rope", "cache"])
def test_model_forward_with_operands_off_16_bytes(gpu, what, compiled):
    """Norm weights, a RoPE table or a cache in views that start off 16 bytes (a flat parameter buffer's,
    say) give what aligned ones give, eager and compiled into one graph."""
    from weightshared_torchtitan_amd.qwen3_shared import KVCache, SharedQwen3, SharedQwen3Args
    _say(f"[model forward] {what} off 16 bytes, compiled={compiled}")
    a = SharedQwen3Args(dim=128, n_layers=2, n_unique_blocks=1, n_heads=2, n_kv_heads=1, head_dim=64, hidden_dim=128,
                        vocab_size=300, embed_rank=64, lora_rank=8, max_seq_len=64)
    m = SharedQwen3(a)
    m.init_random(seed=2, std=0.05)
    m = m.to(gpu).to(torch.bfloat16)
    toks = torch.arange(40, device=gpu).view(2, 20)

    def off(t):  # the same values one element into a buffer of their own
        buf = torch.zeros(t.numel() + 1, dtype=t.dtype, device=t.device)
        buf[1:] = t.flatten()
        return buf[1:].view(t.shape)

    with torch.no_grad():
        cache = KVCache(a, 2, 24, gpu)
        assert m._prefill_fused_ok(toks, cache)
        want = m(toks, cache), cache.k, cache.v
        cache = KVCache(a, 2, 24, gpu)
        blk = m.base_blocks[0]
        if what == "cache":
            cache.k, cache.v = off(cache.k), off(cache.v)
        elif what == "rope":
            m.rope = off(m.rope.float())
        else:
            norm = {"norm": blk.ffn_norm, "q norm": blk.attention.q_norm, "k norm": blk.attention.k_norm}[what]
            norm.weight = torch.nn.Parameter(off(norm.weight.detach()))
        assert m._prefill_fused_ok(toks, cache)
        torch._dynamo.reset()
        got = (torch.compile(m, backend="eager", fullgraph=True) if compiled else m)(toks, cache)
    for x, y in zip((got, cache.k, cache.v), want):
        assert torch.equal(x, y)


def test_opcheck_prompt_ops(gpu):
    from weightshared_torchtitan_amd import ops  # noqa: F401
    utils = ("test_schema", "test_faketensor", "test_aot_dispatch_dynamic")
    q, k, v, qw, kw, rope = inputs(gpu, 2, 40, 4, 2, 64, 6)
    kc = torch.zeros(2, 2, 48, 64, device=gpu, dtype=torch.bfloat16)
    torch.library.opcheck(torch.ops.wsl.kv_norm_rope.default, (k, v, kw, 1e-6, rope, kc, kc.clone()), test_utils=utils)
    torch.library.opcheck(torch.ops.wsl.prefill_attention.default, (q, qw, 1e-6, rope, kc, kc, 4, 0.125), test_utils=utils)
    torch.library.opcheck(torch.ops.wsl.swiglu_pair.default, (q, q * 2), test_utils=utils)
