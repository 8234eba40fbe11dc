"""The workloads that the kernels of this repository are timed on.

Each case is one call, or one training step, of what a program built on the framework runs:
fused LoRA linears from one decode token to a full prefill batch, bf16 and fp8 base weights,
the forward and backward of LoRA fine-tuning and of full training, the shared-base
projections, and two whole calls of the weight-shared Qwen3 model (a prompt and a decode
step). Projection widths are those of Qwen3-0.6B, 1.7B and 8B, the configurations that
``bench.py`` and the tests use; inputs follow them too (x ~ N(0, 1), weights ~ N(0, 0.02^2),
LoRA B non-zero).

    listed()            the named cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what a program holds before the call
    run(state)          one pass, and all its outputs
    work(case)          bytes and operations that the pass cannot do without
    tolerance(case)     how far another correct implementation's outputs may be
    exact(case, seed)   the outputs in 64-bit arithmetic, in plain torch
"""
from __future__ import annotations

import math

import torch

import weightshared_torchtitan_amd as wsl
from weightshared_torchtitan_amd import ops
from weightshared_torchtitan_amd.qwen3_shared import KVCache, SharedQwen3, SharedQwen3Args

DEV = "cuda:0"
FP8_MAX = 448.0

# (N, K) of the projections, and the widths of their grouped launches
Q06 = {"q": (2048, 1024), "kv": (1024, 1024), "o": (1024, 2048), "gate": (3072, 1024), "down": (1024, 3072)}
Q17 = {"q": (2048, 2048), "kv": (1024, 2048), "gate": (6144, 2048), "down": (2048, 6144)}
Q8 = {"q": (4096, 4096), "kv": (1024, 4096), "gate": (12288, 4096), "down": (4096, 12288)}
GROUPS = {"0.6B qkv": ((2048, 1024, 1024), 1024), "0.6B gate_up": ((3072, 3072), 1024),
          "1.7B qkv": ((2048, 1024, 1024), 2048), "1.7B gate_up": ((6144, 6144), 2048),
          "8B qkv": ((4096, 1024, 1024), 4096), "8B gate_up": ((12288, 12288), 4096)}


def listed():
    return [
        # one token of interactive decoding through one projection: latency
        {"name": "decode_1", "kind": "linear", "M": 1, "N": 2048, "K": 2048, "r": 64, "fp8": False},
        # a decode batch through gate|up, stacked in one launch as a serving loop does
        {"name": "decode_32_gate_up", "kind": "grouped", "M": 32, "group": "1.7B gate_up", "r": 64, "fp8": False},
        # a decode batch on the fp8 base of the 8B model, its longest reduction
        {"name": "decode_16_fp8_down", "kind": "linear", "M": 16, "N": 4096, "K": 12288, "r": 128, "fp8": True},
        # a short prompt, or a chunk of one, of ragged length
        {"name": "chunk_200_down", "kind": "linear", "M": 200, "N": 2048, "K": 6144, "r": 64, "fp8": False},
        # the same on the fp8 base, q|k|v stacked
        {"name": "chunk_333_fp8_qkv", "kind": "grouped", "M": 333, "group": "8B qkv", "r": 128, "fp8": True},
        # a full prefill batch, q|k|v stacked (the benchmark's shape)
        {"name": "prefill_8192_qkv", "kind": "grouped", "M": 8192, "group": "0.6B qkv", "r": 32, "fp8": False},
        # LoRA fine-tuning: frozen base, gradients of the input and the two factors
        {"name": "finetune_4096_gate", "kind": "train", "M": 4096, "N": 6144, "K": 2048, "r": 16, "frozen": True},
        # full training of a projection: every gradient
        {"name": "train_8192_down", "kind": "train", "M": 8192, "N": 1024, "K": 3072, "r": 32, "frozen": False},
        # a training step of q|k|v on one shared base (the reference's qkv sharing)
        {"name": "shared_qkv_train", "kind": "shared", "M": 4096, "N": 2048, "base_n": 2048, "g": 1, "groups": 3,
         "K": 2048, "r": 32},
        # a fine-tuning step of a model of other widths and rank, none of them on a tile grid
        {"name": "ragged_finetune", "kind": "train", "M": 777, "N": 1500, "K": 1000, "r": 12, "frozen": True},
        # a batch of prompts through the weight-shared model: logits and the filled cache
        {"name": "model_prefill", "kind": "model_prefill", "batch": 8, "seq": 512},
        # one decode step of the same model, captured as generate() captures it
        {"name": "model_decode", "kind": "model_decode", "batch": 8, "pos": 640},
    ]


# ------------------------------------------------------------------------------------- draws
def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode_fp8", "chunk", "chunk", "chunk_fp8", "prefill", "finetune",
                       "finetune", "train", "shared", "ragged", "model_prefill", "model_decode"])
    wide = list(Q06.values()) + list(Q17.values())
    if kind in ("decode", "chunk", "prefill"):
        lo, hi = {"decode": (1, 64), "chunk": (65, 1024), "prefill": (1025, 8192)}[kind]
        M, r = _log_int(rng, lo, hi), rng.choice([0, 8, 16, 32, 64, 128])
        if rng.random() < 0.5:
            return {"kind": "grouped", "M": M, "group": rng.choice(sorted(GROUPS)[:4]), "r": r, "fp8": False}
        N, K = rng.choice(wide)
        return {"kind": "linear", "M": M, "N": N, "K": K, "r": r, "fp8": False}
    if kind in ("decode_fp8", "chunk_fp8"):
        M = _log_int(rng, 1, 64) if kind == "decode_fp8" else _log_int(rng, 65, 2048)
        r = rng.choice([16, 64, 128])
        if rng.random() < 0.5:
            return {"kind": "grouped", "M": M, "group": rng.choice(sorted(GROUPS)[4:]), "r": r, "fp8": True}
        N, K = rng.choice(list(Q8.values()))
        return {"kind": "linear", "M": M, "N": N, "K": K, "r": r, "fp8": True}
    if kind in ("finetune", "train"):
        N, K = rng.choice(wide)
        return {"kind": "train", "M": _log_int(rng, 128, 8192), "N": N, "K": K, "r": rng.choice([4, 8, 16, 32, 64]),
                "frozen": kind == "finetune"}
    if kind == "shared":
        groups, per, g = rng.choice([(1, 2, 2), (1, 2, 4), (2, 1, 1), (3, 1, 1)])
        base_n = rng.choice([1024, 2048])
        return {"kind": "shared", "M": _log_int(rng, 128, 4096), "N": base_n * per, "base_n": base_n, "g": g,
                "groups": groups, "K": rng.choice([1024, 2048]), "r": rng.choice([8, 16, 32, 64])}
    if kind == "ragged":
        return {"kind": "train", "M": _log_int(rng, 64, 1024), "N": rng.randint(200, 2000), "K": rng.randint(200, 2000),
                "r": rng.randint(2, 32), "frozen": rng.random() < 0.5}
    if kind == "model_prefill":
        batch = rng.randint(1, 8)
        return {"kind": kind, "batch": batch, "seq": _log_int(rng, 16, min(1000, 4096 // batch))}
    return {"kind": kind, "batch": rng.randint(1, 32), "pos": _log_int(rng, 16, 1000)}


# ------------------------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(gen, *shape, std=1.0):
    return (torch.randn(*shape, generator=gen, device=DEV) * std).bfloat16()


def _quantize(w):
    """e4m3 codes and one fp32 scale per row, the largest magnitude of a row on 448."""
    wf = w.float()
    s = wf.abs().amax(1) / FP8_MAX
    return (wf / s[:, None]).clamp(-FP8_MAX, FP8_MAX).to(torch.float8_e4m3fn), s


def _linear_inputs(case, seed):
    g = _gen(seed)
    gn, K = (GROUPS[case["group"]] if case["kind"] == "grouped" else ((case["N"],), case["K"]))
    N, r = sum(gn), case["r"]
    t = {"x": _randn(g, case["M"], K), "w": _randn(g, N, K, std=0.02), "ws": None, "a": None, "b": None,
         "gn": list(gn), "scale": 2.0}
    if r:
        t["a"] = _randn(g, len(gn) * r, K, std=0.02)
        t["b"] = _randn(g, N, r, std=0.02)
    if case.get("fp8"):
        t["w"], t["ws"] = _quantize(t["w"])
        t["scale"] = 1.0
    return t


def _train_inputs(case, seed):
    g = _gen(seed)
    M, N, K, r, G = case["M"], case["N"], case["K"], case["r"], case.get("groups", 1)
    return {"x": _randn(g, M, K), "w": _randn(g, case.get("base_n", N), K, std=0.02), "a": _randn(g, G * r, K, std=0.02),
            "b": _randn(g, G * N, r, std=0.02), "gy": _randn(g, M, G * N), "scale": 2.0}


def _model_args():
    return SharedQwen3Args()  # Qwen3-0.6B widths, 28 layers from 4 unique blocks, rank 32


def _model_weights(seed):
    """Name -> bf16 tensor, under the model's own parameter names."""
    a, g, w = _model_args(), _gen(seed), {}
    # an embedding whose rows are of the residual stream's size, as a trained one's are (0.02
    # would let the first layers outweigh it, and magnify every rounding of theirs)
    w["tok_embeddings.emb"] = _randn(g, a.vocab_size, a.embed_rank, std=0.5)
    w["tok_embeddings.proj.weight"] = _randn(g, a.dim, a.embed_rank, std=0.0625)
    sub = lambda n: "attention" if n in ("wq", "wk", "wv", "wo") else "feed_forward"  # noqa: E731
    for i in range(a.n_unique_blocks):
        p = f"base_blocks.{i}."
        for n, (out, inp) in a.proj_shapes().items():
            w[f"{p}{sub(n)}.{n}.weight"] = _randn(g, out, inp, std=0.02)
        for n, d in (("attention.q_norm", a.head_dim), ("attention.k_norm", a.head_dim), ("attention_norm", a.dim),
                     ("ffn_norm", a.dim)):
            w[f"{p}{n}.weight"] = (1 + 0.1 * torch.randn(d, generator=g, device=DEV)).bfloat16()
    for i in range(a.n_layers):
        for n, (out, inp) in a.proj_shapes().items():
            w[f"layer_loras.{i}.{n}.w_a.weight"] = _randn(g, a.lora_rank, inp, std=0.02)
            w[f"layer_loras.{i}.{n}.w_b.weight"] = _randn(g, out, a.lora_rank, std=0.02)
    w["norm.weight"] = (1 + 0.1 * torch.randn(a.dim, generator=g, device=DEV)).bfloat16()
    return w


def _model_inputs(case, seed):
    a = _model_args()
    w = _model_weights(seed)
    g = _gen(seed + 1_000_003)
    if case["kind"] == "model_prefill":
        return a, w, torch.randint(0, a.vocab_size, (case["batch"], case["seq"]), generator=g, device=DEV), None, None
    token = torch.randint(0, a.vocab_size, (case["batch"], 1), generator=g, device=DEV)
    shape = (a.n_layers, case["batch"], a.n_kv_heads, case["pos"], a.head_dim)
    return a, w, token, _randn(g, *shape), _randn(g, *shape, std=0.6)  # normed keys; values of x . W_v^T


def _build_model(a, w):
    with torch.device(DEV):
        model = SharedQwen3(a).to(torch.bfloat16)
    params = dict(model.named_parameters())
    if set(params) != set(w):
        raise ValueError("the model's parameters have other names")
    with torch.no_grad():
        for n, p in params.items():
            p.copy_(w[n])
    return model


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("linear", "grouped"):
        return {"kind": kind, **_linear_inputs(case, seed)}
    if kind in ("train", "shared"):
        t = _train_inputs(case, seed)
        if kind == "shared":
            for n in ("x", "w", "a", "b"):
                t[n].requires_grad_()
            return {"kind": kind, "g": case["g"], "groups": case["groups"], **t}
        base = torch.nn.Linear(case["K"], case["N"], bias=False, device="meta")
        base.weight = torch.nn.Parameter(t["w"], requires_grad=not case["frozen"])
        lora = wsl.LoRAModule(case["K"], case["N"], rank=case["r"], device="meta")
        lora.w_a.weight, lora.w_b.weight = torch.nn.Parameter(t["a"]), torch.nn.Parameter(t["b"])
        wrt = [t["x"].requires_grad_(), lora.w_a.weight, lora.w_b.weight] + ([] if case["frozen"] else [base.weight])
        return {"kind": kind, "module": wsl.LoRALinear(base, lora), "x": t["x"], "gy": t["gy"], "wrt": wrt}
    a, w, tokens, past_k, past_v = _model_inputs(case, seed)
    model = _build_model(a, w)
    if kind == "model_prefill":
        return {"kind": kind, "model": model, "tokens": tokens, "cache": KVCache(a, case["batch"], case["seq"] + 16, DEV)}
    cache = KVCache(a, case["batch"], a.max_seq_len, DEV)
    cache.k[:, :, :, :case["pos"]] = past_k
    cache.v[:, :, :, :case["pos"]] = past_v
    pos = torch.full((), case["pos"], dtype=torch.int64, device=DEV)
    with torch.no_grad():  # one step captured, as generate() does: warm up on the capture stream first
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            model.decode_step(tokens, pos, cache)
        torch.cuda.current_stream().wait_stream(stream)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            logits = model.decode_step(tokens, pos, cache)
    return {"kind": kind, "model": model, "tokens": tokens, "pos": pos, "cache": cache, "graph": graph, "logits": logits,
            "at": case["pos"]}


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return wsl.lora_linear(state["x"], state["w"], state["a"], state["b"], state["scale"], w_scale=state["ws"])
    if kind == "grouped":
        return ops.lora_linear_grouped_op(state["x"], state["w"], state["ws"], state["a"], state["b"], state["scale"],
                                          state["gn"])
    if kind == "train":
        y = state["module"](state["x"])
        return [y, *torch.autograd.grad(y, state["wrt"], state["gy"])]
    if kind == "shared":
        y = ops.lora_linear_bcast_op(state["x"], state["w"], None, state["a"], state["b"], state["scale"], state["g"],
                                     state["groups"])
        return [y, *torch.autograd.grad(y, [state["x"], state["a"], state["b"], state["w"]], state["gy"])]
    if kind == "model_prefill":
        cache = state["cache"]
        with torch.no_grad():
            logits = state["model"](state["tokens"], cache)
        return {"logits": logits, "k": cache.k, "v": cache.v}
    state["graph"].replay()
    at, cache = state["at"], state["cache"]
    return {"logits": state["logits"], "k": cache.k[:, :, :, at], "v": cache.v[:, :, :, at]}


# -------------------------------------------------------------------------------------- work
def work(case):
    kind = case["kind"]
    if kind in ("linear", "grouped"):
        gn, K = (GROUPS[case["group"]] if kind == "grouped" else ((case["N"],), case["K"]))
        M, N, r, G = case["M"], sum(gn), case["r"], len(gn)
        return {"bytes": N * K * (1 if case["fp8"] else 2) + (4 * N if case["fp8"] else 0)
                + 2 * (M * K + M * N + r * (G * K + N)), "flops": 2 * M * (N * K + r * (G * K + N))}
    if kind in ("train", "shared"):
        M, N, K, r, G = case["M"], case["N"], case["K"], case["r"], case.get("groups", 1)
        base_n = case.get("base_n", N)
        dw = kind == "shared" or not case["frozen"]
        # x, gy in and y, dx out; w, a, b in and their gradients out
        nbytes = 2 * (2 * M * K + 2 * M * G * N + base_n * K * (2 if dw else 1) + 2 * G * r * (K + N))
        # the expanded base is multiplied once per template row, as are its gradients
        flops = 2 * M * base_n * K * (3 if dw else 2) + 2 * M * G * r * (K + N) * 3
        return {"bytes": nbytes, "flops": flops}
    a = _model_args()
    per_block = sum(o * i for o, i in a.proj_shapes().values())
    per_lora = sum(a.lora_rank * (o + i) for o, i in a.proj_shapes().values())
    head = a.embed_rank * (a.dim + a.vocab_size)
    kv_row = a.n_layers * 2 * a.n_kv_heads * a.head_dim  # elements of one position's k and v
    weights = a.n_unique_blocks * per_block + a.n_layers * per_lora
    if kind == "model_prefill":
        T, s = case["batch"] * case["seq"], case["seq"]
        attn = a.n_layers * case["batch"] * a.n_heads * 2 * a.head_dim * s * (s + 1)  # causal q.k and p.v
        return {"bytes": 2 * (weights + head + T * (kv_row + a.vocab_size)),
                "flops": 2 * T * (a.n_layers * (per_block + per_lora) + head) + attn}
    b, L = case["batch"], case["pos"] + 1
    attn = a.n_layers * b * a.n_heads * 4 * a.head_dim * L
    return {"bytes": 2 * (weights + head + b * (kv_row * L + a.vocab_size)),
            "flops": 2 * b * (a.n_layers * (per_block + per_lora) + head) + attn}


def tolerance(case):
    # bf16 outputs of fp32 sums are 1.7e-3 (one rounding) to 2.6e-3 (T rounded to bf16 as well)
    # from the 64-bit result; the two-term fp8 activations about the same. In the model the
    # roundings of 28 layers add up.
    return {"rel": {"model_prefill": 0.03, "model_decode": 0.03}.get(case["kind"], 0.01)}


# --------------------------------------------------------------------------- 64-bit reference
def _expand_rows(base_n, N, g, device):
    """Base row of every output column of one shared projection (g templates of base_n / g rows)."""
    c, d = torch.arange(N, device=device), base_n // g
    return c // ((N // base_n) * d) * d + c % d


def exact(case, seed):
    kind = case["kind"]
    if kind in ("linear", "grouped"):
        t = _linear_inputs(case, seed)
        x, w = t["x"].double(), t["w"].double()
        if t["ws"] is not None:
            w = w * t["ws"].double()[:, None]
        y = x @ w.t()
        if t["a"] is not None:
            r, n0 = case["r"], 0
            for j, n in enumerate(t["gn"]):
                y[:, n0:n0 + n] += t["scale"] * (x @ t["a"][j * r:(j + 1) * r].double().t()) @ t["b"][n0:n0 + n].double().t()
                n0 += n
        return y
    if kind in ("train", "shared"):
        t = _train_inputs(case, seed)
        x, w, a, b, gy, s = t["x"].double(), t["w"].double(), t["a"].double(), t["b"].double(), t["gy"].double(), t["scale"]
        N, r, G = case["N"], case["r"], case.get("groups", 1)
        rows = _expand_rows(case.get("base_n", N), N, case.get("g", 1), DEV)
        y, dx, dw = [], torch.zeros_like(x), torch.zeros_like(w)
        da, db = torch.empty_like(a), torch.empty_like(b)
        for j in range(G):
            aj, bj, gj = a[j * r:(j + 1) * r], b[j * N:(j + 1) * N], gy[:, j * N:(j + 1) * N]
            y.append(x @ w[rows].t() + s * (x @ aj.t()) @ bj.t())
            u = gj @ bj
            dx += gj @ w[rows] + s * u @ aj
            dw.index_add_(0, rows, gj.t() @ x)
            da[j * r:(j + 1) * r] = s * u.t() @ x
            db[j * N:(j + 1) * N] = s * gj.t() @ (x @ aj.t())
        out = [torch.cat(y, 1), dx, da, db]
        return out + ([dw] if kind == "shared" or not case["frozen"] else [])
    return _model_exact(case, seed)


def _model_exact(case, seed):
    a, w, tokens, past_k, past_v = _model_inputs(case, seed)
    W = lambda n: w[n + ".weight"].double()  # noqa: E731
    b, s = tokens.shape
    p0 = 0 if past_k is None else case["pos"]
    hd, rep = a.head_dim, a.n_heads // a.n_kv_heads
    t = torch.arange(p0, p0 + s, device=DEV, dtype=torch.float64)
    # the frequencies are the model's 32-bit table, their angles in 64 bits
    f = 1.0 / (a.rope_theta ** (torch.arange(0, hd, 2, device=DEV).float() / hd)).double()
    ang = torch.outer(t, f).repeat(1, 2)[:, None]
    cos, sin = ang.cos(), ang.sin()

    def norm(x, n):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + a.norm_eps) * W(n)

    def rope(x):
        return x * cos + torch.cat((-x[..., hd // 2:], x[..., :hd // 2]), -1) * sin

    E = w["tok_embeddings.emb"].double()
    P = W("tok_embeddings.proj")
    h = E[tokens] @ P.t()
    mask = torch.ones(s, p0 + s, dtype=torch.bool, device=DEV).tril(p0)
    ks, vs = [], []
    for l in range(a.n_layers):
        blk, lo = f"base_blocks.{a.block_of(l)}.", f"layer_loras.{l}."

        def proj(x, n):
            sub = "attention" if n in ("wq", "wk", "wv", "wo") else "feed_forward"
            return x @ W(f"{blk}{sub}.{n}").t() + 2.0 * (x @ W(f"{lo}{n}.w_a").t()) @ W(f"{lo}{n}.w_b").t()

        x = norm(h, blk + "attention_norm")
        q = rope(norm(proj(x, "wq").view(b, s, -1, hd), blk + "attention.q_norm")).transpose(1, 2)
        k = rope(norm(proj(x, "wk").view(b, s, -1, hd), blk + "attention.k_norm")).transpose(1, 2)
        v = proj(x, "wv").view(b, s, -1, hd).transpose(1, 2)
        ks.append(k)
        vs.append(v)
        if p0:
            k = torch.cat((past_k[l].double(), k), 2)
            v = torch.cat((past_v[l].double(), v), 2)
        k, v = k.repeat_interleave(rep, 1), v.repeat_interleave(rep, 1)
        p = ((q @ k.transpose(2, 3).contiguous()) * hd ** -0.5).masked_fill(~mask, -math.inf).softmax(-1)
        h = h + proj((p @ v).transpose(1, 2).reshape(b, s, -1), "wo")
        x = norm(h, blk + "ffn_norm")
        h = h + proj(torch.nn.functional.silu(proj(x, "w1")) * proj(x, "w3"), "w2")
    logits = norm(h, "norm") @ P @ E.t()
    if p0:
        return {"logits": logits[:, 0], "k": torch.stack([k[:, :, 0] for k in ks]), "v": torch.stack([v[:, :, 0] for v in vs])}
    pad = lambda t: torch.nn.functional.pad(torch.stack(t), (0, 0, 0, 16))  # noqa: E731  (the cache's free positions)
    return {"logits": logits, "k": pad(ks), "v": pad(vs)}
