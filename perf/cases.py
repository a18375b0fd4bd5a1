"""The measured work of kvengine_amd: what a serving program has it do on one GPU.

A case is one pass of one of six kinds, over the Qwen2.5 0.5B (draft) and 3B
(target) architectures with seeded random weights:

  layers   forward_hidden over a few layers of a model: `seqs` sequences of
           `q` new tokens each on top of ragged histories (decode, verify)
  attn     the paged verify attention of a pass: one plan, then the launch of
           every layer
  prefill  forward_packed / forward_packed_wide: a batch of prompts admitted
           together
  prompt   forward_with_own_cache on one prompt in a fresh sequence
  step     forward_with_own_cache on one token of a whole model
  head     lmhead_argmax with the row maxima (and the runner-up, which the
           near-tie accounting asks for)

Decode and verify passes are captured once as a HIP graph and replayed, as
SpecEngine and speculative_greedy run them; prefills, the fp32 model and the
single-token API are issued eagerly, as they are there.
"""

import math
import random

import torch

from kvengine_amd import kernels
from kvengine_amd.arch import QWEN25_0_5B, QWEN25_3B, layer_slice
from kvengine_amd.forward import (forward_hidden, forward_packed, forward_packed_wide,
                                  forward_with_own_cache)
from kvengine_amd.model import build_model
from kvengine_amd.paged import DeviceKV, PagedKVCache

ARCHS = {"0.5b": QWEN25_0_5B, "3b": QWEN25_3B}
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
BS = 16  # tokens per block


def listed():
    return [
        # The draft's pass for a single live request: one token, the smallest
        # and most frequent launch sequence of a run.
        {"name": "draft_1", "kind": "layers", "arch": "0.5b", "dtype": "bf16", "layers": 4,
         "seqs": 1, "q": 1, "ctx_lo": 611, "ctx_hi": 611, "unit": 0, "kw": 0, "gemm_rows": 0,
         "graph": True, "spread": 1},
        # The draft's pass of the batched workload: 32 requests, ragged
        # histories of a few hundred tokens.
        {"name": "draft_32", "kind": "layers", "arch": "0.5b", "dtype": "bf16", "layers": 4,
         "seqs": 32, "q": 1, "ctx_lo": 48, "ctx_hi": 860, "unit": 0, "kw": 0, "gemm_rows": 0,
         "graph": True, "spread": 2},
        # The target's verify pass of one live request (k = 4: five tokens), on
        # the layer the engine takes at every width.
        {"name": "verify_1x5", "kind": "layers", "arch": "3b", "dtype": "bf16", "layers": 2,
         "seqs": 1, "q": 5, "ctx_lo": 600, "ctx_hi": 600, "unit": 8, "kw": 2, "gemm_rows": 160,
         "graph": True, "spread": 3},
        # The target's verify pass of the full batch: 32 x 5 rows.
        {"name": "verify_32x5", "kind": "layers", "arch": "3b", "dtype": "bf16", "layers": 2,
         "seqs": 32, "q": 5, "ctx_lo": 48, "ctx_hi": 860, "unit": 8, "kw": 2, "gemm_rows": 160,
         "graph": True, "spread": 4},
        # The same pass in fp32 (the parity configuration): four requests.
        {"name": "verify_fp32", "kind": "layers", "arch": "0.5b", "dtype": "fp32", "layers": 4,
         "seqs": 4, "q": 5, "ctx_lo": 200, "ctx_hi": 1500, "unit": 0, "kw": 0, "gemm_rows": 0,
         "graph": False, "spread": 5},
        # Verify attention on its own, 32 sequences of lognormal context: the
        # benchmark's attention roofline, four layers of it behind one plan.
        {"name": "attn_verify_32", "kind": "attn", "arch": "0.5b", "dtype": "bf16", "layers": 4,
         "seqs": 32, "q": 5, "ctx_lo": 64, "ctx_hi": 4096, "shared": 0, "unit": 0, "kw": 0,
         "graph": True, "spread": 6},
        # Verify attention of the prefix-shared workload near the end of its
        # contexts: 16 sequences behind a shared 2048-token prefix, k = 8.
        {"name": "attn_verify_long", "kind": "attn", "arch": "3b", "dtype": "bf16", "layers": 2,
         "seqs": 16, "q": 9, "ctx_lo": 7000, "ctx_hi": 8192, "shared": 2048, "unit": 16, "kw": 2,
         "graph": True, "spread": 7},
        # Admission of the batched workload's prompts into the target: 30
        # prompts of 16 to 1024 tokens in one packed forward.
        {"name": "prefill_30", "kind": "prefill", "arch": "3b", "layers": 2, "prompts": 30,
         "lo": 16, "hi": 1024, "median": 128, "unit": 8, "kw": 2, "spread": 8},
        # Admission of the prefix-shared workload's first prompts: a few long
        # prompts of a shared prefix's size, odd lengths.
        {"name": "prefill_long", "kind": "prefill", "arch": "3b", "layers": 2, "prompts": 2,
         "lo": 2303, "hi": 2305, "median": 2304, "unit": 16, "kw": 2, "spread": 9},
        # One prompt through the single-request API, the 0.5B's heads.
        {"name": "prompt_1777", "kind": "prompt", "arch": "0.5b", "layers": 4, "tokens": 1777},
        # One token of plain greedy decoding through the single-request API:
        # a whole model, every launch issued from the host.
        {"name": "greedy_step", "kind": "step", "arch": "0.5b", "tokens": 67},
        # The target's LM head + argmax over a full batch's verify rows.
        {"name": "head_160", "kind": "head", "arch": "3b", "dtype": "bf16", "rows": 160,
         "blocked": True, "second": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layers", "layers", "layers", "attn", "attn", "prefill", "prefill", "prompt",
                       "step", "head"])
    arch = rng.choice(["0.5b", "3b"])
    spread = rng.randrange(1000)
    if kind == "layers":
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp32"])
        if dtype == "fp32":
            arch = "0.5b"
        seqs = _log_int(rng, 1, 32)
        q = rng.choice([1, 2, 3, 5]) if arch == "3b" or dtype == "fp32" else rng.choice([1, 1, 2])
        hi = _log_int(rng, 60, 880)
        wide = arch == "3b"
        return {"kind": "layers", "arch": arch, "dtype": dtype, "layers": 2, "seqs": seqs, "q": q,
                "ctx_lo": max(1, hi // rng.choice([1, 4, 12])), "ctx_hi": hi,
                "unit": 8 if wide else 0, "kw": 2 if wide else 0, "gemm_rows": 160 if wide else 0,
                "graph": dtype == "bf16", "spread": spread}
    if kind == "attn":
        q = rng.choice([1, 2, 3, 5, 9])
        hi = _log_int(rng, 300, 8192)
        fixed = rng.random() < 0.5
        return {"kind": "attn", "arch": arch, "dtype": "bf16", "layers": 2,
                "seqs": _log_int(rng, 1, min(32, 131072 // hi)), "q": q,
                "ctx_lo": max(q, hi // rng.choice([1, 4, 16])), "ctx_hi": hi, "shared": 0,
                "unit": (16 if hi > 4096 else 8) if fixed else 0, "kw": 2 if fixed else 0,
                "graph": True, "spread": spread}
    if kind == "prefill":
        median = _log_int(rng, 40, 1500)
        hi = min(2 * median, 2300)
        wide = arch == "3b"
        return {"kind": "prefill", "arch": arch, "layers": 2, "lo": max(16, median // 4), "hi": hi,
                "median": median, "prompts": max(2, _log_int(rng, 2, max(3, 4600 // hi))),
                "unit": 8 if wide else 0, "kw": 2 if wide else 0, "spread": spread}
    if kind == "prompt":
        return {"kind": "prompt", "arch": arch, "layers": 2, "tokens": _log_int(rng, 20, 2400)}
    if kind == "step":
        return {"kind": "step", "arch": "0.5b", "tokens": _log_int(rng, 8, 300)}
    return {"kind": "head", "arch": arch, "dtype": "bf16", "rows": _log_int(rng, 1, 160),
            "blocked": arch == "3b", "second": rng.random() < 0.3}


# ---- inputs -------------------------------------------------------------------

def _arch(case):
    a = ARCHS[case["arch"]]
    return layer_slice(a, case["layers"]) if "layers" in case else a


def _lens(case):
    """History lengths (new tokens included) of an attention or layer pass:
    spread evenly over the logarithm of the range."""
    r = random.Random(case["spread"])
    return [_log_int(r, max(case["ctx_lo"], case["q"]), max(case["ctx_hi"], case["q"]))
            for _ in range(case["seqs"])]


def _prompt_lens(case):
    """Prompt lengths: lognormal around the median, longest first as the engine
    packs them."""
    r = random.Random(case["spread"])
    lens = [round(math.exp(r.gauss(math.log(case["median"]), 0.6))) for _ in range(case["prompts"])]
    return sorted((min(case["hi"], max(case["lo"], n)) for n in lens), reverse=True)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _weights(arch, dtype, g):
    """A state dict drawn on the GPU: linear weights, biases and the embedding
    N(0, 0.02), norm gains around 1."""
    def n(*shape):
        return (torch.randn(shape, generator=g, device="cuda") * 0.02).to(dtype)

    def gain():
        return (1 + 0.1 * torch.randn(arch.hidden, generator=g, device="cuda")).to(dtype)

    h, f, qd, kd = arch.hidden, arch.ffn, arch.q_dim, arch.kv_dim
    sd = {"model.embed_tokens.weight": n(arch.vocab, h)}
    for i in range(arch.num_layers):
        p = f"model.layers.{i}."
        for name, out, inp in (("self_attn.q_proj", qd, h), ("self_attn.k_proj", kd, h),
                               ("self_attn.v_proj", kd, h), ("self_attn.o_proj", h, qd),
                               ("mlp.gate_proj", f, h), ("mlp.up_proj", f, h),
                               ("mlp.down_proj", h, f)):
            sd[p + name + ".weight"] = n(out, inp)
        for name, out in (("q_proj", qd), ("k_proj", kd), ("v_proj", kd)):
            sd[p + f"self_attn.{name}.bias"] = n(out)
        sd[p + "input_layernorm.weight"] = gain()
        sd[p + "post_attention_layernorm.weight"] = gain()
    sd["model.norm.weight"] = gain()
    return sd


def _tables(lens, seed, shared=0, spare=1.25):
    """Block tables of sequences of `lens` tokens: physical blocks in random
    order, the first `shared` tokens' blocks common to all. (tables, pool size)"""
    common = shared // BS
    need = [-(-n // BS) for n in lens]
    total = common + sum(n - common for n in need)
    nb = math.ceil(spare * total) + 1
    ids = list(range(nb))
    random.Random(seed).shuffle(ids)
    head, at, out = ids[:common], common, []
    for n in need:
        out.append(head + ids[at:at + n - common])
        at += n - common
    return out, nb


def _device_tables(tables):
    t = torch.full((len(tables), max(map(len, tables))), -1, dtype=torch.int32)
    for i, ids in enumerate(tables):
        t[i, :len(ids)] = torch.tensor(ids, dtype=torch.int32)
    return t.cuda()


def _pools(arch, nb, dtype, g, scale):
    """K [L, NB, Hkv, 16, D] and V [L, NB, Hkv, D, 16] holding a history."""
    L, H, D = arch.num_layers, arch.num_kv_heads, arch.head_dim
    k = (torch.randn(L, nb, H, BS, D, generator=g, device="cuda") * scale).to(dtype)
    v = (torch.randn(L, nb, H, D, BS, generator=g, device="cuda") * scale).to(dtype)
    return k, v


def _draw_inputs(case, seed):
    """Everything random of a case, from its seed alone."""
    g, kind = _gen(seed), case["kind"]
    arch = _arch(case)
    dtype = DTYPES[case.get("dtype", "bf16")]
    x = {}
    if kind == "head":
        x["hidden"] = torch.randn(case["rows"], arch.hidden, generator=g, device="cuda").to(dtype)
        x["weight"] = (torch.randn(arch.vocab, arch.hidden, generator=g, device="cuda")
                       * 0.02).to(dtype)
        return x
    if kind == "attn":
        lens = _lens(case)
        x["tables"], nb = _tables(lens, seed, case["shared"])
        x["k"], x["v"] = _pools(arch, nb, dtype, g, 1.0)
        x["q"] = torch.randn(arch.num_layers, case["seqs"], case["q"], arch.num_q_heads,
                             arch.head_dim, generator=g, device="cuda").to(dtype)
        return x
    x["sd"] = _weights(arch, dtype, g)

    def tokens(*shape):
        return torch.randint(0, arch.vocab, shape, generator=g, device="cuda")

    if kind == "layers":
        x["tables"], nb = _tables(_lens(case), seed)
        # keys and values have about the spread of a projected unit-RMS row
        x["k"], x["v"] = _pools(arch, nb, dtype, g, 0.02 * arch.hidden ** 0.5)
        x["ids"] = tokens(case["seqs"], case["q"])
    elif kind == "prefill":
        lens = _prompt_lens(case)
        x["tables"], x["nb"] = _tables(lens, seed)
        x["ids"] = tokens(sum(lens))
    else:
        x["ids"] = tokens(1, case["tokens"])
    return x


# ---- the passes ---------------------------------------------------------------

class _Replayed:
    """A pass captured as a HIP graph, its outputs the graph's own buffers."""

    def __init__(self, fn):
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            fn()
        torch.cuda.current_stream().wait_stream(s)
        self.fn = fn  # what the graph reads stays alive with it
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph, stream=s):
            self.out = fn()

    def __call__(self):
        self.graph.replay()
        return self.out


def prepare(case, seed):
    x = _draw_inputs(case, seed)
    arch, kind = _arch(case), case["kind"]
    dtype = DTYPES[case.get("dtype", "bf16")]
    if kind == "head":
        h, w = x["hidden"], x["weight"]
        if case["blocked"]:
            h, w = kernels.to_blocked(h), kernels.to_blocked(w)
        m = case["rows"]
        out = {"ids": torch.empty(m, dtype=torch.int32, device="cuda"),
               "max": torch.empty(m, device="cuda")}
        if case["second"]:
            out["second_id"] = torch.empty(m, dtype=torch.int32, device="cuda")
            out["second"] = torch.empty(m, device="cuda")

        def head():
            kernels.lmhead_argmax(h, w, argmax=out["ids"], maxval=out["max"],
                                  second_id=out.get("second_id"), second_val=out.get("second"),
                                  blocked=case["blocked"], rows=m)
            return out
        return head
    order = (case.get("unit", 0), case.get("kw", 0))
    if kind == "attn":
        lens = _lens(case)
        tables = _device_tables(x["tables"])
        start = torch.tensor([n - case["q"] for n in lens], dtype=torch.int32, device="cuda")
        q, k, v = x["q"], x["k"], x["v"]
        L, B, T, Hq, D = q.shape
        ctx = max(lens)

        def attn():
            plan = kernels.attn_plan(tables, start, B, T, Hq, arch.num_kv_heads, D, BS, k.shape[1],
                                     ctx, dtype, unit_blocks=order[0], key_waves=order[1])
            return [kernels.paged_verify_attn(q[i], k[i], v[i], tables, start, ctx,
                                              unit_blocks=order[0], key_waves=order[1], plan=plan)
                    for i in range(L)]
        return _Replayed(attn) if case["graph"] else attn
    model = build_model(arch, x["sd"], dtype=dtype, device="cuda")
    ids = x["ids"]
    if kind == "layers":
        lens = _lens(case)
        start = torch.tensor([n - case["q"] for n in lens], dtype=torch.int32, device="cuda")
        kv = DeviceKV(x["k"], x["v"], _device_tables(x["tables"]), start, BS)
        rows = torch.arange(case["seqs"], dtype=torch.int32, device="cuda")
        ctx = max(lens)

        def layers():
            h = forward_hidden(model, ids, kv, rows, ctx, attn_order=order,
                               gemm_rows=case["gemm_rows"] or None)
            return {"hidden": h, "k": kv.k, "v": kv.v}
        return _Replayed(layers) if case["graph"] else layers
    if kind == "prefill":
        lens = _prompt_lens(case)
        B, T = len(lens), max(lens)
        k, v = (torch.zeros(s, dtype=dtype, device="cuda") for s in (
            (arch.num_layers, x["nb"], arch.num_kv_heads, BS, arch.head_dim),
            (arch.num_layers, x["nb"], arch.num_kv_heads, arch.head_dim, BS)))
        kv = DeviceKV(k, v, _device_tables(x["tables"]),
                      torch.zeros(B, dtype=torch.int32, device="cuda"), BS)
        rows = torch.arange(B, dtype=torch.int32, device="cuda")
        q_lens = torch.tensor(lens, dtype=torch.int32, device="cuda")
        dst = torch.tensor([b * T + t for b, n in enumerate(lens) for t in range(n)], device="cuda")
        fwd = forward_packed_wide if case["arch"] == "3b" else forward_packed

        def prefill():
            h = fwd(model, ids, dst, B, T, kv, rows, T, q_lens, attn_order=order)
            return {"hidden": h, "k": kv.k, "v": kv.v}
        return prefill
    n = case["tokens"]
    pool = PagedKVCache.for_model(model, num_blocks=-(-n // BS) + 8, max_seqs=4)
    if kind == "prompt":
        def prompt():
            seq = pool.new_sequence("prompt")
            h = forward_with_own_cache(model, ids, seq, all_logits=True, return_hidden=True)
            logits = model.lm_head(h[:, -1:])
            seq.free()
            return {"hidden": h, "logits": logits}
        return prompt
    seq = pool.new_sequence("step")
    if n > 1:
        forward_with_own_cache(model, ids[:, :-1], seq)
    last = ids[:, -1:].contiguous()

    def step():
        logits = forward_with_own_cache(model, last, seq)
        seq.truncate(n - 1)
        return {"logits": logits, "k": pool.k, "v": pool.v}
    return step


def run(state):
    return state()


# ---- what a pass cannot do without ----------------------------------------------

def work(case):
    arch, kind = _arch(case), case["kind"]
    e = 4 if case.get("dtype") == "fp32" else 2
    if kind == "head":
        m = case["rows"]
        return {"bytes": e * arch.hidden * (arch.vocab + m) + 16 * m,
                "flops": 2 * m * arch.hidden * arch.vocab}
    if kind in ("layers", "attn"):
        lens, new = _lens(case), [case["q"]] * case["seqs"]
    elif kind == "prefill":
        lens = new = _prompt_lens(case)
    elif kind == "prompt":
        lens = new = [case["tokens"]]
    else:
        lens, new = [case["tokens"]], [1]
    L, rows = arch.num_layers, sum(new)
    kv_row = 2 * arch.kv_dim * e
    pairs = sum(n * (c - n) + n * (n + 1) // 2 for c, n in zip(lens, new))
    # keys and values read: a shared prefix's once
    keys = sum(lens) - case.get("shared", 0) * (len(lens) - 1)
    attn_flops = 4 * arch.q_dim * pairs
    if kind == "attn":
        return {"bytes": L * (keys * kv_row + 2 * rows * arch.q_dim * e), "flops": L * attn_flops}
    proj = arch.hidden * (2 * arch.q_dim + 2 * arch.kv_dim) + 3 * arch.hidden * arch.ffn
    out = {"bytes": L * (proj * e + keys * kv_row) + 2 * rows * arch.hidden * e,
           "flops": L * (2 * rows * proj + attn_flops)}
    if kind in ("prompt", "step"):
        out["bytes"] += arch.vocab * (arch.hidden + 1) * e
        out["flops"] += 2 * arch.vocab * arch.hidden
    return out


def tolerance(case):
    """About four times what a pass differs from the same in 64 bits."""
    kind = case["kind"]
    if case.get("dtype") == "fp32":
        return {"rel": 2e-5, "max": 2e-4}
    if kind == "head":
        # a sum next to a rounding boundary moves a maximum by one bf16 step
        return {"rel": 1e-3, "max": 1e-2, "differ": 0.03}
    if kind == "attn":
        return {"rel": 7e-3, "max": 6e-2}
    if kind == "step":
        return {"rel": 7e-2, "max": 0.4}
    return {"rel": 5e-2, "max": 0.3}


# ---- the same in 64 bits ----------------------------------------------------------

def _attend(q, k, v):
    """Causal attention of the newest rows: q [T, Hq, D], k/v [C, Hkv, D]."""
    T, Hq, D = q.shape
    C, Hkv, _ = k.shape
    out = torch.empty_like(q)
    mask = torch.arange(C, device=q.device)[None] > torch.arange(C - T, C, device=q.device)[:, None]
    for h in range(Hq):
        kh, vh = (t[:, h // (Hq // Hkv)].contiguous() for t in (k, v))
        s = (q[:, h].contiguous() @ kh.t().contiguous()) * D ** -0.5
        out[:, h] = torch.softmax(s.masked_fill_(mask, -math.inf), -1) @ vh
    return out


def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _rope(x, pos, theta):
    """Rotary embedding of x [N, heads, D] at positions pos [N]."""
    D = x.shape[-1]
    inv = theta ** (-torch.arange(0, D, 2, device=x.device, dtype=torch.float64) / D)
    f = pos.double()[:, None] * inv
    c, s = torch.cos(f).repeat(1, 2)[:, None], torch.sin(f).repeat(1, 2)[:, None]
    half = torch.cat([-x[..., D // 2:], x[..., :D // 2]], -1)
    return x * c + half * s


def _model64(arch, sd, ids, starts, new, history=None):
    """Qwen2 in float64: final-normed rows of the packed tokens `ids` and each
    layer's new keys and values. history(layer, sequence) -> earlier k, v."""
    dev = ids.device
    pos = torch.cat([torch.arange(s, s + n, device=dev) for s, n in zip(starts, new)])
    x = sd["model.embed_tokens.weight"][ids].double()
    D, kvs = arch.head_dim, []
    for i in range(arch.num_layers):
        w = {n[len(f"model.layers.{i}."):]: t.double() for n, t in sd.items()
             if n.startswith(f"model.layers.{i}.")}

        def proj(name, h):
            y = h @ w[name + ".weight"].t()
            return y + w[name + ".bias"] if name + ".bias" in w else y

        h = _rms(x, w["input_layernorm.weight"], arch.rms_eps)
        q, k, v = (proj(f"self_attn.{n}_proj", h).view(len(pos), -1, D) for n in "qkv")
        q, k = _rope(q, pos, arch.rope_theta), _rope(k, pos, arch.rope_theta)
        kvs.append((k, v))
        att, at = torch.empty_like(q), 0
        for b, n in enumerate(new):
            kb, vb = k[at:at + n], v[at:at + n]
            if history is not None:
                hk, hv = history(i, b)
                kb, vb = torch.cat([hk, kb]), torch.cat([hv, vb])
            att[at:at + n] = _attend(q[at:at + n], kb, vb)
            at += n
        x = x + proj("self_attn.o_proj", att.view(len(pos), -1))
        h = _rms(x, w["post_attention_layernorm.weight"], arch.rms_eps)
        x = x + proj("mlp.down_proj", torch.nn.functional.silu(proj("mlp.gate_proj", h))
                     * proj("mlp.up_proj", h))
    return _rms(x, sd["model.norm.weight"].double(), arch.rms_eps), kvs


def _gathered(x, layer, b, n):
    """The first n tokens' keys and values of sequence b, [n, Hkv, D] in 64 bits."""
    ids = torch.tensor(x["tables"][b], device="cuda")
    k = x["k"][layer][ids].permute(0, 2, 1, 3).flatten(0, 1)
    v = x["v"][layer][ids].permute(0, 3, 1, 2).flatten(0, 1)
    return k[:n].double(), v[:n].double()


def exact(case, seed):
    x = _draw_inputs(case, seed)
    arch, kind = _arch(case), case["kind"]
    if kind == "head":
        # the entry point's logits are those of the model's type
        logits = torch.empty(case["rows"], arch.vocab, dtype=torch.float64, device="cuda")
        for a in range(0, arch.vocab, 32768):
            logits[:, a:a + 32768] = x["hidden"].double() @ x["weight"][a:a + 32768].double().t()
        logits = logits.to(x["hidden"].dtype).double()

        def first(t):
            top = t.max(1).values
            i = torch.arange(arch.vocab, device="cuda").expand_as(t)
            return top, torch.where(t == top[:, None], i, arch.vocab).min(1).values
        top, ids = first(logits)
        if not case["second"]:
            return {"ids": ids, "max": top}
        second, sid = first(logits.scatter(1, ids[:, None], -math.inf))
        return {"ids": ids, "max": top, "second_id": sid, "second": second}
    if kind == "attn":
        outs = []
        for i in range(arch.num_layers):
            rows = []
            for b, n in enumerate(_lens(case)):
                rows.append(_attend(x["q"][i, b].double(), *_gathered(x, i, b, n)))
            outs.append(torch.stack(rows))
        return outs
    sd, ids = x["sd"], x["ids"].reshape(-1)
    if kind in ("prompt", "step"):
        n = case["tokens"]
        h, _ = _model64(arch, sd, ids, [0], [n])
        logits = (h[-1:] @ sd["model.embed_tokens.weight"].double().t())[None]
        if kind == "prompt":
            return {"hidden": h[None], "logits": logits}
        return {"logits": logits, "k": None, "v": None}  # the allocator places the blocks
    if kind == "layers":
        new = [case["q"]] * case["seqs"]
        starts = [n - case["q"] for n in _lens(case)]
        h, kvs = _model64(arch, sd, ids, starts, new,
                          lambda i, b: _gathered(x, i, b, starts[b]))
        h = h.view(case["seqs"], case["q"], -1)
        k, v = x["k"].double(), x["v"].double()
    else:
        new = _prompt_lens(case)
        starts = [0] * len(new)
        h, kvs = _model64(arch, sd, ids, starts, new)
        k = torch.zeros(arch.num_layers, x["nb"], arch.num_kv_heads, BS, arch.head_dim,
                        dtype=torch.float64, device="cuda")
        v = torch.zeros(arch.num_layers, x["nb"], arch.num_kv_heads, arch.head_dim, BS,
                        dtype=torch.float64, device="cuda")
    pos = [(b, s + t) for b, (s, n) in enumerate(zip(starts, new)) for t in range(n)]
    blk = torch.tensor([x["tables"][b][p // BS] for b, p in pos], device="cuda")
    off = torch.tensor([p % BS for _, p in pos], device="cuda")
    for i, (kn, vn) in enumerate(kvs):
        k[i, blk, :, off] = kn
        v[i, blk, :, :, off] = vn
    return {"hidden": h, "k": k, "v": v}
