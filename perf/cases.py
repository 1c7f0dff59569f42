"""The work a user of this package has it do, as cases to time and compare: every check through its public entry point.

serve     one model step under ServeGuard: the check of each of a decoder layer's four linear layers (decode at a few
          rows, prefill at thousands)
linear    both block checks of a linear layer (column blocks and row blocks) from one read of its output
train     one layer's training step under a guard's Group: the checks of y = x W^T + b, dx = dy W and dW = dy^T x
product   one matmul's check with the score of every checksum (2-D, or a batched product)
moe       the check of a MoE layer's grouped product (the experts' sums made in the call, or once as when served)
quant     the check of an int8 (exact) or fp8 (scaled) product, in one call or with the weight's constants kept
precise   the float64 check of an fp32 product (an accumulator before it is rounded)
paged     a decode step's integrity checks of a paged KV cache: block fingerprints against the ledger, and the
          sampled attention recompute of every layer
"""
import math
import os

os.environ.setdefault("SDCGUARD_SIGN_SEED", "1")        # the signed sums' pattern: the same in every process

import torch

BLOCK = 128
ALARM = 6.0
FLOOR = 1e-20
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


# ---------------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # The four linear layers of a Qwen2.5-7B decoder layer at a decode step of 16 sequences: the smallest calls of
        # a served model, bound by launches and latency.
        {"name": "serve_decode_16", "kind": "serve", "rows": 16, "hidden": 3584, "qkv": 4608, "inter": 18944,
         "dtype": "bf16"},
        # The same layers at a prefill of 4096 tokens.
        {"name": "serve_prefill_4096", "kind": "serve", "rows": 4096, "hidden": 3584, "qkv": 4608, "inter": 18944,
         "dtype": "bf16"},
        # Both block checks of a Llama MLP up projection (the benchmark's layer).
        {"name": "linear_both_4096", "kind": "linear", "m": 4096, "k": 4096, "n": 14336},
        # A training step of the same layer: forward, input gradient and weight gradient.
        {"name": "train_mlp_4096", "kind": "train", "m": 4096, "k": 4096, "n": 14336, "dtype": "bf16",
         "bias": False},
        # A training step of GPT-2's output head: an odd number of columns, so rows of y and dy start at any 2 bytes.
        {"name": "train_head_50257", "kind": "train", "m": 1024, "k": 768, "n": 50257, "dtype": "bf16",
         "bias": False},
        # One 1024^3 matmul answered with every score: the ordinary small check.
        {"name": "product_1024", "kind": "product", "batch": 0, "m": 1024, "k": 1024, "n": 1024, "dtype": "bf16",
         "bias": True},
        # The q k^T products of a vision transformer's attention (577 tokens: 24 x 24 patches and a class token) in
        # fp16, k passed as the transposed view that attention code passes.
        {"name": "batched_96x577", "kind": "product", "batch": 96, "m": 577, "k": 64, "n": 577, "dtype": "fp16",
         "bias": False},
        # A MoE layer's grouped product in training (4096 tokens, 8 of 64 experts with Zipf loads).
        {"name": "moe_train_4096", "kind": "moe", "tokens": 4096, "topk": 8, "experts": 64, "k": 2048, "n": 1408,
         "kept": False, "dtype": "bf16"},
        # An int8 product judged in one call, as a screen of a device does it: with a few bits flipped.
        {"name": "judge_int8_2048", "kind": "quant", "mode": "int8", "m": 2048, "k": 7168, "n": 4096, "kept": False},
        # A served fp8 linear layer (scales per token and per channel, bf16 output), its constants made at load.
        {"name": "fp8_served_4096", "kind": "quant", "mode": "fp8", "m": 4096, "k": 4096, "n": 14336, "kept": True},
        # The precise check of a 4096^3 product.
        {"name": "precise_4096", "kind": "precise", "m": 4096, "k": 4096, "n": 4096, "dtype": "bf16"},
        # A decode step of 64 sequences over a 28-layer paged cache.
        {"name": "paged_decode_64", "kind": "paged", "layers": 28, "blocks": 4096, "seqs": 64, "longest": 2048,
         "heads": 16, "kv_heads": 8, "dim": 128, "samples": 16},
    ]


def draw(rng):
    def log(lo, hi, step=1):
        return max(step, int(math.exp(rng.uniform(math.log(lo), math.log(hi)))) // step * step)

    def size(lo, hi):
        # half of the sizes round (multiples of 256 or 64), half odd
        return log(lo, hi, rng.choice((1, 1, 64, 256)))

    dt = rng.choice(("bf16", "bf16", "fp16"))
    kind = rng.choice(("serve", "serve", "linear", "train", "train", "product", "batched", "moe", "quant", "quant",
                       "precise", "paged"))
    if kind == "serve":
        return {"kind": kind, "rows": log(1, 4096), "hidden": log(512, 3584, rng.choice((8, 64, 256))),
                "qkv": size(768, 4608), "inter": log(1024, 18944, rng.choice((8, 64, 256))), "dtype": dt}
    if kind == "linear":
        return {"kind": kind, "m": log(16, 4096, rng.choice((1, 128))), "k": log(256, 4096, rng.choice((8, 256))),
                "n": log(256, 14336, rng.choice((8, 128)))}
    if kind == "train":
        return {"kind": kind, "m": size(128, 4096), "k": size(256, 4096), "n": size(256, 14336), "dtype": dt,
                "bias": rng.random() < 0.5}
    if kind == "product":
        return {"kind": kind, "batch": 0, "m": size(64, 4096), "k": size(64, 4096), "n": size(64, 8192), "dtype": dt,
                "bias": rng.random() < 0.5}
    if kind == "batched":
        return {"kind": "product", "batch": log(4, 96), "m": size(32, 600), "k": log(32, 256, rng.choice((1, 8))),
                "n": size(32, 600), "dtype": dt, "bias": False}
    if kind == "moe":
        return {"kind": kind, "tokens": log(16, 4096), "topk": rng.choice((2, 4, 8)), "experts": rng.choice((16, 32, 64)),
                "k": log(512, 2048, rng.choice((8, 512))), "n": size(256, 1408), "kept": rng.random() < 0.5,
                "dtype": dt}
    if kind == "quant":
        mode = rng.choice(("int8", "fp8"))
        k = log(512, 7168, rng.choice((16, 1024)))
        return {"kind": kind, "mode": mode, "m": size(64, 4096), "k": k,
                "n": log(256, 4096 if mode == "int8" else 14336, rng.choice((8, 128))), "kept": rng.random() < 0.5}
    if kind == "precise":
        return {"kind": kind, "m": size(64, 4096), "k": size(128, 4096), "n": size(128, 4096), "dtype": dt}
    kvh = rng.choice((2, 4, 8))
    return {"kind": kind, "layers": log(2, 28), "blocks": log(256, 4096), "seqs": log(4, 64),
            "longest": log(128, 2048), "heads": kvh * rng.choice((1, 2, 4)), "kv_heads": kvh,
            "dim": rng.choice((64, 128)), "samples": rng.choice((4, 16))}


# ------------------------------------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, dtype, std=1.0):
    t = torch.empty(*shape, dtype=dtype, device="cuda")
    return t.normal_(0.0, std, generator=g)


def _serve_layers(c):
    """(name, inputs, outputs, bias) of a decoder layer's linear layers."""
    h, i = c["hidden"], c["inter"]
    return [("qkv", h, c["qkv"], True), ("o", h, h, False), ("gate_up", h, 2 * i, False), ("down", i, h, False)]


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, _gen(seed), seed)


def _prepare_serve(c, g, seed):
    from sdcguard_amd import ServeGuard
    dt = DTYPES[c["dtype"]]
    guard = ServeGuard()
    slots, xs, ys = [], [], []
    for name, k, n, has_bias in _serve_layers(c):
        lin = torch.nn.Linear(k, n, bias=has_bias, device="cuda", dtype=dt).requires_grad_(False)
        lin.weight.normal_(0.0, 0.02, generator=g)
        if has_bias:
            lin.bias.normal_(0.0, 0.1, generator=g)
        x = _randn(g, c["rows"], k, dtype=dt)
        slots.append(guard.add_layer(lin, name))
        xs.append(x)
        ys.append(lin(x))
    return {"kind": "serve", "guard": guard, "slots": slots, "xs": xs, "ys": ys, "rows": guard.state("cuda")}


def _prepare_linear(c, g, seed):
    from sdcguard_amd import LayerChecksums
    x = _randn(g, c["m"], c["k"], dtype=torch.bfloat16)
    w = _randn(g, c["n"], c["k"], dtype=torch.bfloat16, std=0.02)
    return {"kind": "linear", "x": x, "w": w, "y": torch.nn.functional.linear(x, w),
            "cs": LayerChecksums(w, None, BLOCK)}


def _prepare_train(c, g, seed):
    dt = DTYPES[c["dtype"]]
    x = _randn(g, c["m"], c["k"], dtype=dt)
    w = _randn(g, c["n"], c["k"], dtype=dt, std=0.02)
    b = _randn(g, c["n"], dtype=dt, std=0.1) if c["bias"] else None
    dy = _randn(g, c["m"], c["n"], dtype=dt, std=0.02)
    return {"kind": "train", "x": x, "w": w, "b": b, "dy": dy, "y": torch.nn.functional.linear(x, w, b),
            "dx": torch.mm(dy, w), "dw": torch.mm(dy.t(), x)}


def _prepare_product(c, g, seed):
    dt = DTYPES[c["dtype"]]
    if c["batch"]:
        q = _randn(g, c["batch"], c["m"], c["k"], dtype=dt)
        kt = _randn(g, c["batch"], c["n"], c["k"], dtype=dt)
        out = torch.bmm(q, kt.transpose(1, 2).contiguous())
        return {"kind": "product", "A": q, "B": kt.transpose(1, 2), "C": out, "bias": None,
                "scores": torch.empty(c["batch"], c["m"], -(-c["n"] // BLOCK), 2, device="cuda")}
    a = _randn(g, c["m"], c["k"], dtype=dt)
    b = _randn(g, c["k"], c["n"], dtype=dt, std=0.05)
    bias = _randn(g, c["n"], dtype=dt, std=0.1) if c["bias"] else None
    out = torch.mm(a, b) if bias is None else torch.addmm(bias, a, b)
    return {"kind": "product", "A": a, "B": b, "C": out, "bias": bias,
            "scores": torch.empty(1, c["m"], -(-c["n"] // BLOCK), 2, device="cuda")}


def _expert_loads(c, seed):
    gen = torch.Generator().manual_seed(seed)
    p = torch.tensor([1.0 / (r + 1) ** 1.1 for r in range(c["experts"])], dtype=torch.float64)
    picks = torch.multinomial(p.expand(c["tokens"], c["experts"]), c["topk"], replacement=False, generator=gen)
    return torch.bincount(picks.reshape(-1), minlength=c["experts"])


def _prepare_moe(c, g, seed):
    from sdcguard_amd.checksum import GroupedChecksums
    dt = DTYPES[c["dtype"]]
    loads = _expert_loads(c, seed)
    rows = int(loads.sum())
    a = _randn(g, rows, c["k"], dtype=dt)
    w = _randn(g, c["experts"], c["k"], c["n"], dtype=dt, std=0.02)
    out = torch.empty(rows, c["n"], dtype=dt, device="cuda")
    start = 0
    for e, load in enumerate(loads.tolist()):
        if load:
            out[start:start + load] = a[start:start + load] @ w[e]
        start += load
    return {"kind": "moe", "a": a, "w": w, "out": out, "offs": torch.cumsum(loads, 0).to(torch.int32).cuda(),
            "kept": GroupedChecksums(w) if c["kept"] else None,
            "scores": torch.empty(rows, -(-c["n"] // BLOCK), 2, device="cuda")}


def _prepare_quant(c, g, seed):
    from sdcguard_amd import modes
    m, k, n = c["m"], c["k"], c["n"]
    if c["mode"] == "int8":
        a = torch.randint(-127, 128, (m, k), device="cuda", generator=g, dtype=torch.int32).to(torch.int8)
        b = torch.randint(-127, 128, (k, n), device="cuda", generator=g, dtype=torch.int32).to(torch.int8)
        out = (a.double() @ b.double()).to(torch.int32)
        # eight flipped bits among the accumulators
        r = torch.randint(0, m, (8,), device="cuda", generator=g)
        j = torch.randint(0, n, (8,), device="cuda", generator=g)
        out[r, j] = out[r, j] ^ (1 << torch.randint(0, 30, (8,), device="cuda", generator=g, dtype=torch.int32))
        sa = sb = None
    else:
        a = (torch.randn(m, k, device="cuda", generator=g) * 4).clamp(-448, 448).to(torch.float8_e4m3fn)
        b = (torch.randn(k, n, device="cuda", generator=g) * 4).clamp(-448, 448).to(torch.float8_e4m3fn)
        sa = (10.0 ** (torch.rand(m, device="cuda", generator=g) * 2 - 3)).float()
        sb = (10.0 ** (torch.rand(n, device="cuda", generator=g) * 2 - 3)).float()
        out = ((a.float() @ b.float()) * sa[:, None] * sb[None, :]).bfloat16()
    return {"kind": "quant", "mode": c["mode"], "a": a, "b": b, "C": out, "sa": sa, "sb": sb,
            "kept": modes.QuantChecksums.make(b, sb) if c["kept"] else None}


def _prepare_precise(c, g, seed):
    dt = DTYPES[c["dtype"]]
    a = _randn(g, c["m"], c["k"], dtype=dt)
    w = _randn(g, c["n"], c["k"], dtype=dt, std=0.02)
    return {"kind": "precise", "A": a, "B": w.t(), "C": a.float() @ w.float().t().contiguous(),
            "scores": torch.empty(1, c["m"], -(-c["n"] // BLOCK), 2, device="cuda")}


def _prepare_paged(c, g, seed):
    from sdcguard_amd import serve_attn
    from sdcguard_amd.kv import KVLedger
    layers, nblk, seqs, dim, hq, hk, ntok = c["layers"], c["blocks"], c["seqs"], c["dim"], c["heads"], c["kv_heads"], 16
    cpu = torch.Generator().manual_seed(seed)
    lens = torch.randint(max(1, c["longest"] // 4), c["longest"] + 1, (seqs,), generator=cpu)
    lens = torch.minimum(lens, torch.tensor(nblk * ntok))
    width = -(-c["longest"] // ntok)
    table = torch.full((seqs, width), -1, dtype=torch.int64)
    for r in range(seqs):
        used = -(-int(lens[r]) // ntok)
        table[r, :used] = torch.randperm(nblk, generator=cpu)[:used]
    pos = lens - 1
    tail = table[torch.arange(seqs), pos // ntok]
    slots = (tail * ntok + pos % ntok).cuda()
    dev_table, dev_lens = table.cuda(), lens.to(torch.int32).cuda()
    live = torch.arange(width * ntok, device="cuda")[None, :] < dev_lens[:, None]
    out = {"kind": "paged", "layers": [], "ledgers": [], "table": dev_table, "lens": dev_lens, "slots": slots,
           "attn_table": dev_table.clamp(min=0).to(torch.int32), "scale": dim ** -0.5, "samples": c["samples"],
           "qsl": torch.arange(seqs + 1, dtype=torch.int32, device="cuda"), "step": 1000 + seed % 1000}
    for _ in range(layers):
        kv = _randn(g, nblk, hk, ntok, 2 * dim, dtype=torch.bfloat16)
        q = _randn(g, seqs, hq, dim, dtype=torch.bfloat16, std=0.5)
        rows = kv[dev_table.clamp(min=0)].permute(0, 1, 3, 2, 4).reshape(seqs, width * ntok, hk, 2 * dim).float()
        keys = rows[..., :dim].permute(0, 2, 1, 3).contiguous()
        vals = rows[..., dim:].permute(0, 2, 1, 3).contiguous()
        s = torch.matmul(q.float().view(seqs, hk, hq // hk, dim), keys.transpose(-1, -2).contiguous()) * dim ** -0.5
        s = s.masked_fill(~live[:, None, None, :], float("-inf"))
        o = torch.matmul(torch.softmax(s, -1), vals).reshape(seqs, hq, dim).bfloat16()
        b, t = tail.cuda(), (pos % ntok).cuda()
        ledger = KVLedger(kv, seqs, width)
        ledger.record(dev_table)
        # one block of the cache changed since: a flipped bit in one of its words
        at = int(torch.randint(0, nblk, (1,), generator=cpu))
        kv.view(torch.int16)[at, 0, 0, 0] ^= 1
        out["layers"].append((kv, q, o, kv[b, :, t, :dim].contiguous(), kv[b, :, t, dim:].contiguous()))
        out["ledgers"].append(ledger)
        del rows, keys, vals, s
    out["bufs"] = serve_attn.buffers("cuda", layers, dim, 64, torch.bfloat16, samples=c["samples"])
    out["bufs"]["ctrl"].copy_(torch.tensor([out["step"], 1]))
    out["scores"] = torch.zeros(layers, c["samples"], dim, device="cuda")
    return out


_PREPARE = {"serve": _prepare_serve, "linear": _prepare_linear, "train": _prepare_train, "product": _prepare_product,
            "moe": _prepare_moe, "quant": _prepare_quant, "precise": _prepare_precise, "paged": _prepare_paged}


# ------------------------------------------------------------------------------------------------------ one pass
def run(state):
    return _RUN[state["kind"]](state)


def _worst(rows):
    """The worst score of every int64 result row (the high half of its key), as the rows hold it: a view."""
    return rows.view(torch.float32)[:, 1]


def _run_serve(s):
    for slot, x, y in zip(s["slots"], s["xs"], s["ys"]):
        s["guard"].check(slot, x, y)
    # (the rows also count the checks since the last poll, which is the number of passes)
    rows = s["rows"][:len(s["slots"])]
    return {"worst": _worst(rows), "unjudged": rows[:, 3]}


def _run_linear(s):
    from sdcguard_amd.linear import check_linear_both
    state, rows = check_linear_both(s["x"], s["w"], None, s["y"], s["cs"])
    return {"worst": _worst(state.view(1, -1)), "worst_rows": _worst(rows.view(1, -1)), "unjudged": state[3:],
            "unjudged_rows": rows[2:]}


def _run_train(s):
    from sdcguard_amd import Group
    g = Group(s["y"].device, s["y"].dtype)
    g.add(s["x"], s["w"].t(), s["y"], s["b"], 1.0, 1.0)
    g.add(s["dy"], s["w"], s["dx"], None, 1.0, 1.0)
    g.add(s["dy"].t(), s["x"], s["dw"], None, 1.0, 1.0)
    g.launch()
    return {"worst": _worst(g.result), "unjudged": g.result[:, 2]}


def _run_product(s):
    from sdcguard_amd import matmul_zscores
    st = matmul_zscores(s["A"], s["B"], s["C"], s["bias"], scores_out=s["scores"])
    return {"scores": s["scores"], "unjudged": st.result[2:]}


def _run_moe(s):
    from sdcguard_amd.checksum import grouped_zscores
    w = None if s["kept"] is not None else s["w"]
    st = grouped_zscores(s["a"], w, s["out"], s["offs"], checksums=s["kept"], scores_out=s["scores"])
    return {"scores": s["scores"], "worst": _worst(st.results), "unjudged": st.results[:, 2]}


def _run_quant(s):
    from sdcguard_amd import modes
    if s["kept"] is None:
        r = modes.judge(s["mode"], s["a"], s["b"], s["C"], sa=s["sa"], sb=s["sb"])
        return {"z": r["z"], "wrong": r["wrong_blocks"], "nonfinite": r["nonfinite_blocks"]}
    st = modes.quant_zscores(s["a"], s["kept"], s["C"], sa=s["sa"])
    if s["mode"] == "int8":                                 # (the row: the last wrong block, its count)
        return {"row": st.result}
    return {"worst": _worst(st.result.view(1, -1)), "wrong": st.result[2:3], "nonfinite": st.result[3:]}


def _run_precise(s):
    from sdcguard_amd.checksum import matmul_zscores_acc
    st = matmul_zscores_acc(s["A"], s["B"], s["C"], nfma=16, scores_out=s["scores"])
    return {"scores": s["scores"], "unjudged": st.result[2:]}


def _run_paged(s):
    from sdcguard_amd import serve_attn
    b, checks = s["bufs"], []
    for i, (kv, q, o, key, val) in enumerate(s["layers"]):
        serve_attn.attn_check(q, o, kv, key, val, s["qsl"], s["lens"], s["attn_table"], s["slots"], b["state"], i,
                              b["ctrl"], 1, 0, s["scale"], -1, serve_attn.ATTN_Z, b["capm"], b["capq"], b["capo"],
                              None, None, b["ws"], True, False, samples=s["samples"], scores_out=s["scores"][i])
        checks.append(s["ledgers"][i].verify(s["table"]))
    return {"scores": s["scores"], "counts": [c.count for c in checks],
            "mismatch": checks[0].mismatch, "mismatch_last": checks[-1].mismatch}


_RUN = {"serve": _run_serve, "linear": _run_linear, "train": _run_train, "product": _run_product, "moe": _run_moe,
        "quant": _run_quant, "precise": _run_precise, "paged": _run_paged}


# ------------------------------------------------------------------------------------------- what a pass must do
def work(case):
    """Each input read once and each output written once; the products are those of the expected sides (every row
    against two sums a block)."""
    c = case
    kind = c["kind"]

    def product(m, k, n):
        return 2.0 * m * k * 2 * -(-n // BLOCK)

    if kind == "serve":
        ls = _serve_layers(c)
        # (the layer's sums, not its weights, are what a served check reads: two fp32 sums a block)
        return {"bytes": sum(c["rows"] * (k + n) * 2 + k * 2 * -(-n // BLOCK) * 4 for _, k, n, _ in ls),
                "flops": sum(product(c["rows"], k, n) for _, k, n, _ in ls)}
    if kind in ("linear", "train"):
        m, k, n = c["m"], c["k"], c["n"]
        mats = 2.0 * (m * k + n * k + m * n)
        if kind == "linear":
            return {"bytes": mats, "flops": product(m, k, n) + product(n, k, m)}
        return {"bytes": 2.0 * mats, "flops": product(m, k, n) + product(m, n, k) + product(n, m, k)}
    if kind == "product":
        b, m, k, n = max(1, c["batch"]), c["m"], c["k"], c["n"]
        return {"bytes": b * (2.0 * (m * k + k * n + m * n) + 8.0 * m * -(-n // BLOCK)), "flops": b * product(m, k, n)}
    if kind == "moe":
        rows, k, n = c["tokens"] * c["topk"], c["k"], c["n"]
        sums = c["experts"] * k * (2 * -(-n // BLOCK) * 4.0 if c["kept"] else 2.0 * n)
        return {"bytes": 2.0 * rows * (k + n) + sums + 8.0 * rows * -(-n // BLOCK), "flops": product(rows, k, n)}
    if kind == "quant":
        m, k, n = c["m"], c["k"], c["n"]
        sums = k * 2 * -(-n // BLOCK) * 4.0 if c["kept"] else 1.0 * k * n
        scores = 0.0 if c["kept"] else 4.0 * m * -(-n // BLOCK)
        return {"bytes": m * k + sums + m * n * (4.0 if c["mode"] == "int8" else 2.0) + scores,
                "flops": product(m, k, n)}
    if kind == "precise":
        m, k, n = c["m"], c["k"], c["n"]
        return {"bytes": 2.0 * (m * k + k * n) + 4.0 * m * n + 8.0 * m * -(-n // BLOCK), "flops": product(m, k, n)}
    # paged: the blocks the tables point at (five eighths of the longest context on average), and the sampled rows
    tokens = 0.625 * c["longest"]
    block = c["kv_heads"] * 16 * 2 * c["dim"] * 2
    return {"bytes": c["layers"] * (c["seqs"] * tokens / 16 * block + c["samples"] * tokens * 2 * c["dim"] * 2),
            "flops": c["layers"] * c["samples"] * tokens * 4 * c["dim"]}


def tolerance(case):
    """Scores are a small difference of two large sums over a noise estimate: the expected side's fp32 sums (three
    16-bit parts of each block sum, added over the depth in any order) show in them at about 1e-4."""
    if case["kind"] == "quant" and case["mode"] == "int8":
        return "exact"
    if case["kind"] == "precise":                           # float64 sums on both sides, scores rounded to fp32
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 2e-3, "max": 2e-2}


# ---------------------------------------------------------------------------------------------- the same in 64 bits
def _signs(width):
    seed = int(os.environ["SDCGUARD_SIGN_SEED"])
    g = torch.Generator().manual_seed((seed + width) % (2 ** 63))
    return (torch.randint(0, 2, (width,), generator=g) * 2 - 1).double()


def _pairs(x):
    """(..., n) float64 -> (..., nb, 2): the plain and the signed sum of every block of 128 (the last may be
    narrower, with the pattern of its own width)."""
    n = x.shape[-1]
    full, rem = divmod(n, BLOCK)
    out = []
    if full:
        v = x[..., :full * BLOCK].reshape(*x.shape[:-1], full, BLOCK)
        out.append(torch.stack([v.sum(-1), (v * _signs(BLOCK).to(x.device)).sum(-1)], -1))
    if rem:
        v = x[..., full * BLOCK:]
        out.append(torch.stack([v.sum(-1), (v * _signs(rem).to(x.device)).sum(-1)], -1).unsqueeze(-2))
    return torch.cat(out, -2)


def _per_block(x, fn):
    """fn over every block of x's last dimension: (..., n) -> (..., nb)."""
    full, rem = divmod(x.shape[-1], BLOCK)
    out = []
    if full:
        out.append(fn(x[..., :full * BLOCK].reshape(*x.shape[:-1], full, BLOCK)))
    if rem:
        out.append(fn(x[..., full * BLOCK:]).unsqueeze(-1))
    return torch.cat(out, -1)


def _widths(n, device):
    full, rem = divmod(n, BLOCK)
    return torch.tensor([float(BLOCK)] * full + ([float(rem)] if rem else []), dtype=torch.float64, device=device)


def _norm(x):
    return x.square().sum(-1).sqrt()


def _z64(A, B, C, bias=None):
    """Every checksum's score of a 16-bit C = A @ B (+ bias): (..., m, nb, 2) in float64."""
    u, h = (2.0 ** -8, 0.0) if C.dtype == torch.bfloat16 else (2.0 ** -11, 2.0 ** -25)
    A, B, C = A.double(), B.double(), C.double()
    k = A.shape[-1]
    b2 = _pairs(B)                                                          # (..., k, nb, 2)
    nb = b2.shape[-2]
    e = torch.matmul(A, b2.flatten(-2)).unflatten(-1, (nb, 2))
    if bias is not None:
        e = e + _pairs(bias.double())
    actual = _pairs(C)
    l1c = max(1e-5, k * 2.0 ** -27)
    an, al = _norm(A)[..., None, None], A.abs().sum(-1)[..., None, None]
    b2n, b2m = b2.square().sum(-3).sqrt().unsqueeze(-3), b2.abs().amax(-3).unsqueeze(-3)
    floor = torch.minimum(an * b2n * 1e-5, al * b2m * l1c)
    w = _widths(C.shape[-1], C.device)
    d = (e - actual).abs()
    cn, c1 = _per_block(C, _norm), _per_block(C, lambda v: v.abs().sum(-1))
    z = d / (cn[..., None] * u + floor + FLOOR + (w.sqrt() * h)[:, None])
    worst = c1 * 1.25 * u + 1.25 * w * h + floor[..., 0] + FLOOR
    z[..., 0] = torch.minimum(z[..., 0], d[..., 0] / worst * ALARM)
    return z


def _z64_precise(A, B, C, nfma):
    u = 2.0 ** -24
    A, B, C = A.double(), B.double(), C.double()
    k = A.shape[-1]
    b2 = _pairs(B)
    nb = b2.shape[-2]
    d = ((A @ b2.flatten(-2)).unflatten(-1, (nb, 2)) - _pairs(C)).abs()
    frob = _per_block(B.square().sum(0), lambda v: v.sum(-1)).sqrt()
    per_out = math.sqrt(k) + k / nfma + _widths(C.shape[-1], C.device).sqrt()
    prod = _norm(A)[:, None] * frob * (0.6 * math.sqrt(k) * u)
    z = d / (_per_block(C, _norm) * per_out * u + prod + FLOOR)[..., None]
    worst = _per_block(C, lambda v: v.abs().sum(-1)) * per_out * u + prod + FLOOR
    z[..., 0] = torch.minimum(z[..., 0], d[..., 0] / worst * ALARM)
    return z


def _z64_fp8(a, sa, b, sb, C):
    a, b, C = a.double() * sa.double()[:, None], b.double() * sb.double(), C.double()
    k = a.shape[1]
    b2 = _pairs(b)
    d = ((a @ b2.flatten(-2)).unflatten(-1, (b2.shape[-2], 2)) - _pairs(C)).abs().amax(-1)
    frob = _per_block(b.square().sum(0), lambda v: v.sum(-1)).sqrt()
    cn = _per_block(C, _norm)
    return d / (2.0 ** -14 * (_norm(a)[:, None] * frob + (math.sqrt(k) + k / 16) * cn) + 2.0 ** -8 * cn)


def _sampled(step, j, seqs, heads):
    """The (token row, head) of sample j of a decode step (one token a sequence, every layer checked)."""
    return divmod((step * 1000003 + j * 7919) % (seqs * heads), heads)


def _z64_attention(s, c, layer):
    kv, q, o, _, _ = s["layers"][layer]
    dim, out = c["dim"], []
    for j in range(c["samples"]):
        row, head = _sampled(s["step"], j, c["seqs"], c["heads"])
        t = torch.arange(int(s["lens"][row]), device="cuda")
        kvr = kv[s["table"][row, t // 16], head // (c["heads"] // c["kv_heads"]), t % 16].double()
        K, V, qv, ov = kvr[:, :dim], kvr[:, dim:], q[row, head].double(), o[row, head].double()
        sc = K @ qv * s["scale"]
        m = sc.max()
        p = (sc - m).exp()
        total = p.sum()
        ref, A = p @ V / total, p @ V.abs() / total
        e = (dim + 8) * 2.0 ** -23 * s["scale"] * (K.abs() @ qv.abs()) + 2.0 ** -22 * sc.abs() + 2.0 ** -21
        E = ((p * e) @ V.abs() + ref.abs() * (p * e).sum()) / total
        spacing = 2.0 ** -126 * V.abs().sum(0) / total
        gamma = (t.numel() / 16 + 32) * 2.0 ** -22 + 2.0 ** -22 * m.abs()
        out.append((ov - ref).abs() / ((2.0 ** -7 + gamma) * (A + ref.abs()) + E + spacing + 1e-37))
    return torch.stack(out)


def exact(case, seed):
    """What run() returns, in 64 bits (counts and flags, which are whole numbers, as None)."""
    s, kind = prepare(case, seed), case["kind"]
    if kind == "serve":
        worst = []
        for slot, x, y in zip(s["slots"], s["xs"], s["ys"]):
            lin = s["guard"].layers[slot]["module"]
            worst.append(_z64(x, lin.weight.t(), y, lin.bias).max())
        return {"worst": torch.stack(worst), "unjudged": None}
    if kind == "linear":
        return {"worst": _z64(s["x"], s["w"].t(), s["y"]).max().view(1),
                "worst_rows": _z64(s["w"], s["x"].t(), s["y"].t()).max().view(1), "unjudged": None,
                "unjudged_rows": None}
    if kind == "train":
        x, w, dy = s["x"], s["w"], s["dy"]
        zs = [_z64(x, w.t(), s["y"], s["b"]).max(), _z64(dy, w, s["dx"]).max(), _z64(dy.t(), x, s["dw"]).max()]
        return {"worst": torch.stack(zs), "unjudged": None}
    if kind == "product":
        z = _z64(s["A"], s["B"], s["C"], s["bias"])
        return {"scores": z if z.dim() == 4 else z.unsqueeze(0), "unjudged": None}
    if kind == "moe":
        ends, start, zs, worst = s["offs"].tolist(), 0, [], []
        for e, end in enumerate(ends):
            if end > start:
                zs.append(_z64(s["a"][start:end], s["w"][e], s["out"][start:end]))
            worst.append(zs[-1].max() if end > start else torch.zeros((), dtype=torch.float64, device="cuda"))
            start = end
        return {"scores": torch.cat(zs), "worst": torch.stack(worst), "unjudged": None}
    if kind == "quant":
        if case["mode"] == "int8" and case["kept"]:
            return None
        if case["mode"] == "int8":
            d = _pairs(s["C"].double()) != (s["a"].double() @ _pairs(s["b"].double()).flatten(-2)).unflatten(-1, (-1, 2))
            return {"z": torch.where(d.any(-1), float("inf"), 0.0).double(), "wrong": None, "nonfinite": None}
        z = _z64_fp8(s["a"], s["sa"], s["b"], s["sb"], s["C"])
        return {"worst" if case["kept"] else "z": z.max().view(1) if case["kept"] else z, "wrong": None,
                "nonfinite": None}
    if kind == "precise":
        return {"scores": _z64_precise(s["A"], s["B"], s["C"], 16).unsqueeze(0), "unjudged": None}
    z = torch.stack([_z64_attention(s, case, i) for i in range(case["layers"])])
    return {"scores": z, "counts": None, "mismatch": None, "mismatch_last": None}
