"""The work that is timed when the kernels change: what a SiQ-VL training or
evaluation step has this package do, one layer or block per case, through the
entry points a training script calls.

A case is a dict of plain values.  Its ``kind`` picks the path:

* ``attn``       ``flash_attn_varlen_func`` on a packed batch;
* ``rope_attn``  ``flash_attn_varlen_rope_func`` (rotary embedding + attention);
* ``ce``         ``fused_linear_cross_entropy`` (lm_head + loss);
* ``proj``       ``pixel_shuffle_linear`` (vision-to-text projector);
* ``splice``     ``splice_vision_tokens`` (embedding gather + vision rows).

``grad`` says whether the backward runs too.  Packed sequence lengths follow
from the case alone (``_lengths``), values from the seed alone.
"""

from __future__ import annotations

import math
import random

import torch

from siq_vl_amd.attention import flash_attn_varlen_func, flash_attn_varlen_rope_func
from siq_vl_amd.cross_entropy import fused_linear_cross_entropy
from siq_vl_amd.projector import pixel_shuffle_linear
from siq_vl_amd.splice import splice_vision_tokens

VOCAB = 151936  # Qwen2.5's table
IGNORE = -100
DEV = "cuda"


# --------------------------------------------------------------------------- the cases
def _attn(name, heads, kv_heads, dim, causal, tokens, seqs, spread, grad, kind="attn", cos="bf16"):
    case = {"name": name, "kind": kind, "heads": heads, "kv_heads": kv_heads, "dim": dim, "causal": causal,
            "tokens": tokens, "seqs": seqs, "spread": spread, "grad": grad}
    if kind == "rope_attn":
        case["cos"] = cos
    return case


def _ce(name, rows, hidden, vocab, mode, masked):
    return {"name": name, "kind": "ce", "rows": rows, "hidden": hidden, "vocab": vocab, "mode": mode, "masked": masked}


def _proj(name, tiles, side, dim, factor, out, grad):
    return {"name": name, "kind": "proj", "tiles": tiles, "side": side, "dim": dim, "factor": factor, "out": out,
            "grad": grad}


def _splice(name, tokens, vision, hidden, vocab, dtype, grad):
    return {"name": name, "kind": "splice", "tokens": tokens, "vision": vision, "hidden": hidden, "vocab": vocab,
            "dtype": dtype, "grad": grad}


def listed():
    return [
        # one short prompt through a 0.5B decoder layer's attention: launch and latency bound, the smallest call
        _attn("attn prompt", 14, 2, 64, True, 197, 1, "equal", False),
        # an evaluation batch of the 0.5B decoder: forward only, 8 ragged sequences
        _attn("attn eval packed", 14, 2, 64, True, 4096, 8, "ragged", False),
        # the ordinary training batch of the 1.5B decoder: 32 packed sequences of very different lengths
        _attn("attn train packed", 12, 2, 128, True, 16384, 32, "ragged", True),
        # the vision tower's attention while it is trained: 16 images of 1024 patches, every patch sees every other
        _attn("attn train tower", 16, 16, 64, False, 16384, 16, "equal", True),
        # long documents beside short ones: a half, a quarter, the rest in short pieces
        _attn("attn train skewed", 12, 2, 128, True, 32768, 24, "skewed", True),
        # one decoder layer's rotary embedding and attention on an odd-sized batch
        _attn("rope attn train", 12, 2, 128, True, 5003, 9, "ragged", True, kind="rope_attn"),
        # the lm_head and loss of the 1.5B model in full training: the largest call
        _ce("ce train", 16384, 1536, VOCAB, "train", 0.3),
        # the same with a frozen lm_head (projector or LoRA training) of the 0.5B model, an odd row count
        _ce("ce frozen head", 4099, 896, VOCAB, "frozen", 0.3),
        # evaluation loss of a small batch
        _ce("ce eval", 1000, 1536, VOCAB, "eval", 0.5),
        # the projector in training, tower included: 16 tiles of 32 x 32 patches
        _proj("proj train", 16, 32, 1024, 2, 1536, True),
        # the projector on one image of 27 x 27 patches, 3 x 3 merged: an odd-sized small call
        _proj("proj one image", 1, 27, 1152, 3, 896, False),
        # embeddings of a training batch with 16 images of 256 tokens, and the table's gradient
        _splice("splice train", 16384, 4096, 1536, VOCAB, "bf16", True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["attn", "attn", "attn", "rope_attn", "ce", "ce", "proj", "splice"])
    if kind in ("attn", "rope_attn"):
        heads, kv_heads, dim = rng.choice([(14, 2, 64), (12, 2, 128), (16, 16, 64), (28, 4, 128), (12, 12, 64)])
        causal = kv_heads != heads or kind == "rope_attn"
        tokens = _log_int(rng, 128, 32768)
        seqs = rng.randint(1, max(1, min(48, tokens // 100)))
        spread = rng.choice(["equal", "ragged", "ragged", "skewed"])
        if not causal:
            seqs, spread = max(1, seqs, tokens // 4096), "equal"
        case = _attn("", heads, kv_heads, dim, causal, tokens, seqs, spread, rng.random() < 0.7, kind,
                     rng.choice(["bf16", "fp32"]))
        while work(case)["flops"] > 3.2e12:  # no dearer than the listed ones
            case["tokens"] //= 2
    elif kind == "ce":
        hidden = rng.choice([320, 896, 1536, 2048])
        rows = min(_log_int(rng, 64, 16384), 16384 * 1536 // hidden)
        case = _ce("", rows, hidden, rng.choice([VOCAB, VOCAB, 32008, 49152]), rng.choice(["train", "frozen", "eval"]),
                   rng.choice([0.0, 0.3, 0.7]))
    elif kind == "proj":
        factor = rng.choice([1, 2, 3])
        case = _proj("", _log_int(rng, 1, 24), factor * rng.randint(4, 32 // factor), rng.choice([768, 1024, 1152]), factor,
                     rng.choice([896, 1536, 2048]), rng.random() < 0.6)
    else:
        tokens = _log_int(rng, 128, 40000)
        case = _splice("", tokens, int(tokens * rng.choice([0.1, 0.25, 0.6])), rng.choice([896, 1536, 2048]), VOCAB,
                       rng.choice(["bf16", "bf16", "fp32"]), rng.random() < 0.6)
    del case["name"]
    return case


# --------------------------------------------------------------------------- sizes that follow from a case
def _lengths(case):
    """The packed sequences' lengths (each at least 1, their sum is ``tokens``)."""
    total, n = case["tokens"], case["seqs"]
    if case["spread"] == "equal":
        return [total // n + (1 if i < total % n else 0) for i in range(n)]
    rng = random.Random(total * 1009 + n)
    if case["spread"] == "skewed" and n > 2:
        head = [total // 2, total // 4]
        weights, left = [rng.uniform(81, 600) for _ in range(n - 2)], total - sum(head)
    else:  # ragged: lognormal around the mean, as packed chat samples are
        head, weights, left = [], [math.exp(0.75 * rng.gauss(0, 1)) for _ in range(n)], total
    lens = [max(1, int(left * w / sum(weights))) for w in weights]
    lens[lens.index(max(lens))] += left - sum(lens)
    return head + lens


def _pairs(case):
    return sum(n * (n + 1) // 2 if case["causal"] else n * n for n in _lengths(case))


def _elem(dtype):
    return 4 if dtype == "fp32" else 2


def work(case):
    if case["kind"] in ("attn", "rope_attn"):
        t, hq, hkv, d = case["tokens"], case["heads"], case["kv_heads"], case["dim"]
        qb, kb = 2 * t * hq * d, 2 * t * hkv * d
        nbytes, flops = 2 * qb + 2 * kb, 4.0 * d * hq * _pairs(case)  # q, k, v -> out
        if case["grad"]:
            nbytes, flops = nbytes + 2 * qb + 2 * kb, flops * 3  # dout -> dq, dk, dv (the rest is read once already)
        if case["kind"] == "rope_attn":
            nbytes += 2 * t * d * _elem(case["cos"])
        return {"bytes": nbytes, "flops": flops}
    if case["kind"] == "ce":
        n, h, v = case["rows"], case["hidden"], case["vocab"]
        counted = sum(1 for y in _label_mask(case) if y)
        grads = {"train": 3, "frozen": 2, "eval": 1}[case["mode"]]
        nbytes = 2 * n * h + 2 * v * h + 8 * n
        nbytes += (2 * n * h if grads > 1 else 0) + (2 * v * h if grads > 2 else 0)
        return {"bytes": nbytes, "flops": 2.0 * grads * counted * h * v}
    if case["kind"] == "proj":
        k = case["factor"] ** 2 * case["dim"]
        m = case["tiles"] * (case["side"] // case["factor"]) ** 2
        nbytes, flops = 2 * (m * k + case["out"] * k + m * case["out"]), 2.0 * m * k * case["out"]
        return {"bytes": nbytes * (2 if case["grad"] else 1), "flops": flops * (3 if case["grad"] else 1)}
    e, h = _elem(case["dtype"]), case["hidden"]
    nbytes = case["tokens"] * (2 * e * h + 8)
    if case["grad"]:  # the upstream gradient read, the vision rows' and the table's gradients written
        nbytes += e * h * (case["tokens"] + case["vision"] + case["vocab"])
    return {"bytes": nbytes, "flops": 0.0}


def _label_mask(case):
    """Rows whose label counts: the head of each sample (prompt, image) is ignored."""
    rng, mask = random.Random(case["rows"]), []
    while len(mask) < case["rows"]:
        n = max(16, min(4096, int(400 * math.exp(0.75 * rng.gauss(0, 1)))))
        ignored = int(round(case["masked"] * n))
        mask += [False] * ignored + [True] * (n - ignored)
    mask = mask[:case["rows"]]
    mask[-1] = True
    return mask


# --------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, *shape, std=1.0, dtype=torch.bfloat16):
    return (std * torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)).to(dtype)


def _zipf(g, n, vocab):
    """Token ids as text has them: the frequency of an id falls as 1 / rank."""
    u = torch.rand(n, generator=g, device=DEV, dtype=torch.float64)
    return (torch.exp(u * math.log(vocab)).to(torch.int64) - 1).clamp_(0, vocab - 1)


def _cos_sin(case):
    pos = torch.cat([torch.arange(n) for n in _lengths(case)]).to(DEV, torch.float32)
    inv = 1.0 / 1e6 ** (torch.arange(0, case["dim"], 2, device=DEV, dtype=torch.float32) / case["dim"])
    ang = torch.outer(pos, inv)
    ang = torch.cat([ang, ang], dim=1)
    dtype = torch.float32 if case["cos"] == "fp32" else torch.bfloat16
    return ang.cos().to(dtype), ang.sin().to(dtype)


def prepare(case, seed):
    g = _gen(seed)
    st = {"case": case}
    if case["kind"] in ("attn", "rope_attn"):
        t, d = case["tokens"], case["dim"]
        lens = _lengths(case)
        cu = [0]
        for n in lens:
            cu.append(cu[-1] + n)
        st["cu"] = torch.tensor(cu, dtype=torch.int32, device=DEV)
        st["longest"] = max(lens)
        st["in"] = [_normal(g, t, case["heads"], d), _normal(g, t, case["kv_heads"], d), _normal(g, t, case["kv_heads"], d)]
        if case["kind"] == "rope_attn":
            st["cos"], st["sin"] = _cos_sin(case)
        if case["grad"]:
            st["up"] = _normal(g, t, case["heads"], d)
    elif case["kind"] == "ce":
        n, h, v = case["rows"], case["hidden"], case["vocab"]
        w = _normal(g, v, h, std=0.02)
        y = _zipf(g, n, v)
        # a trained model's rows lean towards their label, some hardly and some strongly
        lean = 16 * torch.rand(n, 1, generator=g, device=DEV) / (0.02 ** 2 * h)
        hid = (torch.randn(n, h, generator=g, device=DEV) + lean * w[y].float()).to(torch.bfloat16)
        y[~torch.tensor(_label_mask(case), device=DEV)] = IGNORE
        st["in"] = [hid, w]
        st["labels"] = y
        # the trainer hands the number of supervised tokens to a training step; evaluation takes the mean
        st["items"] = None if case["mode"] == "eval" else (y != IGNORE).sum()
    elif case["kind"] == "proj":
        r, k = case["factor"], case["factor"] ** 2 * case["dim"]
        st["in"] = [_normal(g, case["tiles"], case["side"] ** 2, case["dim"]), _normal(g, case["out"], k, std=0.02)]
        if case["grad"]:
            st["up"] = _normal(g, case["tiles"], (case["side"] // r) ** 2, case["out"])
    else:
        t, nv, v = case["tokens"], case["vision"], case["vocab"]
        dtype = torch.float32 if case["dtype"] == "fp32" else torch.bfloat16
        ids = _zipf(g, t, v - 1)
        # the image placeholders in runs, spread evenly over the batch
        run = min(256, max(1, nv))
        nruns = (nv + run - 1) // run
        gap = t // max(1, nruns)
        for i in range(nruns):
            n = min(run, nv - i * run)
            ids[i * gap:i * gap + n] = v - 1
        st["ids"] = ids.view(1, t)
        st["image"] = v - 1
        st["in"] = [_normal(g, v, case["hidden"], std=0.02, dtype=dtype), _normal(g, int((ids == v - 1).sum()), case["hidden"],
                                                                              dtype=dtype)]
        if case["grad"]:
            st["up"] = _normal(g, 1, t, case["hidden"], dtype=dtype)
    trained = case["mode"] != "eval" if case["kind"] == "ce" else case["grad"]
    if trained:
        frozen = 1 if case.get("mode") == "frozen" else None
        for i, x in enumerate(st["in"]):
            x.requires_grad_(i != frozen)
    return st


# --------------------------------------------------------------------------- one pass
def run(st):
    case = st["case"]
    if case["kind"] == "attn":
        out = flash_attn_varlen_func(*st["in"], st["cu"], st["cu"], st["longest"], st["longest"], causal=case["causal"])
    elif case["kind"] == "rope_attn":
        q, k, v = st["in"]
        out = flash_attn_varlen_rope_func(q, k, v, st["cos"], st["sin"], st["cu"], st["cu"], st["longest"], st["longest"],
                                          causal=case["causal"])
    elif case["kind"] == "ce":
        hid, w = st["in"]
        loss = fused_linear_cross_entropy(hid, w, st["labels"], num_items_in_batch=st["items"])
        leaves = [x for x in st["in"] if x.requires_grad]
        return [loss.detach(), *torch.autograd.grad(loss, leaves)] if leaves else [loss]
    elif case["kind"] == "proj":
        out = pixel_shuffle_linear(*st["in"], case["factor"])
    else:
        out = splice_vision_tokens(st["ids"], *st["in"], st["image"])
    if not case["grad"]:
        return [out]
    return [out.detach(), *torch.autograd.grad(out, st["in"], st["up"])]


# --------------------------------------------------------------------------- how far results may differ
def tolerance(case):
    # Each about four times the distance between this package's result and ``exact`` (2-norms).
    if case["kind"] in ("attn", "rope_attn"):
        return {"rel": 1.2e-2}  # bf16 probabilities, score gradients and outputs
    if case["kind"] == "ce":
        return {"rel": 1e-5} if case["mode"] == "eval" else {"rel": 1e-2}  # fp32 sums; bf16 gradients
    if case["kind"] == "proj":
        return {"rel": 7e-3}  # bf16 outputs of fp32 sums
    return "exact"  # rows copied; the table's gradient in a stated order


# --------------------------------------------------------------------------- the same in 64 bits
def _f64(x):
    return x.detach().double()


def _exact_attention(case, q, k, v, up):
    """Per sequence and head, dense; gradients of sum(out * up) when ``up`` is given."""
    scale, rep = case["dim"] ** -0.5, case["heads"] // case["kv_heads"]
    out = torch.empty_like(q)
    dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
    a = 0
    for n in _lengths(case):
        s = slice(a, a + n)
        hidden = torch.ones(n, n, dtype=torch.bool, device=DEV).triu_(1) if case["causal"] else None
        for h in range(case["heads"]):
            qs, ks, vs = q[s, h], k[s, h // rep], v[s, h // rep]
            p = scale * (qs @ ks.T.contiguous())
            if hidden is not None:
                p.masked_fill_(hidden, -math.inf)
            p = torch.softmax(p, dim=1)
            out[s, h] = p @ vs
            if up is None:
                continue
            us = up[s, h]
            dv[s, h // rep] += p.T.contiguous() @ us
            ds = us @ vs.T.contiguous()
            ds -= (us * out[s, h]).sum(1, keepdim=True)
            ds *= p
            ds *= scale
            dq[s, h] = ds @ ks
            dk[s, h // rep] += ds.T.contiguous() @ qs
        a += n
    return [out] if up is None else [out, dq, dk, dv]


def _turn(x, cos, sin):
    half = x.shape[-1] // 2
    return x * cos[:, None] + torch.cat([-x[..., half:], x[..., :half]], dim=-1) * sin[:, None]


def _turn_back(g, cos, sin):
    half = g.shape[-1] // 2
    gs = g * sin[:, None]
    return g * cos[:, None] + torch.cat([gs[..., half:], -gs[..., :half]], dim=-1)


def _exact_ce(case, st):
    hid, w = (_f64(x) for x in st["in"])
    y = st["labels"]
    keep = torch.nonzero(y != IGNORE).flatten()
    grads = case["mode"] != "eval"
    dh = torch.zeros_like(hid) if grads else None
    dw = torch.zeros_like(w) if case["mode"] == "train" else None
    total, wt = torch.zeros((), dtype=torch.float64, device=DEV), w.T.contiguous()
    for c in range(0, keep.numel(), 1024):
        rows = keep[c:c + 1024]
        z = hid[rows] @ wt
        at = (torch.arange(rows.numel(), device=DEV), y[rows])
        lse = torch.logsumexp(z, dim=1)
        total += (lse - z[at]).sum()
        if not grads:
            continue
        z = z.sub_(lse[:, None]).exp_()
        z[at] -= 1
        z /= keep.numel()
        dh[rows] = z @ w
        if dw is not None:
            dw += z.T.contiguous() @ hid[rows]
    return [total / keep.numel()] + ([dh] if grads else []) + ([dw] if dw is not None else [])


def exact(case, seed):
    st = prepare(case, seed)
    up = _f64(st["up"]) if "up" in st else None
    if case["kind"] == "attn":
        return _exact_attention(case, *(_f64(x) for x in st["in"]), up)
    if case["kind"] == "rope_attn":
        q, k, v = (_f64(x) for x in st["in"])
        cos, sin = _f64(st["cos"]), _f64(st["sin"])
        res = _exact_attention(case, _turn(q, cos, sin), _turn(k, cos, sin), v, up)
        if up is not None:
            res[1], res[2] = _turn_back(res[1], cos, sin), _turn_back(res[2], cos, sin)
        return res
    if case["kind"] == "ce":
        return _exact_ce(case, st)
    if case["kind"] == "proj":
        x, w = (_f64(t) for t in st["in"])
        r, n, d = case["factor"], case["side"] // case["factor"], case["dim"]
        xs = x.view(-1, n, r, n, r, d).permute(0, 1, 3, 2, 4, 5).reshape(-1, r * r * d)
        y = (xs @ w.T.contiguous()).view(case["tiles"], n * n, -1)
        if up is None:
            return [y]
        g = up.reshape(-1, case["out"])
        dx = (g @ w).view(-1, n, n, r, r, d).permute(0, 1, 3, 2, 4, 5).reshape(x.shape)
        return [y, dx, g.T.contiguous() @ xs]
    table, vision = (_f64(t) for t in st["in"])
    ids = st["ids"].view(-1)
    image = ids == st["image"]
    out = table[ids]
    out[image] = vision
    if up is None:
        return [out.view(1, *out.shape)]
    g = up.view(-1, case["hidden"])
    dtable = torch.zeros_like(table)
    dtable.index_add_(0, ids[~image], g[~image])
    return [out.view(1, *out.shape), dtable, g[image]]
