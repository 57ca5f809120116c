"""The calls a program makes of this package, as cases that can be timed and
checked: decode steps, chunked and whole prefills, training steps (forward and
backward) of the attention layer, and the operator over explicit index lists.

A case's ``kind`` says which call it is:

* ``decode``    one new row per sequence against a cache (``cache_position``)
* ``chunk``     ``rows`` consecutive rows at the end of a cache
* ``prefill``   the whole sequence, no gradients
* ``train``     the whole sequence, then the gradients of q, k and v
* ``operator``  ``ElasticSparseAttentionFunction`` over explicit index lists,
                then the gradients of q, k and v

``strided`` cases hold q, k, v as ``[B, L, H, D]`` (what a projection writes)
and pass the transposed views; the others hold ``[B, H, L, D]`` (a cache).
"""
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "elastic-sparse-attention_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from elastic_sparse_attention import (  # noqa: E402
    ElasticSparseAttention, ElasticSparseAttentionFunction)

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _case(kind, dtype, B, H, Hkv, L, D, layer, layers=8, w=64, rows=0, strided=False):
    return {"kind": kind, "dtype": dtype, "B": B, "H": H, "Hkv": Hkv, "L": L, "D": D,
            "layer": layer, "layers": layers, "w": w, "rows": rows, "strided": strided}


def listed():
    cases = {
        # one conversation's next token: latency
        "decode_one": _case("decode", "bf16", 1, 32, 8, 32768, 128, 4, rows=1),
        # a serving batch's next tokens
        "decode_batch": _case("decode", "bf16", 128, 32, 8, 32768, 128, 4, rows=1),
        # a long prompt's last part, prefilled in chunks
        "chunk_4096_of_32k": _case("chunk", "bf16", 1, 32, 32, 32768, 128, 4, rows=4096),
        # a long prompt at once (the benchmark's headline shape)
        "prefill_32k": _case("prefill", "bf16", 1, 32, 32, 32768, 128, 4),
        # prompts of an odd length, in half precision, fewer kv heads
        "prefill_ragged_f16": _case("prefill", "f16", 2, 16, 4, 5003, 64, 6, w=48, strided=True),
        # training at the benchmark's three shapes: middle and last layers
        "train_8k": _case("train", "bf16", 1, 32, 32, 8192, 128, 4),
        "train_batched_4k": _case("train", "bf16", 8, 16, 16, 4096, 64, 7, strided=True),
        "train_long_128k": _case("train", "bf16", 1, 8, 8, 131072, 128, 7),
        # ... and the first layer, whose pattern is a sliding window
        "train_window_32k": _case("train", "bf16", 1, 32, 8, 32768, 128, 0, strided=True),
        # training in full precision
        "train_f32": _case("train", "f32", 2, 8, 8, 4096, 64, 3, strided=True),
        # training a model whose head dim is neither 64 nor 128, odd length
        "train_head_dim_96": _case("train", "bf16", 1, 16, 4, 5001, 96, 5, strided=True),
        # the operator, driven by a program's own index lists
        "operator_4k": _case("operator", "bf16", 2, 8, 8, 4096, 128, 4),
    }
    return [dict(case, name=name) for name, case in cases.items()]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["decode", "chunk", "prefill", "train", "train", "train_gather", "operator"])
    layers = rng.choice([4, 8, 12, 24])
    layer = rng.randrange(layers)
    w = rng.choice([32, 48, 64, 64, 64])
    D = rng.choice([64, 128])
    dtype = rng.choice(["bf16", "bf16", "bf16", "f16"])
    Hkv = rng.choice([1, 2, 4, 8])
    H = Hkv * rng.choice([1, 2, 4])
    strided = rng.random() < 0.5
    if kind == "decode":
        L = _log_int(rng, 1000, 32768)
        return _case(kind, dtype, _log_int(rng, 1, 64), H, Hkv, L, D, layer, layers, w, 1)
    if kind == "chunk":
        L = _log_int(rng, 4000, 65536)
        return _case(kind, dtype, 1, H, Hkv, L, D, layer, layers, w, _log_int(rng, 32, 4000))
    if kind == "train_gather":  # full precision, or other head dims
        if rng.random() < 0.5:
            dtype = "f32"
            D = rng.choice([32, 64, 80, 128])
        else:
            D = rng.choice([32, 80, 96, 160])
        L = _log_int(rng, 500, 5000)
        B = rng.choice([1, 1, 2])
        return _case("train", dtype, B, min(H, 16), min(Hkv, 4), L, D, layer, layers, w, 0,
                     strided)
    if kind == "operator":
        L = _log_int(rng, 500, 5000)
        return _case(kind, rng.choice(["bf16", "f16", "f32"]), rng.choice([1, 1, 2]), min(H, 16),
                     min(Hkv, 4), L, D, layer, layers, w)
    B = rng.choice([1, 1, 2, 4])
    L = _log_int(rng, 1000, 1000000 // (B * H)) if B * H <= 32 else _log_int(rng, 1000, 12000)
    L = min(L, 100000)
    return _case(kind, dtype, B, H, Hkv, L, D, layer, layers, w, 0, strided)


def _rows(case):
    return case["rows"] if case["kind"] in ("decode", "chunk") else case["L"]


def _grads(case):
    return case["kind"] in ("train", "operator")


def _inputs(case, seed):
    """q, k, v (normalised activations: unit variance, so the scaled scores
    have unit variance too) and the output's gradient."""
    dev = torch.device("cuda", 0)
    gen = torch.Generator(device=dev).manual_seed(seed)
    dt = _DTYPES[case["dtype"]]
    B, H, Hkv, L, D = (case[x] for x in ("B", "H", "Hkv", "L", "D"))
    Lq = _rows(case)

    def make(heads, length):
        if case["strided"]:
            t = torch.randn(B, length, heads, D, generator=gen, device=dev, dtype=dt)
            return t.transpose(1, 2)
        return torch.randn(B, heads, length, D, generator=gen, device=dev, dtype=dt)

    q, k, v = make(H, Lq), make(Hkv, L), make(Hkv, L)
    g = None
    if _grads(case):
        shape = (B, H, Lq, D) if case["kind"] == "operator" else (B, Lq, H * D)
        g = torch.randn(shape, generator=gen, device=dev, dtype=dt)
    return q, k, v, g


def prepare(case, seed):
    q, k, v, g = _inputs(case, seed)
    attn = ElasticSparseAttention(
        layer_idx=case["layer"], num_hidden_layers=case["layers"],
        num_attention_heads=case["H"], head_dim=case["D"], attention_length=case["w"],
        max_seq_len=case["L"], num_key_value_heads=case["Hkv"]).to(q.device)
    state = {"kind": case["kind"], "attn": attn, "q": q, "k": k, "v": v, "g": g}
    if _grads(case):
        for t in (q, k, v):
            t.requires_grad_()
    if case["kind"] in ("decode", "chunk"):
        state["pos"] = torch.arange(case["L"] - case["rows"], case["L"], device=q.device)
    if case["kind"] == "operator":
        state["idx"] = attn.sparse_attention_indices
        state["mask"] = attn.sparse_causal_mask
    return state


def run(state):
    q, k, v, attn = state["q"], state["k"], state["v"], state["attn"]
    kind = state["kind"]
    if kind in ("decode", "chunk"):
        return attn(q, k, v, cache_position=state["pos"])[0]
    if kind == "prefill":
        return attn(q, k, v)[0]
    if kind == "operator":
        out = ElasticSparseAttentionFunction.apply(q, k, v, state["idx"], state["mask"],
                                                   attn.scaling, attn.num_kv_groups)
    else:
        out = attn(q, k, v)[0]
    dq, dk, dv = torch.autograd.grad(out, (q, k, v), state["g"])
    return {"out": out.detach(), "dq": dq, "dk": dk, "dv": dv}


def _pairs(case):
    """(query row, key) pairs of one head and batch element."""
    L, w, n = case["L"], case["w"], _rows(case)
    first = L - n
    short = max(0, min(L, w) - first)  # rows with fewer than w keys: first .. w - 1
    return sum(range(first + 1, first + short + 1)) + (n - short) * w


def work(case):
    B, H, Hkv, L, D = (case[x] for x in ("B", "H", "Hkv", "L", "D"))
    es = 4 if case["dtype"] == "f32" else 2
    Lq = _rows(case)
    pairs = B * H * _pairs(case)
    rows = B * H * Lq * D * es                       # q, or out
    keys = min(B * Hkv * L, pairs) * D * es          # k, or v: no more than is listed
    if not _grads(case):
        # scores and weighted sum: 2 D flops each per pair
        return {"bytes": 2 * rows + 2 * keys, "flops": 4 * D * pairs}
    lists = H * L * case["w"] * 16 if case["kind"] == "operator" else 0
    # q, k, v and the output's gradient read; out, dq, dk, dv written; scores
    # and weighted sum, then dP, dV, dQ and dK
    return {"bytes": 4 * rows + 4 * keys + lists, "flops": 12 * D * pairs}


def tolerance(case):
    # four times what the path is off its 64-bit value: outputs and gradients
    # in bf16 2.4e-3, in f16 3e-4, in f32 5e-7 (all sums in 32 bits)
    return {"rel": {"bf16": 1e-2, "f16": 1.5e-3, "f32": 4e-6}[case["dtype"]]}


# ---------------------------------------------------------------------------
# the same values from plain torch, in 64 bits
# ---------------------------------------------------------------------------
def _index_rows(case, head, pos):
    """The keys that the rows at positions ``pos`` list in ``head``, and which
    of them count, by the pattern's definition (each step rounds to float32):
    [rows, w] on the CPU."""
    w, H = case["w"], case["H"]
    alpha = case["layer"] / max(case["layers"] - 1, 1)
    end = torch.clamp(pos, min=w - 1)
    distance = w * (1 - alpha) + (end + 1) * alpha
    start = (end + 1 - distance).round().clamp(min=0).long()
    spacing = (end + 1 - start) / w
    offsets = start[:, None] + (torch.arange(w + 1)[None] * spacing[:, None]).round().long()
    t = torch.tensor(head) / (H - 1) if H > 1 else torch.tensor(0.0)
    idx = (offsets[:, :w].float() * (1 - t) + (offsets[:, 1:] - 1).float() * t).round().long()
    return idx, idx <= pos[:, None]


def exact(case, seed):
    q, k, v, g = _inputs(case, seed)
    B, H, Hkv, L, D = (case[x] for x in ("B", "H", "Hkv", "L", "D"))
    Lq = _rows(case)
    pos = torch.arange(L - Lq, L)
    scale = D ** -0.5
    dev = q.device
    f64 = dict(dtype=torch.float64, device=dev)
    # the gradients' float64 sums; outputs in the layout run() gives them
    out = torch.empty(B, H, Lq, D, **f64)
    if _grads(case):
        dq = torch.empty(B, H, Lq, D, **f64)
        dk, dv = torch.zeros(B, Hkv, L, D, **f64), torch.zeros(B, Hkv, L, D, **f64)
        go = g if case["kind"] == "operator" else g.view(B, Lq, H, D).transpose(1, 2)
    step = 4096
    for h in range(H):
        kvh = h // (H // Hkv)
        for r0 in range(0, Lq, step):
            idx, ok = (x.to(dev) for x in _index_rows(case, h, pos[r0:r0 + step]))
            idx = torch.where(ok, idx, torch.zeros_like(idx))
            n = idx.shape[0]
            for b in range(B):
                qr = q[b, h, r0:r0 + n].double()
                kr = k[b, kvh][idx].double()
                vr = v[b, kvh][idx].double()
                s = torch.matmul(kr, qr[:, :, None])[:, :, 0] * scale
                p = torch.softmax(s.masked_fill(~ok, float("-inf")), dim=-1)
                o = torch.matmul(p[:, None], vr)[:, 0]
                out[b, h, r0:r0 + n] = o
                if not _grads(case):
                    continue
                gr = go[b, h, r0:r0 + n].double()
                dp = torch.matmul(vr, gr[:, :, None])[:, :, 0]
                ds = p * (dp - (gr * o).sum(-1, keepdim=True)) * scale
                dq[b, h, r0:r0 + n] = torch.matmul(ds[:, None], kr)[:, 0]
                flat = idx.reshape(-1)
                dk[b, kvh].index_add_(0, flat, (ds[:, :, None] * qr[:, None]).reshape(-1, D))
                dv[b, kvh].index_add_(0, flat, (p[:, :, None] * gr[:, None]).reshape(-1, D))
    if case["kind"] != "operator":
        out = out.transpose(1, 2).reshape(B, Lq, H * D)
    if not _grads(case):
        return out
    return {"out": out, "dq": dq, "dk": dk, "dv": dv}
