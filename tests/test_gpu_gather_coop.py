"""The gather backward's cooperative-row kernels at the sizes where they can
go wrong: head dims that leave lanes of a row idle, entry counts around the
chunk of 16 / 32 / 64, keys listed by no row, by one and by more rows than one
wave sums (the windowed parts), kv groups, dropout; and the slower forms that
unaligned rows take.

Reference: float64 gradients by autograd through an explicit gather.  Bars:
float32 1e-5 x max |reference|: a score is a sum of D float32 products, off by
at most D 2^-24 sum |q k| scale = 0.64 D^1.5 2^-24 (1.6e-4 at D = 256) with every
rounding aligned, and about 1 / sqrt(D) of that, 1e-5, with independent ones;
p, and with it the gradients, carry that error as a relative one.  bfloat16 and
float16: one rounding of the stored gradient, 2^-8 and 2^-11, plus the same
sums: 6e-3 and 1e-3.
"""
import time

import pytest
import torch

import elastic_sparse_attention as esa
from elastic_sparse_attention import (elastic_attention_bwd_rows, elastic_attention_rows,
                                      make_pattern, sparse_attention_bwd, sparse_attention_fwd)

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
BAR = {torch.float32: 1e-5, torch.bfloat16: 6e-3, torch.float16: 1e-3}


def inputs(B, H, Hkv, L, D, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    make = lambda h: torch.randn(B, h, L, D, generator=g).to(dtype)  # noqa: E731
    return make(H), make(Hkv), make(Hkv), make(H), g


def reference(q, k, v, go, idx, ok, scale):
    """float64 dq, dk, dv for explicit lists ``idx`` / ``ok`` [H, L, w]."""
    q, k, v, go = (t.double().requires_grad_(i < 3) for i, t in enumerate((q, k, v, go)))
    H, grp = q.shape[1], q.shape[1] // k.shape[1]
    outs = []
    for h in range(H):
        i = torch.where(ok[h], idx[h], torch.zeros_like(idx[h]))
        kk, vv = k[:, h // grp][:, i], v[:, h // grp][:, i]
        s = torch.einsum("bld,blwd->blw", q[:, h], kk) * scale
        p = torch.softmax(s.masked_fill(~ok[h], float("-inf")), -1)
        outs.append(torch.einsum("blw,blwd->bld", p, vv))
    o = torch.stack(outs, 1)
    return torch.autograd.grad(o, (q, k, v), go)


def rel(got, ref):
    return ((got.double().cpu() - ref).abs().max() / ref.abs().max()).item()


def check(got, ref, dtype):
    e = [rel(a, b) for a, b in zip(got, ref)]
    print("  dq %.2e dk %.2e dv %.2e" % tuple(e), flush=True)
    assert max(e) <= BAR[dtype]


@pytest.mark.parametrize("dtype,D", [(torch.float32, 4), (torch.float32, 32), (torch.float32, 60),
                                     (torch.float32, 128), (torch.float32, 132),
                                     (torch.float32, 256), (torch.bfloat16, 8),
                                     (torch.bfloat16, 72), (torch.bfloat16, 128),
                                     (torch.bfloat16, 256), (torch.bfloat16, 36),
                                     (torch.float16, 64), (torch.float16, 136)])
@pytest.mark.parametrize("w", [2, 16, 33, 65])
def test_operator_head_dims_and_entry_counts(dtype, D, w):
    B, H, Hkv, L = 2, 4, 2, 67
    print(f"{dtype} D={D} w={w}", flush=True)
    q, k, v, go, g = inputs(B, H, Hkv, L, D, dtype, D * 100 + w)
    idx = torch.randint(0, L, (H, L, w), generator=g)
    idx[idx == 5] = 6                        # a key no row lists
    ok = torch.rand(H, L, w, generator=g) > 0.2
    ok[:, :, 0] = True
    scale = D ** -0.5
    d = [t.to(DEV) for t in (q, k, v, idx, ok, go)]
    o, lse = sparse_attention_fwd(*d[:5], scale, H // Hkv)
    got = sparse_attention_bwd(*d[:3], o, lse, d[5], d[3], d[4], scale)
    assert got[1][:, :, 5].abs().max() == 0 and got[2][:, :, 5].abs().max() == 0
    check(got, reference(q, k, v, go, idx, ok, scale), dtype)


@pytest.mark.parametrize("dtype,D", [(torch.float32, 64), (torch.bfloat16, 96)])
@pytest.mark.parametrize("L", [511, 513, 1537])
def test_keys_that_every_row_lists(dtype, D, L):
    """Keys 0 and 7 in every row's list (segments of H / Hkv L entries: below,
    at and above the two windows one wave sums), the rest at random."""
    B, H, Hkv, w = 2, 4, 2, 12
    print(f"{dtype} D={D} L={L}", flush=True)
    q, k, v, go, g = inputs(B, H, Hkv, L, D, dtype, L)
    idx = torch.randint(0, L, (H, L, w), generator=g)
    idx[:, :, 3], idx[:, :, 5] = 0, 7
    ok = torch.ones(H, L, w, dtype=torch.bool)
    d = [t.to(DEV) for t in (q, k, v, idx, ok, go)]
    o, lse = sparse_attention_fwd(*d[:5], 0.1, H // Hkv)
    got = sparse_attention_bwd(*d[:3], o, lse, d[5], d[3], d[4], 0.1)
    check(got, reference(q, k, v, go, idx, ok, 0.1), dtype)
    again = sparse_attention_bwd(*d[:3], o, lse, d[5], d[3], d[4], 0.1)
    assert all(torch.equal(a, b) for a, b in zip(got, again))


@pytest.mark.parametrize("dtype,D", [(torch.float32, 64), (torch.bfloat16, 80)])
@pytest.mark.parametrize("dropout_p", [0.0, 0.3])
def test_unaligned_rows_agree(dtype, D, dropout_p, monkeypatch):
    """A q one element off 16 bytes takes the per-lane kernels (coop_applies
    wants every tensor aligned); both forms give the same gradients to float32
    summation order, also with dropout (the same keep decisions)."""
    B, H, Hkv, L = 2, 4, 2, 700
    pat = make_pattern(L, 64, 7, 8, H)
    q, k, v, go, _ = inputs(B, H, Hkv, L, D, dtype, 3)
    go = go.transpose(1, 2).contiguous()
    d = [t.to(DEV) for t in (q, k, v)]
    o, lse = elastic_attention_rows(*d, pat, 0.1, dropout_p=dropout_p, seed=9)
    want = elastic_attention_bwd_rows(*d, o, lse, go.to(DEV), pat, 0.1, dropout_p=dropout_p,
                                      seed=9)
    monkeypatch.setattr(esa, "_row_align", lambda t: 1)  # as given: q one element off
    off = torch.empty(q.numel() + 1, dtype=dtype, device=DEV)[1:].view(q.shape)
    off.copy_(d[0])
    got = elastic_attention_bwd_rows(off, *d[1:], o, lse, go.to(DEV), pat, 0.1,
                                     dropout_p=dropout_p, seed=9)
    check(got, [t.double().cpu() for t in want], dtype)


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 80), (torch.float16, 64)])
def test_rows_four_elements_off(dtype, D, monkeypatch):
    """q, k, v and dO 4 elements (8 bytes) off 16 bytes: as given they take the
    per-lane kernels; by default they are copied to aligned rows first, and the
    gradients are the aligned call's bit for bit."""
    B, H, Hkv, L = 2, 4, 2, 300
    pat = make_pattern(L, 48, 5, 8, H)
    q, k, v, go, _ = inputs(B, H, Hkv, L, D, dtype, 4)
    d = [t.to(DEV) for t in (q, k, v, go.transpose(1, 2).contiguous())]

    def off(t):
        r = torch.empty(t.numel() + 4, dtype=dtype, device=DEV)[4:].view(t.shape)
        assert r.data_ptr() % 16 == 8
        return r.copy_(t)

    o, lse = elastic_attention_rows(*d[:3], pat, 0.1)
    want = elastic_attention_bwd_rows(*d[:3], o, lse, d[3], pat, 0.1)
    e = [off(t) for t in d]
    copied = elastic_attention_bwd_rows(*e[:3], o, lse, e[3], pat, 0.1)
    assert all(torch.equal(a, b) for a, b in zip(copied, want))
    monkeypatch.setattr(esa, "_row_align", lambda t: 4)
    check(elastic_attention_bwd_rows(*e[:3], o, lse, e[3], pat, 0.1),
          [t.double().cpu() for t in want], dtype)


@pytest.mark.parametrize("dtype,D", [(torch.float32, 64), (torch.float32, 132),
                                     (torch.bfloat16, 96), (torch.float16, 256)])
def test_strided_rows(dtype, D):
    """q, k, v and dO as transposed views of [B, L, heads, D], as a projection
    writes them, and K and V as the first rows of a longer cache: the contiguous
    call's gradients bit for bit (the same kernels, only other strides)."""
    B, H, Hkv, L = 2, 6, 2, 333
    pat = make_pattern(L, 64, 6, 8, H)
    q, k, v, go, g = inputs(B, H, Hkv, L, D, dtype, 5)
    d = [t.to(DEV) for t in (q, k, v)]
    dout = go.transpose(1, 2).contiguous().to(DEV)
    o, lse = elastic_attention_rows(*d, pat, 0.1)
    want = elastic_attention_bwd_rows(*d, o, lse, dout, pat, 0.1)
    s = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in d]
    assert not s[0].is_contiguous()
    o1, lse1 = elastic_attention_rows(*s, pat, 0.1)
    assert torch.equal(o1, o) and torch.equal(lse1, lse)
    # dO of [B, H, L, D] storage, passed as [B, L, H, D]
    got = elastic_attention_bwd_rows(*s, o, lse, go.to(DEV).transpose(1, 2), pat, 0.1)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    cache = [torch.randn(B, Hkv, L + 50, D, generator=g).to(dtype).to(DEV) for _ in range(2)]
    for c, t in zip(cache, d[1:]):
        c[:, :, :L] = t
    got = elastic_attention_bwd_rows(d[0], cache[0][:, :, :L], cache[1][:, :, :L], o, lse, dout,
                                     pat, 0.1)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("dtype,H,Hkv,L,D,layer", [
    (torch.float32, 2, 1, 9001, 128, 4),   # 5.3 MB of keys a head: rows in turn
    (torch.float32, 3, 1, 8003, 128, 4),   # 4.7 MB: a range an XCD
    (torch.float32, 2, 2, 5001, 64, 7),    # weight 1
    (torch.bfloat16, 5, 1, 12001, 160, 6)])
def test_row_orders(dtype, H, Hkv, L, D, layer):
    """The order in which the XCDs take the rows (in ranges or in turn, by the
    keys a head's rows list) leaves no row out: the whole call against the same
    rows at 150 positions, whose few keys take ranges.  The two take chunks of
    different lengths: float32 sums, and one rounding to bf16."""
    g = torch.Generator(device=DEV).manual_seed(L)
    q, k, v = (torch.randn(1, h, L, D, generator=g, device=DEV, dtype=dtype)
               for h in (H, Hkv, Hkv))
    p = make_pattern(L, 64, layer, 8, H)
    o, lse = elastic_attention_rows(q, k, v, p, 0.1)
    pos = torch.randperm(L, generator=g, device=DEV)[:150]
    pos[:3] = torch.tensor([0, L - 1, L - 2], device=DEV)
    o1, lse1 = elastic_attention_rows(q[:, :, pos].contiguous(), k, v, p, 0.1, positions=pos)
    bar = 2e-6 if dtype == torch.float32 else 2.0 ** -8
    assert (lse[:, :, pos] - lse1).abs().max() <= 2e-6 * lse.abs().max()
    assert (o[:, pos].float() - o1.float()).abs().max() <= bar * o.abs().max().item()
    assert torch.isfinite(o.float()).all()


def test_long_rows_by_window():
    """Rows whose keys exceed an XCD's L2: layer 4's rows list keys of the last
    four sevenths of what layer 7's do and take no longer (an order that keeps a
    head on one XCD made them 10% slower; bar 3%)."""
    H, L, D = 8, 32768, 128
    g = torch.Generator(device=DEV).manual_seed(1)
    sets = [tuple(torch.randn(1, h, L, D, generator=g, device=DEV) for h in (H, 2, 2))
            for _ in range(2)]
    best = [float("inf")] * 2
    for _ in range(6):
        for i, layer in enumerate((4, 7)):
            p = make_pattern(L, 64, layer, 8, H)
            elastic_attention_rows(*sets[0], p, 0.1)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for n in range(8):
                elastic_attention_rows(*sets[n % 2], p, 0.1)
            torch.cuda.synchronize()
            best[i] = min(best[i], (time.perf_counter() - t0) / 8)
    print(f"  layer 4 {best[0] * 1e6:.0f} us, layer 7 {best[1] * 1e6:.0f} us", flush=True)
    assert best[0] <= 1.03 * best[1]
