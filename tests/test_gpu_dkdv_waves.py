"""The band dK/dV with several waves per key block, at sizes where the rule
picks 1, 2, 4 and 8: kv groups that divide among the waves and that do not, a
last key block that is not full, the last layer's split first block
(groups * q_len > 6144), layer 0's window form, both 16-bit types.

test_matches_block_sparse: the block-sparse kernels' dK and dV, which round P
and dS to the same 16 bits and sum in float32.  Bar: each of a gradient's products carries
two roundings of 2^-9 in the mean (bf16; 2^-12 in f16) and the stored gradients
one more each; independent over the >= 64 products of a key, at most 4 2^-9 of the
largest gradient: 8e-3 and 1e-3."""
import time

import pytest
import torch

from elastic_sparse_attention import (ElasticSparseAttention, build_indices,
                                      elastic_attention_bwd, elastic_attention_fwd)

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
BAR = {torch.bfloat16: 8e-3, torch.float16: 1e-3}


@pytest.mark.parametrize("B,H,Hkv,L,D,layer,dtype", [
    (1, 8, 1, 500, 128, 7, torch.bfloat16), (1, 3, 1, 777, 64, 7, torch.bfloat16),
    (1, 8, 1, 2000, 64, 7, torch.float16), (2, 4, 2, 8200, 128, 7, torch.bfloat16),
    (1, 4, 4, 9000, 128, 7, torch.bfloat16), (1, 4, 1, 1003, 128, 3, torch.bfloat16),
    (1, 6, 2, 1500, 64, 4, torch.bfloat16), (1, 4, 4, 8200, 128, 5, torch.float16),
    (1, 4, 2, 17000, 64, 2, torch.bfloat16), (1, 2, 2, 150, 128, 4, torch.bfloat16),
    (1, 6, 2, 333, 128, 0, torch.bfloat16), (1, 4, 1, 16, 64, 0, torch.float16)])
def test_matches_block_sparse(B, H, Hkv, L, D, layer, dtype):
    g = torch.Generator(device=DEV).manual_seed(L + H)
    q, k, v = (torch.randn(B, h, L, D, generator=g, device=DEV, dtype=dtype)
               for h in (H, Hkv, Hkv))
    lay = ElasticSparseAttention(layer, 8, H, D, 64, L, num_key_value_heads=Hkv).layout(DEV)
    o, lse = elastic_attention_fwd(q, k, v, lay, D ** -0.5)
    go = torch.randn(B, L, H, D, generator=g, device=DEV, dtype=dtype)
    run = lambda kind: elastic_attention_bwd(q, k, v, o, lse, go, lay, D ** -0.5,  # noqa: E731
                                             dq_kernel="band", dkdv_kernel=kind)
    got, ref = run("band"), run("tile")
    for a, b in zip(got[1:], ref[1:]):
        err = ((a.float() - b.float()).abs().max() / b.float().abs().max()).item()
        print(f"  {err:.2e}", flush=True)
        assert err <= BAR[dtype]
    again = run("band")
    assert all(torch.equal(a, b) for a, b in zip(got, again))


def test_shorter_call_is_not_slower():
    """The rule's several waves a block must not cost time where they are taken:
    with whole kv heads on the XCDs a grid of 5.9 rounds of resident waves
    against one of 6.03 at the same pattern, where one wave takes a block.  Two
    waves made the shorter call 15% slower; with one it is 2% faster (bar 4%,
    two runs of one side differ by 1%)."""
    H, Hkv, D = 16, 8, 128
    calls = []
    for L in (24161, 24700):
        g = torch.Generator(device=DEV).manual_seed(L)
        q, k, v = (torch.randn(1, h, L, D, generator=g, device=DEV, dtype=torch.bfloat16)
                   for h in (H, Hkv, Hkv))
        lay = ElasticSparseAttention(6, 8, H, D, 32, L, num_key_value_heads=Hkv).layout(DEV)
        o, lse = elastic_attention_fwd(q, k, v, lay, 0.1)
        calls.append(lambda a=(q, k, v, o, lse, torch.randn_like(o), lay, 0.1):
                     elastic_attention_bwd(*a, dq_kernel="band", dkdv_kernel="band"))
    best = [float("inf")] * 2
    for _ in range(8):
        for i, f in enumerate(calls):
            f()
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for _ in range(8):
                f()
            torch.cuda.synchronize()
            best[i] = min(best[i], (time.perf_counter() - t0) / 8)
    print(f"  {best[0] * 1e6:.0f} us, longer {best[1] * 1e6:.0f} us", flush=True)
    assert best[0] <= 1.04 * best[1]


def gradients64(q, k, v, o, lse, go, idx, ok, scale):
    """float64 dK and dV of the lists ``idx`` / ``ok`` [H, L, w] for the output
    and lse that the forward stored: p = exp(s - lse), dS = p (dP - dO . O)."""
    B, H, L, D = q.shape
    grp = H // k.shape[1]
    dk = torch.zeros(k.shape, dtype=torch.float64, device=DEV)
    dv = torch.zeros_like(dk)
    for b in range(B):
        for h in range(H):
            for r0 in range(0, L, 2048):
                r = slice(r0, r0 + 2048)
                i, m = idx[h, r], ok[h, r]
                kk, vv = k[b, h // grp][i].double(), v[b, h // grp][i].double()
                qr, gr = q[b, h, r].double(), go[b, r, h].double()
                s = torch.bmm(kk, qr[:, :, None])[:, :, 0] * scale
                p = torch.exp(s - lse[b, h, r, None].double()) * m
                dp = torch.bmm(vv, gr[:, :, None])[:, :, 0]
                delta = (gr * o[b, r, h].double()).sum(-1, keepdim=True)
                ds = p * (dp - delta) * scale
                flat = i.reshape(-1)
                dk[b, h // grp].index_add_(0, flat, (ds[:, :, None] * qr[:, None]).reshape(-1, D))
                dv[b, h // grp].index_add_(0, flat, (p[:, :, None] * gr[:, None]).reshape(-1, D))
    return dk, dv


@pytest.mark.parametrize("B,H,Hkv,L,D,layer,dtype", [
    (1, 4, 4, 5000, 128, 4, torch.bfloat16),    # 2 waves share each head's steps
    (1, 6, 2, 9001, 128, 5, torch.bfloat16),    # ... of 3 heads
    (1, 16, 8, 4400, 64, 2, torch.float16),     # one wave, two heads
    (1, 16, 4, 5990, 128, 4, torch.bfloat16),   # 4 waves, a head each
    (1, 4, 4, 34000, 128, 7, torch.bfloat16),   # 2 waves, block 0 split
    (1, 8, 2, 3001, 64, 7, torch.float16),      # 8 waves, block 0 split
    (1, 4, 2, 31000, 64, 7, torch.bfloat16),    # 4 waves, block 0 split
    (1, 8, 4, 8201, 128, 0, torch.bfloat16),    # layer 0, one wave over two heads
    (1, 8, 1, 2001, 64, 0, torch.float16),      # ... two waves over eight
    (1, 4, 2, 16387, 64, 1, torch.bfloat16)])   # 2 waves, a head each
def test_matches_float64_by_key(B, H, Hkv, L, D, layer, dtype):
    """Each key's row of dK and dV against float64, by the row's own size.  A
    gradient's products carry the rounding of P or dS, at most u = 2^-8 of each
    (float16 2^-11), independent ones a sum of at most u / sqrt(3) of the root
    sum of their squares, which is about the row's root mean square r.  The
    largest of 10^7 such errors is 5.5 of these, 3.2 u r; 4.5 u r allows for r
    (of 64 or 128 dims, sums of few products) to be 1.4 times too small; and the
    stored value's own rounding, u max.  One pair of a row's 64 and more left out
    is off by 10 u r and more."""
    u = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    g = torch.Generator(device=DEV).manual_seed(L + H)
    q, k, v = (torch.randn(B, h, L, D, generator=g, device=DEV, dtype=dtype)
               for h in (H, Hkv, Hkv))
    lay = ElasticSparseAttention(layer, 8, H, D, 64, L, num_key_value_heads=Hkv).layout(DEV)
    scale = D ** -0.5
    o, lse = elastic_attention_fwd(q, k, v, lay, scale)
    go = torch.randn(B, L, H, D, generator=g, device=DEV, dtype=dtype)
    got = elastic_attention_bwd(q, k, v, o, lse, go, lay, scale, dq_kernel="band",
                                dkdv_kernel="band")[1:]
    idx, ok = build_indices(lay.pattern, DEV, torch.int64)
    ref = gradients64(q, k, v, o, lse, go, idx, ok, scale)
    for name, a, b in zip(("dk", "dv"), got, ref):
        err = (a.double() - b).abs().amax(-1)
        bar = 4.5 * u * b.pow(2).mean(-1).sqrt() + u * b.abs().amax(-1) + 1e-7
        worst = (err / bar).max().item()
        print(f"  {name} {worst:.2f} of the bar", flush=True)
        assert worst <= 1
