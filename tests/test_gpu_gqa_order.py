"""The order in which the band and window kernels take the query heads of a
kv group changes no bit of a row group's result: a call with kv heads shared
by `groups` query heads against the same call with K and V repeated per query
head (groups = 1, the heads one after another).  Sizes: a last row group that
is not full, group counts that leave the last XCD short, chunks whose grids
take the few-round rule (a head's K and V above 4 MB), the window kernels."""
import time

import pytest
import torch

from elastic_sparse_attention import (ElasticSparseAttention, elastic_attention_band,
                                      elastic_attention_bwd, elastic_attention_fwd, make_pattern)

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def make(B, H, Hkv, Lq, L, D, dtype):
    g = torch.Generator(device=DEV).manual_seed(L + D)
    f = lambda h, n: torch.randn(B, h, n, D, generator=g, device=DEV, dtype=dtype)  # noqa: E731
    q, k, v = f(H, Lq), f(Hkv, L), f(Hkv, L)
    return q, k, v, k.repeat_interleave(H // Hkv, 1), v.repeat_interleave(H // Hkv, 1)


@pytest.mark.parametrize("B,H,Hkv,L,D,dtype", [(2, 8, 2, 333, 64, torch.bfloat16),
                                               (1, 6, 2, 1000, 128, torch.float16),
                                               (1, 4, 1, 8200, 128, torch.bfloat16),
                                               (1, 2, 1, 31, 64, torch.bfloat16),
                                               (3, 21, 3, 1043, 64, torch.bfloat16)])
def test_window_kernels(B, H, Hkv, L, D, dtype):
    q, k, v, kr, vr = make(B, H, Hkv, L, L, D, dtype)
    a = ElasticSparseAttention(0, 8, H, D, 64, L, num_key_value_heads=Hkv).layout(DEV)
    o, lse = elastic_attention_fwd(q, k, v, a, 0.1)
    o1, lse1 = elastic_attention_fwd(q, kr, vr, a, 0.1)
    assert torch.equal(o, o1) and torch.equal(lse, lse1)
    go = torch.randn_like(o)
    dq = elastic_attention_bwd(q, k, v, o, lse, go, a, 0.1)[0]
    dq1 = elastic_attention_bwd(q, kr, vr, o, lse, go, a, 0.1)[0]
    assert torch.equal(dq, dq1)


@pytest.mark.parametrize("H,Hkv,L,rows,D,layer", [(8, 2, 20000, 1003, 128, 4),
                                                  (8, 1, 9000, 3000, 128, 2),
                                                  (6, 3, 40000, 500, 64, 7),
                                                  (32, 4, 12000, 7000, 128, 7),
                                                  (21, 3, 9001, 2999, 128, 5)])
def test_chunks(H, Hkv, L, rows, D, layer):
    q, k, v, kr, vr = make(1, H, Hkv, rows, L, D, torch.bfloat16)
    pos = torch.arange(L - rows, L, device=DEV)
    p = make_pattern(L, 64, layer, 8, H)
    o, lse = elastic_attention_band(q, k, v, p, 0.1, positions=pos)
    o1, lse1 = elastic_attention_band(q, kr, vr, p, 0.1, positions=pos)
    # the entry rotation follows the order, so a row's sums may start at
    # another entry: equal up to float32 sums and one rounding to bf16
    assert (lse - lse1).abs().max().item() <= 1e-5
    assert (o.float() - o1.float()).abs().max().item() <= 2.0 ** -7 * o.float().abs().max().item()


def times(calls, rounds=12, n=40):
    """Seconds a call of each, the best of `rounds` blocks taken in turn."""
    best = [float("inf")] * len(calls)
    for f in calls:
        f()
    for _ in range(rounds):
        for i, f in enumerate(calls):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for _ in range(n):
                f()
            torch.cuda.synchronize()
            best[i] = min(best[i], (time.perf_counter() - t0) / n)
    return best


def test_shared_heads_cost_no_time():
    """A chunk of the sliding-window layer over shared kv heads takes no longer
    than over the same K and V repeated per query head, which reads `groups`
    times the keys and takes the heads in turn: the order must not cost what it
    is there to save.  Bar 5% (two runs of one side differ by 1%)."""
    H, Hkv, L, rows, D = 32, 8, 32768, 3000, 128
    q, k, v, kr, vr = make(1, H, Hkv, rows, L, D, torch.bfloat16)
    pos = torch.arange(L - rows, L, device=DEV)
    p = make_pattern(L, 64, 0, 8, H)
    run = lambda a, b: elastic_attention_band(q, a, b, p, 0.1, False, positions=pos)  # noqa: E731
    shared, repeated = times([lambda: run(k, v), lambda: run(kr, vr)])
    print(f"  shared {shared * 1e6:.1f} us, repeated {repeated * 1e6:.1f} us", flush=True)
    assert shared <= 1.05 * repeated
