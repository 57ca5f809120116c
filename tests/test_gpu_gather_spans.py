"""The gather kernels at rows far apart: K and V heads, and q and dO batch
elements, whose bytes from the first row to past the last are the most that
32-bit buffer offsets reach (2^31 - 8192, exclusive) and the first that they do
not, where the forward reads rows by pointer and the backward takes its
per-lane kernels.  Five rows of each in 2 GiB of storage, against the same rows
side by side.

Bars: the same products in float32, the sums of another chunk length or kernel:
float32 2e-6 x max |reference| (64 to 96 products, 2^-24 each, independent);
bfloat16 one rounding of the stored value more, 2^-8."""
import pytest
import torch

from elastic_sparse_attention import sparse_attention_bwd, sparse_attention_fwd

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
BAR = {torch.float32: 2e-6, torch.bfloat16: 2.0 ** -8}
MOST = (1 << 31) - 8192  # kMaxSpan
ROWS = 5


def apart(t, past):
    """``t`` [1, heads, ROWS, D] with its rows as far apart as the buffer loads
    reach, or (``past``) 16 bytes further a row; a row's heads side by side."""
    _, heads, n, D = t.shape
    es = t.element_size()
    step = 16 // es
    # span = (heads - 1) D + (n - 1) stride + D elements
    stride = (MOST // es - heads * D - 1) // (n - 1) // step * step
    assert ((n - 1) * stride + heads * D) * es < MOST
    if past:
        stride += step
        assert ((n - 1) * stride + heads * D) * es >= MOST
    store = torch.empty((n - 1) * stride + heads * D, dtype=t.dtype, device=DEV)
    out = store.as_strided(t.shape, (store.numel(), D, stride, 1))
    out.copy_(t)
    return out


def rel(a, b):
    return ((a.double() - b.double()).abs().max() / b.double().abs().max()).item()


@pytest.mark.parametrize("dtype,D", [(torch.float32, 64), (torch.bfloat16, 96)])
@pytest.mark.parametrize("past", [False, True])
def test_rows_far_apart(dtype, D, past):
    H, w = 2, 70
    g = torch.Generator().manual_seed(D)
    make = lambda h: torch.randn(1, h, ROWS, D, generator=g).to(dtype).to(DEV)  # noqa: E731
    q, k, v, go = make(H), make(1), make(1), make(H)
    idx = torch.randint(0, ROWS, (H, ROWS, w), generator=g)
    ok = torch.rand(H, ROWS, w, generator=g) > 0.3
    ok[:, :, 0] = True
    idx, ok = idx.to(DEV), ok.to(DEV)
    o, lse = sparse_attention_fwd(q, k, v, idx, ok, 0.1, H)
    grads = sparse_attention_bwd(q, k, v, o, lse, go, idx, ok, 0.1)
    kf, vf = apart(k, past), apart(v, past)
    print(f"{dtype} forward", flush=True)
    o1, lse1 = sparse_attention_fwd(q, kf, vf, idx, ok, 0.1, H)
    errs = [rel(o1, o), rel(lse1, lse)]
    print(f"{dtype} backward, K and V apart", flush=True)
    errs += [rel(a, b) for a, b in zip(sparse_attention_bwd(q, kf, vf, o, lse, go, idx, ok, 0.1),
                                       grads)]
    del kf, vf
    print(f"{dtype} backward, q and dO apart", flush=True)
    qf, gf = apart(q, past), apart(go, past)
    errs += [rel(a, b) for a, b in zip(sparse_attention_bwd(qf, k, v, o, lse, gf, idx, ok, 0.1),
                                       grads)]
    print("  " + " ".join("%.1e" % e for e in errs), flush=True)
    assert max(errs) <= BAR[dtype]
