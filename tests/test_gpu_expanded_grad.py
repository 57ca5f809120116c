"""An incoming gradient that is one value expanded over the output (all
strides 0, as out.sum().backward() gives it) through the gather backward."""
import pytest
import torch

from elastic_sparse_attention import ElasticSparseAttention

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gradient_of_a_sum(dtype):
    """out.sum().backward(): the incoming gradient is one value expanded over
    the output (all strides 0)."""
    B, H, L, D = 1, 2, 90, 96
    g = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn(B, H, L, D, generator=g).to(dtype) for _ in range(3))
    m = ElasticSparseAttention(3, 8, H, D, 64, L)
    a = [t.to(DEV).requires_grad_() for t in (q, k, v)]
    m(*a)[0].sum().backward()
    b = [t.to(DEV).requires_grad_() for t in (q, k, v)]
    out = m(*b)[0]
    out.backward(torch.ones_like(out))
    assert all(torch.equal(x.grad, y.grad) for x, y in zip(a, b))
