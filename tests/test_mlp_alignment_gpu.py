"""Products and networks on matrices that are aligned to their elements only (a view into a larger buffer) and with odd
leading dimensions: the bits of the aligned ones."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from openifs_amd import surrogate as S

pytestmark = pytest.mark.gpu


def shifted(x, n):
    """A copy of x that starts n elements into its buffer."""
    buf = torch.empty(x.numel() + n, dtype=x.dtype, device="cuda")
    y = buf[n:].view(x.shape)
    y.copy_(x)
    return y


# 64 x 64 tiles, 128 x 128 and 256 x 256 where the operands are aligned
@pytest.mark.parametrize("M,N,K", [(128, 128, 32), (256, 128, 96), (2048, 1024, 64), (4096, 4096, 128)])
@pytest.mark.parametrize("da,db,dc,pad", [(1, 0, 0, 0), (0, 3, 0, 0), (4, 2, 1, 0), (0, 0, 1, 1), (0, 0, 0, 3), (7, 5, 3, 2)])
def test_product_is_exact(M, N, K, da, db, dc, pad):
    g = torch.Generator().manual_seed(K)
    a = shifted(torch.randint(-8, 9, (M, K), generator=g).bfloat16(), da)
    b = shifted(torch.randint(-8, 9, (N, K), generator=g).bfloat16(), db)
    guard = 12345.0
    c = shifted(torch.full((M, N + pad), guard), dc)
    S._call("cloudsc_mlp_gemm_tn", a.data_ptr(), K, b.data_ptr(), K, c.data_ptr(), N + pad, M, N, K, S._stream(a.device))
    assert torch.equal(c[:, :N], a.float() @ b.float().T)
    assert (c[:, N:] == guard).all()


@pytest.mark.parametrize("n_in,hidden,layers,n_out,M", [(128, 128, 1, 128, 128), (128, 384, 2, 128, 1152),
                                                        (640, 1024, 2, 256, 2048)])
@pytest.mark.parametrize("dx,dt,dw", [(1, 0, 0), (0, 1, 3), (6, 2, 1)])
def test_training_has_the_aligned_bits(n_in, hidden, layers, n_out, M, dx, dt, dw):
    g = torch.Generator().manual_seed(M + dx)
    x = torch.randn(M, n_in, generator=g).bfloat16()
    t, w = torch.randn(M, n_out, generator=g), torch.rand(n_out, generator=g)
    p, q = (S.MLP(n_in, hidden, layers, n_out, M, seed=4) for _ in range(2))
    xt = x.T.contiguous().cuda()
    for _ in range(2):
        p.train_step(x.cuda(), xt, t.cuda(), w.cuda(), 1e-3)
        q.train_step(shifted(x, dx), xt, shifted(t, dt), shifted(w, dw), 1e-3)
    p.gradients(x.cuda(), xt, t.cuda(), w.cuda())
    q.gradients(shifted(x, dx), xt, shifted(t, dt), shifted(w, dw))
    for l in range(p.n_layers):
        np.testing.assert_array_equal(p.weight(l), q.weight(l))
        np.testing.assert_array_equal(p.bias(l), q.bias(l))
        np.testing.assert_array_equal(p.weight_grad(l), q.weight_grad(l))
        np.testing.assert_array_equal(p.bias_grad(l), q.bias_grad(l))
    assert abs(p.last_loss() - q.last_loss()) <= 1e-5 * p.last_loss()  # summed by atomics


@pytest.mark.parametrize("M", [128, 2048, 16384])
def test_forward_has_the_aligned_bits(M):
    m = S.MLP(384, 1024, 2, 1024, M, seed=5)
    x = torch.randn(M, 384, generator=torch.Generator().manual_seed(5)).bfloat16()
    y = m.forward(x.cuda())
    assert torch.equal(y, m.forward(shifted(x, 1), shifted(torch.zeros_like(y), 1)))
