"""The training products of the MLP at the sizes where their tiles, splits and steps can go wrong, and the statistics of
the surrogate's features and targets against numpy."""
import numpy as np
import pytest

from oracle import mlp_ref as R

pytestmark = pytest.mark.gpu

DEV = "cuda"


def case(seed, n_in, hidden, layers, n_out, M):
    torch = pytest.importorskip("torch")
    from openifs_amd import surrogate as S

    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, n_in, generator=g).bfloat16()
    t = torch.randn(M, n_out, generator=g)
    w = torch.rand(n_out, generator=g)
    dev = [x.to(DEV), x.T.contiguous().to(DEV), t.to(DEV), w.to(DEV)]
    return [S.MLP(n_in, hidden, layers, n_out, M, seed=seed) for _ in range(2)], x, t, w, dev


# 64 x 64 tiles (few groups) and 128 x 128; a contraction of 2 steps (128) and of 544 = 8.5 steps (batch 2,176 split in
# 4); a split in 2 (1,152); widths that are no multiple of 256
SHAPES = [(128, 128, 1, 128, 128), (128, 384, 2, 128, 1152), (256, 128, 2, 384, 2176), (640, 1024, 2, 256, 2048)]


@pytest.mark.parametrize("n_in,hidden,layers,n_out,M", SHAPES)
def test_gradients_match_cpu_reference(n_in, hidden, layers, n_out, M):
    (m, _), x, t, w, dev = case(n_in + M, n_in, hidden, layers, n_out, M)
    m.gradients(*dev)
    ws = [m.weight(l) for l in range(m.n_layers)]
    bs = [m.bias(l) for l in range(m.n_layers)]
    loss, dws, dbs = R.loss_and_grads(ws, bs, x.float().numpy(), t.numpy(), w.numpy(), emulate=True)
    assert abs(m.last_loss() - loss) <= 1e-4 * loss
    for l in range(m.n_layers):
        # bf16 roundings that fall the other way: relative RMS far below the bf16 resolution of an entry
        assert np.linalg.norm(m.weight_grad(l) - dws[l]) <= 2e-3 * np.linalg.norm(dws[l]), f"dW layer {l}"
        assert np.linalg.norm(m.bias_grad(l) - dbs[l]) <= 2e-3 * np.linalg.norm(dbs[l]), f"db layer {l}"


@pytest.mark.parametrize("n_in,hidden,layers,n_out,M", SHAPES)
def test_train_step_equals_gradients_then_adam(n_in, hidden, layers, n_out, M):
    """The update fused with the sums of the partial products gives the separate calls' parameters bit for bit."""
    (a, b), _, _, _, dev = case(7 + M, n_in, hidden, layers, n_out, M)
    for _ in range(3):
        a.train_step(*dev, 1e-3)
        b.gradients(*dev)
        b.adam(1e-3)
    for l in range(a.n_layers):
        np.testing.assert_array_equal(a.weight(l), b.weight(l))
        np.testing.assert_array_equal(a.bias(l), b.bias(l))
        np.testing.assert_array_equal(a.weight_grad(l), b.weight_grad(l))
        np.testing.assert_array_equal(a.bias_grad(l), b.bias_grad(l))


# 256 of the 256 x 256 tiles, contractions of 1 to 8 steps (the ring's unrolled steps are 6) and one that is no multiple
# of 64 (the smaller tiles); entries are small whole numbers, so every sum is exact
@pytest.mark.parametrize("K", [64, 128, 192, 256, 320, 384, 448, 512, 832, 96])
def test_large_product_is_exact(K):
    torch = pytest.importorskip("torch")
    from openifs_amd import surrogate as S

    g = torch.Generator().manual_seed(K)
    a = torch.randint(-8, 9, (4096, K + 8), generator=g).bfloat16().to(DEV)[:, :K]
    b = torch.randint(-8, 9, (4096, K), generator=g).bfloat16().to(DEV)
    assert torch.equal(S.gemm_tn(a, b), a.float() @ b.float().T)


def test_large_forward_equals_small_forward():
    """A batch on the large tiles gives the rows that small batches give, bit for bit (hidden and output layers)."""
    torch = pytest.importorskip("torch")
    from openifs_amd import surrogate as S

    m = S.MLP(384, 1024, 2, 1024, 16384, seed=5)
    x = torch.randn(16384, 384, generator=torch.Generator().manual_seed(5)).bfloat16().to(DEV)
    y = m.forward(x)
    for r in (0, 128, 8064, 16256):
        assert torch.equal(y[r:r + 128], m.forward(x[r:r + 128].contiguous())), r


@pytest.mark.parametrize("ngptot,nproma", [(300, 128), (257, 75)])
def test_statistics_match_numpy(ngptot, nproma, params91):
    """Mean and spread of all 14 features and 6 targets per level (FP64 sums on both sides; entries that are floored
    or left unscaled are those the header names)."""
    torch = pytest.importorskip("torch")
    from openifs_amd import cloudsc as C
    from openifs_amd import surrogate as S
    from tests.helpers import columns
    from tests.test_surrogate_gpu import _features_numpy

    klev = 91
    f = C.BlockedFields(ngptot, nproma, klev, "sp", DEV, fill=0.0)
    C.synth_device(f, params91, 19)
    plude = f["plude"].clone()
    C.cloudsc_blocked(f, params91, 900.0)
    f["plude"].copy_(plude)
    sur = S.Surrogate(klev, hidden=128, hidden_layers=1, max_batch=128, seed=1)
    sur.fit_norm(f, params91)
    nrm = sur.norm()
    x = _features_numpy(f, klev, params91).astype(np.float64)
    spread = x.std(axis=0).reshape(14, klev)
    assert np.all(np.abs(nrm["mu_x"] - x.mean(axis=0)) <= 1e-5 * np.abs(x).max(axis=0))
    scaled = spread > 2e-3 * spread.max(axis=1, keepdims=True)
    np.testing.assert_allclose(nrm["sd_x"].reshape(14, klev)[scaled], spread[scaled], rtol=1e-3)
    col = lambda n: columns(f[n].cpu().numpy(), nproma)[:ngptot].astype(np.float64)  # noqa: E731
    cld = col("ptendency_loc_cld")
    y = np.concatenate([col("ptendency_loc_t"), col("ptendency_loc_q"), col("ptendency_loc_a"), cld[:, 0], cld[:, 1],
                        (col("pfplsl") + col("pfplsn"))[:, 1:]], axis=1)
    np.testing.assert_allclose(nrm["mu_y"], y.mean(axis=0), rtol=1e-5, atol=1e-5 * np.abs(y).max())
    live = nrm["wgt_y"] > 0
    np.testing.assert_allclose(nrm["sd_y"][live], y.std(axis=0)[live], rtol=1e-3)


def test_activation_over_its_whole_range():
    """silu of biases from -92 to 92, each through one weight: bf16 resolution of the value, also beyond -87, where
    1 / (1 + exp(-z)) is denormal."""
    torch = pytest.importorskip("torch")
    from openifs_amd import surrogate as S

    m = S.MLP(128, 128, 1, 128, 128, seed=3)
    z = np.concatenate([np.linspace(-92, -86, 64), np.linspace(-86, 92, 64)]).astype(np.float32)
    scale = np.where(z < -40, 2.0 ** 100, 1.0).astype(np.float32)
    m.weight(0, np.zeros((128, 128), np.float32))
    m.bias(0, z)
    m.weight(1, np.diag(scale))
    m.bias(1, np.zeros(128, np.float32))
    y = m.forward(torch.zeros(128, 128, dtype=torch.bfloat16, device=DEV)).cpu().numpy().astype(np.float64)
    with np.errstate(over="ignore"):  # FP32 throughout: exp(-z) overflows below -88.7 and the activation is 0
        want = (z * (np.float32(1) / (np.float32(1) + np.exp(-z)))).astype(np.float64) * scale
    assert np.all(np.abs(y - want) <= 2.0 ** -8 * np.abs(want) + 1e-30)
