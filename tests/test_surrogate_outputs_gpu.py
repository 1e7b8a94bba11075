"""The surrogate's output writers and the hybrid entry's merge at ragged block sizes: the network is one whose output is
its last bias, so every predicted entry is known exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DEV = "cuda"
SENTINEL = 7.25


def _case(ngptot, nproma, klev, params, seed):
    torch = pytest.importorskip("torch")
    from openifs_amd import cloudsc as C
    from openifs_amd import surrogate as S

    sur = S.Surrogate(klev, hidden=128, hidden_layers=1, max_batch=128, seed=seed)
    last = sur.mlp.n_layers - 1
    bias = np.random.default_rng(seed).standard_normal(sur.mlp.dout[last]).astype(np.float32)
    sur.mlp.weight(last, np.zeros_like(sur.mlp.weight(last)))
    sur.mlp.bias(last, bias)
    f = C.BlockedFields(ngptot, nproma, klev, "sp", DEV, fill=SENTINEL)
    if klev in (91, 137):
        C.synth_device(f, params, seed)
    else:  # no synthetic atmosphere: the prediction needs finite features and a temperature
        g = torch.Generator().manual_seed(seed)
        for n, _, r in C.BLOCKED_ARRAYS:
            if r != "o":
                x = 1.0 + torch.rand(f[n].shape, generator=g)
                f[n].copy_((200.0 * x if n == "pt" else x).to(f[n].dtype))
    return torch, C, sur, f, bias


def _expected(f, bias, params):
    """The network's outputs as {name: (columns, ...)} for all columns of the blocks (padding included)."""
    from openifs_amd import cloudsc as C
    from tests.helpers import columns

    L = f.klev
    e = {n: columns(f[n].cpu().numpy(), f.nproma).copy() for n, _, r in C.BLOCKED_ARRAYS if r == "o"}
    g = f.ngptot
    y = bias[: 6 * L].reshape(6, L)
    e["ptendency_loc_t"][:g], e["ptendency_loc_q"][:g], e["ptendency_loc_a"][:g] = y[0], y[1], y[2]
    e["ptendency_loc_cld"][:g, :4] = 0.0
    e["ptendency_loc_cld"][:g, 0], e["ptendency_loc_cld"][:g, 1] = y[3], y[4]
    liquid = columns(f["pt"].cpu().numpy(), f.nproma)[:g] > np.float32(params.rtt)
    pr = np.maximum(y[5], 0.0)
    for n in ("pfplsl", "pfplsn", "pfhpsl", "pfhpsn", "pfsqlf", "pfsqif", "pfcqnng", "pfcqlng", "pfsqrf", "pfsqsf",
              "pfcqrng", "pfcqsng", "pfsqltur", "pfsqitur"):
        e[n][:g] = 0.0
    e["pfplsl"][:g, 1:] = np.where(liquid, pr, 0.0)
    e["pfplsn"][:g, 1:] = np.where(liquid, 0.0, pr)
    e["pfhpsl"][:g] = -np.float32(params.rlvtt) * e["pfplsl"][:g]
    e["pfhpsn"][:g] = -np.float32(params.rlstt) * e["pfplsn"][:g]
    e["pcovptot"][:g, params.ncldtop - 1:] = 0.0
    e["prainfrac_toprfz"][:] = 0.0
    return e


# batches of 128 columns that end inside a block, blocks of 1 column, of odd length and of a length that allows 16-byte
# stores with a last quad that is not full; entries of a wave (16) that span several quantities (few levels)
@pytest.mark.parametrize("ngptot,nproma,klev", [(300, 75, 11), (257, 1, 20), (130, 36, 33), (515, 100, 40), (201, 64, 5),
                                                (384, 128, 137)])
def test_prediction_writes_every_output(ngptot, nproma, klev, params137):
    torch, C, sur, f, bias = _case(ngptot, nproma, klev, params137, ngptot)
    from tests.helpers import columns

    want = _expected(f, bias, params137)
    sur.predict(f, params137)
    torch.cuda.synchronize()
    for n, w in want.items():
        np.testing.assert_array_equal(columns(f[n].cpu().numpy(), nproma), w, err_msg=n)


@pytest.mark.parametrize("ngptot,nproma", [(300, 75), (257, 1), (515, 100), (384, 128)])
def test_hybrid_merges_plain_columns(ngptot, nproma, params91):
    torch, C, sur, f, bias = _case(ngptot, nproma, 91, params91, ngptot)
    from tests.helpers import columns

    def clone():
        g = C.BlockedFields(ngptot, nproma, 91, "sp", DEV)
        for k in f.t:
            g.t[k].copy_(f.t[k])
        return g

    net, plain, mix = _expected(f, bias, params91), clone(), clone()
    net["plude"] = columns(f["plude"].cpu().numpy(), nproma)
    C.cloudsc_blocked(plain, params91, 900.0)
    n = sur.hybrid(mix, params91, rerun_fraction=0.3, rerun_seed=3)
    torch.cuda.synchronize()
    got = {k: columns(mix[k].cpu().numpy(), nproma) for k in net}
    ref = {k: columns(plain[k].cpu().numpy(), nproma) for k in net}
    same = np.all(got["ptendency_loc_t"] == ref["ptendency_loc_t"], axis=1)
    same[ngptot:] = False
    assert int(same.sum()) == n and 0.15 * ngptot < n < 0.45 * ngptot
    for k in net:
        want = net[k].copy()
        want[same] = ref[k][same]
        if k == "ptendency_loc_cld":  # the fifth species is no output
            got[k], want = got[k][:, :4], want[:, :4]
        np.testing.assert_array_equal(got[k], want, err_msg=k)


# padded batches on both sides of 8,192 columns, of blocks of whole 64-column tiles (non-temporal loads from 8,192 on)
# and of ragged blocks (never): the same columns through the same network, so the same bits
@pytest.mark.parametrize("ngptot", [8064, 8065, 8192, 8321])
@pytest.mark.parametrize("nproma", [64, 128])
def test_features_do_not_depend_on_the_blocking(ngptot, nproma, params91):
    torch = pytest.importorskip("torch")
    from openifs_amd import cloudsc as C
    from openifs_amd import surrogate as S
    from tests.helpers import columns

    def fields(np_):
        f = C.BlockedFields(ngptot, np_, 91, "sp", DEV, fill=SENTINEL)  # a slot that the prediction leaves alone
        C.synth_device(f, params91, 11)
        return f

    f, g, stats = fields(nproma), fields(75), fields(75)
    for n in C.INPUT_NAMES:
        a, b = columns(f[n].cpu().numpy(), nproma)[:ngptot], columns(g[n].cpu().numpy(), 75)[:ngptot]
        np.testing.assert_array_equal(a, b, err_msg=n)
    sur = S.Surrogate(91, hidden=128, hidden_layers=1, max_batch=16384, seed=3)
    C.cloudsc_blocked(stats, params91, 3600.0)  # in-out fields change: a set of its own
    sur.fit_norm(stats, params91)
    for x in (f, g):
        sur.predict(x, params91)
    for n in ("ptendency_loc_t", "ptendency_loc_q", "ptendency_loc_a", "ptendency_loc_cld", "pfplsl", "pfplsn"):
        a, b = columns(f[n].cpu().numpy(), nproma)[:ngptot], columns(g[n].cpu().numpy(), 75)[:ngptot]
        np.testing.assert_array_equal(a, b, err_msg=n)
        assert n.startswith("pf") or n == "ptendency_loc_cld" or np.abs(a).max() > 0, n
