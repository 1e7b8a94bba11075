"""The FP64 exponential and power of the column sweep against numpy in 80 bits, on the ranges that the sweep uses and at
the special cases of their arguments, and the sweep with exponents of 0, which the constants may set."""
import copy
import ctypes
import os

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from openifs_amd import build as B
from openifs_amd import cloudsc as C
from tests.helpers import columns, oracle_blocked, relrms

pytestmark = pytest.mark.gpu

# rounding to nearest 0.5 ulp, the polynomials' own error at most 0.2 ulp (0.69 is stated beside them)
ULP = 0.75


def evaluate(which, x, y=None, z=None):
    lib = ctypes.CDLL(B.DEVICE_CHECK)
    args = [torch.from_numpy(np.broadcast_to(np.asarray(0.0 if v is None else v, np.float64), np.shape(x)).copy()).cuda()
            for v in (x, y, z)]
    out = torch.empty_like(args[0])
    rc = lib.fp64_check(which, *(ctypes.c_void_p(t.data_ptr()) for t in args), ctypes.c_void_p(out.data_ptr()),
                        out.numel(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    return out.cpu().numpy()


def ulps(got, want):
    return np.max(np.abs(got.astype(np.longdouble) - want) / np.spacing(np.abs(want.astype(np.float64))).astype(np.longdouble))


@pytest.mark.parametrize("lo,hi", [(-1.0, 1.0), (-50.0, 50.0), (-700.0, 700.0)])
def test_exp(lo, hi):
    x = np.random.default_rng(1).uniform(lo, hi, 200000)
    assert ulps(evaluate(0, x), np.exp(x.astype(np.longdouble))) <= ULP


@pytest.mark.parametrize("lo,hi,ymax", [(0.5, 2.0, 4.0), (1e-14, 1e14, 3.0), (1e-300, 1e300, 1.0)])
def test_pow(lo, hi, ymax):
    rng = np.random.default_rng(2)
    x = np.exp(rng.uniform(np.log(lo), np.log(hi), 200000))
    y = rng.uniform(-ymax, ymax, x.size)
    assert ulps(evaluate(1, x, y), np.power(x.astype(np.longdouble), y.astype(np.longdouble))) <= ULP
    z = rng.uniform(-1.0, 1.0, x.size)
    want = np.power(x.astype(np.longdouble), y.astype(np.longdouble) * z.astype(np.longdouble))
    # y z is rounded to 53 bits nowhere: y log x keeps two words, and the reference's product 64
    assert ulps(evaluate(2, x, y, z), want) <= ULP + 0.05


def test_special_values():
    inf, nan = np.inf, np.nan
    x = np.array([inf, -inf, nan, 800.0, -800.0, 0.0, -0.0])
    np.testing.assert_array_equal(evaluate(0, x), [inf, 0.0, nan, inf, 0.0, 1.0, 1.0])
    bases = np.array([0.0, -0.0, inf, -inf, nan, -2.0, 1.0, 3.0, 5e-324])
    exps = np.array([0.0, -0.0, 1.0, -1.0, 2.0, -2.0, 3.0, -3.0, 0.5, -0.5])
    x, y = (v.ravel() for v in np.meshgrid(bases, exps))
    with np.errstate(all="ignore"):
        want = np.power(x, y)
    got = evaluate(1, x, y)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want), err_msg=f"{x[np.isnan(got) != np.isnan(want)]}")
    np.testing.assert_allclose(got, want, rtol=2.0 ** -52)
    # as a base: a power of exponent 0 is 1 whatever the base; one beyond the range of FP64 is not rounded to infinity
    for z in (0.4, 2.0, 0.0):
        with np.errstate(all="ignore"):
            want = np.power(np.power(x.astype(np.longdouble), y), z).astype(np.float64)
        np.testing.assert_allclose(evaluate(2, x, y, z), want, rtol=1e-15, err_msg=str(z))


@pytest.mark.parametrize("names", [["rcl_dr"], ["rcl_lam2r"], ["rcl_const6r", "rcl_const4r", "rcl_const3r"],
                                   ["rcl_kkbac", "rcl_kkbaun"], ["rcl_x2r", "rcl_const4s", "rcl_const5s", "rcl_const8s"]])
def test_sweep_with_exponents_of_zero(names, params91):
    p = copy.copy(params91)
    for n in names:
        setattr(p, n, 0.0)
    ngptot, nproma, klev = 1000, 64, 91
    f = C.BlockedFields(ngptot, nproma, klev, "dp", "cuda", fill=0.0)
    C.synth_device(f, p, 23)
    f["pclv"][:, 2, :, ::2] = 0.0  # no rain in every other column: bases of 0
    f["ptendency_cml_cld"][:, 2, :, ::2] = 0.0
    inp = {n: f[n].cpu().numpy().copy() for n in C.INPUT_NAMES}
    C.cloudsc_blocked(f, p, 900.0)
    ref = oracle_blocked("dp", p, inp, ngptot, nproma, klev, nthreads=8)
    for n in [n for n, _, r in C.BLOCKED_ARRAYS if r == "o"] + ["plude"]:
        got, want = (columns(v, nproma)[:ngptot] for v in (f[n].cpu().numpy(), ref[n]))
        written = ~np.isnan(want)
        assert np.isfinite(got[written]).all(), n
        assert relrms(got, np.where(written, want, np.nan)) <= 1e-12, n
