"""The CLOUDSC column sweep on the GPU at the sizes where its launch can go wrong: grids that are no multiple of 8
work-groups (the work-group order of the XCDs), blocks aligned to waves and not, ragged last blocks."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from openifs_amd import cloudsc as C
from tests.helpers import columns, oracle_blocked, relrms

pytestmark = pytest.mark.gpu

OUT = [n for n, _, r in C.BLOCKED_ARRAYS if r == "o"] + ["plude"]


def run(params, prec, ngptot, nproma, klev, seed):
    f = C.BlockedFields(ngptot, nproma, klev, prec, "cuda", fill=float("nan"))
    C.synth_device(f, params, seed)
    inp = {n: f[n].cpu().numpy().copy() for n in C.INPUT_NAMES}
    C.cloudsc_blocked(f, params, 900.0)
    torch.cuda.synchronize()
    return inp, {n: f[n].cpu().numpy() for n in OUT}


@pytest.mark.parametrize("ngptot,nproma", [(1, 64), (2300, 64), (2300, 100), (4353, 64), (4353, 75)])
def test_fp64_on_grids_of_any_size(ngptot, nproma, params91):
    """FP64 to 1e-12 of the FP64 oracle, the padding columns untouched."""
    inp, out = run(params91, "dp", ngptot, nproma, 91, 61)
    ref = oracle_blocked("dp", params91, inp, ngptot, nproma, 91, nthreads=8)
    for n in OUT:
        g, r = columns(out[n], nproma), columns(ref[n], nproma)
        np.testing.assert_array_equal(np.isnan(g), np.isnan(r), err_msg=n)
        assert relrms(g, r) <= 1e-12, n
