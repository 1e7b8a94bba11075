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


@pytest.mark.parametrize("nproma,default", [(64, True), (100, True), (64, False), (100, False)])
@pytest.mark.parametrize("fused", [False, True])
def test_fp64_at_two_waves_per_simd_equals_one(nproma, default, fused, params91):
    """Launches of more waves than the chip has SIMDs use another instantiation; the columns are the same bit for bit."""
    import copy

    from openifs_amd import satadj as A

    params = copy.copy(params91)
    if not default:
        params.rcldiff = params.rcldiff * 1.5

    make = A.FusedFields if fused else C.BlockedFields
    big, small = (make(n, nproma, 91, "dp", "cuda", fill=0.0) for n in (66000, 40 * nproma))
    (A.synth_device if fused else C.synth_device)(big, params, 5)
    for n in big.t:
        small[n].copy_(big[n][:40])
    call = A.satadj_cloudsc_blocked if fused else C.cloudsc_blocked
    call(big, params, 900.0)
    call(small, params, 900.0)
    torch.cuda.synchronize()
    for n in OUT:
        assert torch.equal(big[n][:40], small[n]), n


def _block_call(params, inp, prec, n, klev, kidia, kfdia):
    """Columns 0 .. n-1 of a one-block field set through the per-block entry, outputs prefilled with NaN."""
    arrs = {}
    for name, _, role in C.BLOCKED_ARRAYS:
        if name in inp:
            x = inp[name][0][..., :n]
            arrs[name] = np.asfortranarray(x.T if x.ndim < 3 else x.transpose(2, 1, 0))
    full = C.allocate_block(n, klev, prec, fill=np.nan)
    for name, x in arrs.items():
        full[name][...] = x
    C.CLOUDSC(params, kidia, kfdia, n, klev, 900.0, full, precision=prec)
    return full


def test_per_block_entry_at_all_image_sizes(params137):
    """Blocks that grow and shrink the page-locked image, that exceed its limit (1,000 FP64 columns: array by array) and
    that cover a window, from one thread and from several at once, against the blocked launch."""
    from concurrent.futures import ThreadPoolExecutor

    n = 1000
    inp, out = run(params137, "dp", n, n, 137, 71)

    def check(m, kidia, kfdia):
        got = _block_call(params137, inp, "dp", m, 137, kidia, kfdia)
        for name in OUT:
            ref = out[name][0][..., :m]
            ref = (ref.T if ref.ndim < 3 else ref.transpose(2, 1, 0)).copy()
            rows = slice(kidia - 1, kfdia)
            np.testing.assert_array_equal(got[name][rows], ref[rows], err_msg=f"{name} {m} {kidia}:{kfdia}")
        assert np.isnan(got["ptendency_loc_t"][kfdia:]).all() and np.isnan(got["pfplsl"][: kidia - 1]).all()

    for m, kidia, kfdia in [(8, 1, 8), (300, 1, 300), (33, 1, 20), (n, 1, n), (64, 1, 64)]:
        check(m, kidia, kfdia)
    with ThreadPoolExecutor(4) as ex:
        list(ex.map(lambda m: check(m, 1, m), [40, 100, 8, 64, 200, 16, 128, 32]))


@pytest.mark.parametrize("prec", ["sp", "mixed"])
@pytest.mark.parametrize("nproma,ncldtop,default", [(64, None, True), (100, None, True), (32, 2, True), (75, 91, True),
                                                    (128, 2, False), (33, None, False)])
def test_three_wave_kernel_equals_one_wave_kernel(prec, nproma, ncldtop, default, params91):
    """Small launches take the kernel of three waves to 64 columns, large ones that of one: bit for bit the same, for a
    first cloud level at the top, at the bottom and between, and blocks that leave parts of waves empty."""
    import copy

    params = copy.copy(params91)
    if ncldtop:
        params.ncldtop = ncldtop
    if not default:
        params.rcldiff = params.rcldiff * 1.5
    big = C.BlockedFields(49300, nproma, 91, prec, "cuda", fill=0.0)
    C.synth_device(big, params, 9)
    starts = {1: 0, 40 * nproma: 0, 41 * nproma - 7: 3}
    small = {}
    for n, b0 in starts.items():
        f = C.BlockedFields(n, nproma, 91, prec, "cuda", fill=0.0)
        for name in f.t:
            f[name].copy_(big[name][b0:b0 + f.ngpblks])
        small[n] = f
    C.cloudsc_blocked(big, params, 900.0)
    for n, b0 in starts.items():
        f = small[n]
        C.cloudsc_blocked(f, params, 900.0)
        torch.cuda.synchronize()
        for name in OUT:
            got = columns(f[name].cpu().numpy(), nproma)[:n]
            want = columns(big[name][b0:b0 + f.ngpblks].cpu().numpy(), nproma)[:n]
            np.testing.assert_array_equal(got, want, err_msg=f"{name} {n}")
