"""The instantiations of the FP64 column sweep that launches choose by size -- three waves to 64 columns up to 16,384
columns, one wave with the compiler's registers up to 65,536, and with registers for two waves per SIMD beyond -- give the
same columns bit for bit, and the middle one those of the FP64 oracle."""
import copy

import pytest

torch = pytest.importorskip("torch")

from openifs_amd import autotune as T
from openifs_amd import cloudsc as C
from openifs_amd import satadj as A
from tests.helpers import columns, oracle_blocked, relrms

pytestmark = pytest.mark.gpu

OUT = [n for n, _, r in C.BLOCKED_ARRAYS if r == "o"] + ["plude"]
KLEV, NB = 91, 20


@pytest.mark.parametrize("nproma", [64, 100])
@pytest.mark.parametrize("default", [True, False])
@pytest.mark.parametrize("fused", [False, True])
def test_fp64_by_size(nproma, default, fused, params91):
    params = copy.copy(params91)
    if not default:
        params.rcldiff = params.rcldiff * 1.5
    make, call = (A.FusedFields, A.satadj_cloudsc_blocked) if fused else (C.BlockedFields, C.cloudsc_blocked)
    sizes = [66000, 17000, NB * nproma]  # two waves per SIMD (plain only), one wave, three waves to 64 columns
    sets = [make(n, nproma, KLEV, "dp", "cuda", fill=0.0) for n in sizes]
    (A.synth_device if fused else C.synth_device)(sets[0], params, 31)
    for f in sets[1:]:
        for n in f.t:
            f[n].copy_(sets[0][n][:f.ngpblks])
    inp = {n: sets[2][n].cpu().numpy().copy() for n in C.INPUT_NAMES}
    for f in sets:
        call(f, params, 900.0)
    for n in OUT:
        for f in sets[:2]:
            assert torch.equal(f[n][:NB], sets[2][n]), (n, f.ngptot)
    if not fused:
        ref = oracle_blocked("dp", params, inp, NB * nproma, nproma, KLEV, nthreads=8)
        for n in OUT:
            got, want = columns(sets[1][n][:NB].cpu().numpy(), nproma), columns(ref[n], nproma)
            assert relrms(got, want) <= 1e-12, n


@pytest.mark.parametrize("prec,launches", [("dp", [(64, 0, 0), (256, 0, 0), (128, 2, 1), (512, 0, 0)]),
                                           ("sp", [(128, 4, 1), (256, 0, 0)]), ("mixed", [(128, 3, 1), (256, 4, 0)])])
def test_set_launches_have_the_same_bits(prec, launches, params91):
    """The one-wave kernel on a launch that else takes three waves, in the forms that can be set."""
    ref, f = (C.BlockedFields(1000, 64, KLEV, prec, "cuda", fill=0.0) for _ in range(2))
    C.synth_device(ref, params91, 5)
    start = {n: x.clone() for n, x in ref.t.items()}
    scope = C.lib().cloudsc_tune_get_scope(T.VARIANTS[prec], KLEV)
    was = T.get_launch(prec, KLEV)
    C.cloudsc_blocked(ref, params91, 900.0)
    try:
        for launch in launches:
            for n, x in start.items():
                f[n].copy_(x)
            T.set_launch(prec, KLEV, *launch)
            C.cloudsc_blocked(f, params91, 900.0)
            for n in OUT:
                assert torch.equal(f[n], ref[n]), (n, launch)
    finally:
        (T.set_recorded if scope == 1 else T.set_launch)(prec, KLEV, *(was if scope else (0,)))
