"""CLOUD_SATADJ's launches by size: which use non-temporal words (decided on the host), and on the GPU the same columns bit
for bit from launches of every form."""
import re

import pytest

from tests import fake_device

ROUTE = """
from openifs_amd import satadj as A

L = C.lib()
p = C.default_params(900.0, 137)
buf = np.ones(8, np.float64)  # nothing runs
res = []
for prec, ncol, nproma, klev in {cases}:
    ptr = ctypes.c_void_p(buf.ctypes.data)
    arm()
    rc = getattr(L, "cloudsc_satadj_blocked_" + prec + "_c")(
        ctypes.byref(p), ncol, nproma, klev, -(-ncol // nproma), (ctypes.c_double if prec == "dp" else ctypes.c_float)(900.0),
        *([ptr] * len(A.SATADJ_BLOCKED)), ctypes.c_void_p(0))
    res.append([rc, log()])
print(json.dumps(res))
"""
# precision, columns, NPROMA, KLEV, non-temporal
CASES = [("sp", 4096, 64, 137, 1), ("sp", 16384, 64, 137, 0), ("sp", 32768, 64, 137, 1), ("sp", 24576, 75, 91, 0),
         ("mixed", 12288, 75, 91, 1), ("mixed", 16384, 75, 91, 0), ("dp", 2048, 64, 137, 1), ("dp", 8192, 64, 137, 0),
         ("dp", 16384, 64, 137, 1)]


def test_route(tmp_path):
    res = fake_device.run(fake_device.build(str(tmp_path)), ROUTE.format(cases=[c[:4] for c in CASES]))
    got = []
    for rc, log in res:
        assert rc == 0 and len(log) == 1
        got.append(int(re.search(r"Li[12]ELb([01])E", log[0]).group(1)))
    assert got == [c[4] for c in CASES]


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["sp", "mixed", "dp"])
@pytest.mark.parametrize("nproma", [64, 75])  # two columns a lane, and one
def test_every_form_has_the_same_bits(prec, nproma, params91):
    torch = pytest.importorskip("torch")
    from openifs_amd import satadj as A

    klev, out = 91, ["ptendency_loc_t", "ptendency_loc_q", "ptendency_loc_a", "ptendency_loc_cld"]
    sizes = [45000, 24000, 900] if prec != "dp" else [24000, 12000, 900]  # non-temporal, plain, non-temporal
    sets = [A.SatadjFields(n, nproma, klev, prec, "cuda", fill=0.0) for n in sizes]
    A.synth_device(sets[0], params91, 11)
    for f in sets[1:]:
        for n in f.t:
            f[n].copy_(sets[0][n][:f.ngpblks])
    for f in sets:
        A.satadj_blocked(f, params91, 900.0)
    for n in out:
        for f in sets[1:]:
            whole = f.ngptot // nproma
            assert torch.equal(f[n][:whole], sets[0][n][:whole]), (n, f.ngptot)
