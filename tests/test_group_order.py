"""The order in which the column kernels give work-groups to the XCDs, and the groups of a launch with padding columns.  No
GPU needed, but for the columns themselves."""
import ctypes

import numpy as np
import pytest

from openifs_amd import build as B
from openifs_amd import cloudsc as C
from tests import fake_device

GROUPS = """
L = C.lib()
p = C.default_params(900.0, 91)
some = np.ones(1 << 20, np.float64)  # nothing runs
ptr = ctypes.c_void_p(some.ctypes.data)
res = []
for prec, ncol, nproma in {cases}:
    arm()
    rc = getattr(L, "cloudsc_blocked_" + prec + "_c")(
        ctypes.byref(p), ncol, nproma, 91, -(-ncol // nproma), (ctypes.c_double if prec == "dp" else ctypes.c_float)(900.0),
        *([ptr] * len(C.BLOCKED_ARRAYS)), ctypes.c_void_p(0))
    res.append([rc, [[int(x) for x in l.split()[2:]] for l in log()]])
print(json.dumps(res))
"""


@pytest.mark.parametrize("n", [1, 5, 7, 8, 9, 15, 16, 257, 513, 1024, 2047])
def test_order(n):
    """Every group once; an XCD's groups are neighbours, in order."""
    lib = ctypes.CDLL(B.DEVICE_CHECK)
    order = [lib.group_order(i, n) for i in range(n)]
    assert sorted(order) == list(range(n))
    for x in range(min(8, n)):
        mine = order[x::8]
        assert mine == list(range(mine[0], mine[0] + len(mine)))


# precision, columns, NPROMA -> work-groups and lanes of the sweep, work-groups of the kernel that clears padding columns
CASES = {("sp", 131072, 100): (512, 256, 1), ("sp", 131073, 100): (513, 256, 0), ("dp", 65536, 100): (256, 256, 1),
         ("mixed", 131072, 1000): (512, 256, 4), ("sp", 131072, 128): (512, 256, 0), ("sp", 32768, 100): (512, 192, 1),
         ("sp", 32768, 1000): (512, 192, 1), ("sp", 1, 128): (2, 192, 0), ("sp", 16000, 1000): (250, 192, 0),
         ("sp", 15900, 1000): (250, 192, 0)}


def test_groups_without_columns(tmp_path):
    """Launches that fill the chip have no group of padding columns alone: one XCD would have 65 full groups of the first
    case's 513."""
    res = fake_device.run(fake_device.build(str(tmp_path)), GROUPS.format(cases=list(CASES)))
    for (case, (groups, lanes, clear)), (rc, log) in zip(CASES.items(), res):
        assert rc == 0
        assert log[-1] == [groups, 1, 1, lanes], case
        assert log[:-1] == ([[clear, 1, 1, 256]] if clear else []), case


@pytest.mark.gpu
@pytest.mark.parametrize("prec,ncol,nproma", [("sp", 131072, 100), ("dp", 65536, 100), ("mixed", 65500, 900), ("sp", 32500, 900)])
def test_padding_columns(prec, ncol, nproma, params91):
    """The columns that a small launch gives, bit for bit, in the first and the last blocks; of the padding columns
    PRAINFRAC_TOPRFZ is 0 and nothing else is touched."""
    torch = pytest.importorskip("torch")
    out = [n for n, _, r in C.BLOCKED_ARRAYS if r == "o"] + ["plude"]
    f = C.BlockedFields(ncol, nproma, 91, prec, "cuda", fill=float("nan"))
    C.synth_device(f, params91, 41)
    nb = 3
    small = [C.BlockedFields(nb * nproma, nproma, 91, prec, "cuda", fill=float("nan")),
             C.BlockedFields(ncol - (f.ngpblks - nb) * nproma, nproma, 91, prec, "cuda", fill=float("nan"))]
    starts = [0, f.ngpblks - nb]
    for s, b in zip(small, starts):
        for n in f.t:
            s[n].copy_(f[n][b:b + nb])
    for g in [f, *small]:
        C.cloudsc_blocked(g, params91, 900.0)
    for s, b in zip(small, starts):
        for n in out:
            np.testing.assert_array_equal(f[n][b:b + nb].cpu().numpy(), s[n].cpu().numpy(), err_msg=f"{n} {b}")
    last = ncol - (f.ngpblks - 1) * nproma
    assert (f["prainfrac_toprfz"][-1, last:] == 0).all()
    assert torch.isnan(f["ptendency_loc_t"][-1, :, last:]).all() and torch.isnan(f["pfplsl"][-1, :, last:]).all()
