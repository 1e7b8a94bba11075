"""CLOUDSC2, CLOUDST and CLOUD_S_LAYER in large launches: which of them take the large form (decided on the host), and on
the GPU its columns bit for bit those of a small launch."""
import re

import pytest

from openifs_amd import cloudsc as C
from openifs_amd import cloudsc2 as C2
from tests import fake_device

ROUTE = """
from openifs_amd import cloudsc2 as C2

L = C.lib()
p = C.default_params(900.0, 137)
p2 = C2.default_params2(p)
some = np.ones(1, np.float64)  # nothing runs
ptr = ctypes.c_void_p(some.ctypes.data)
arm()
res = []
for prec, ncol, nproma, klev in {cases}:
    for name, narr in (("cloudsc2", len(C2.CLOUDSC2_ARRAYS)), ("cloudst", len(C2.CLOUDST_ARRAYS))):
        arm()
        rc = getattr(L, name + "_blocked_" + prec + "_c")(
            ctypes.byref(p), ctypes.byref(p2), ptr, ncol, nproma, 1, klev, -(-ncol // nproma), 0,
            (ctypes.c_double if prec == "dp" else ctypes.c_float)(900.0), *([ptr] * narr), ctypes.c_void_p(0))
        res.append([rc, log()])
print(json.dumps(res))
"""
# precision, columns, NPROMA, KLEV, large form of CLOUDSC2 and of CLOUDST
CASES = [("sp", 2048, 64, 137, 0, 0), ("sp", 16384, 64, 137, 0, 0), ("sp", 24576, 64, 137, 1, 0), ("sp", 32768, 128, 137, 1, 1),
         ("dp", 8192, 64, 137, 0, 0), ("dp", 16384, 64, 137, 1, 1), ("sp", 32768, 32, 91, 0, 0), ("sp", 65536, 32, 91, 1, 1),
         ("dp", 65536, 16, 91, 1, 1), ("sp", 65536, 16, 91, 0, 0), ("sp", 131072, 100, 137, 0, 0), ("dp", 131072, 75, 91, 0, 0)]


def test_route(tmp_path):
    res = fake_device.run(fake_device.build(str(tmp_path)), ROUTE.format(cases=[c[:4] for c in CASES]))
    got = []
    for rc, log in res:
        assert rc == 0 and len(log) == 1
        uni, large, layer = re.search(r"kernelI[fd]Lb([01])ELb([01])ELb([01])E", log[0]).groups()
        got.append((int(uni), int(large), int(layer)))
    assert got == [(int(c[2] % 64 == 0), form, 0) for c in CASES for form in c[4:]]


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["cloudsc2", "cloudst", "layer-cloudsc2", "layer-cloudst"])
# aligned blocks beyond 300 MB; ragged blocks of whole lines, whose groups are ordered (FP64 in blocks of 48 too)
@pytest.mark.parametrize("prec,ncol,nproma", [("sp", 45000, 64), ("dp", 22000, 128), ("sp", 66000, 32), ("dp", 66000, 48)])
def test_large_form_has_the_small_bits(which, prec, ncol, nproma, params91):
    torch = pytest.importorskip("torch")
    klev, nb = 91, 9
    p2 = C2.default_params2(params91)
    p2.lepcld2 = int(which != "layer-cloudst")
    f = C2.synth_device(params91, 3, ncol, nproma, klev, prec, "cuda", fill=0.0)
    ceta = torch.from_numpy(C2.reference_eta(klev)).to("cuda", f["papp1"].dtype)
    if which.startswith("layer"):
        src = f
        f = {lay: src[c2] for lay, c2 in C2.LAYER_FROM_CLOUDSC2.items()}
        f["pa"] = torch.rand(f["pq"].shape, generator=torch.Generator(device="cuda").manual_seed(1), device="cuda",
                             dtype=f["pq"].dtype)
        for name, kind, role, _ in C2.LAYER_ARRAYS:
            if role == "o":
                f[name] = torch.zeros(C2.layer_shape(kind, nproma, klev, f["pq"].shape[0]), dtype=f["pq"].dtype, device="cuda")
        call, outs = C2.cloud_s_layer_blocked, [n for n, _, r, _ in C2.LAYER_ARRAYS if r == "o"]
    elif which == "cloudst":
        for n, _, _ in C2.CLOUDST_ARRAYS:
            if n not in f:
                f[n] = torch.zeros_like(f["papp1"])
        call, outs = C2.cloudst_blocked, [n for n, _, r in C2.CLOUDST_ARRAYS if r == "o"]
    else:
        call, outs = C2.cloudsc2_blocked, [n for n, _, r in C2.CLOUDSC2_ARRAYS if r == "o"]
    blocks = f["plude"].shape[0]
    starts = [0, blocks // 2, blocks - nb]
    small = [{n: x[b:b + nb].clone() for n, x in f.items()} for b in starts]
    call(f, params91, p2, ceta, ncol, nproma, klev, 900.0, prec)
    for b, s in zip(starts, small):
        n = nb * nproma if b + nb < blocks else ncol - b * nproma
        call(s, params91, p2, ceta, n, nproma, klev, 900.0, prec)
        for name in outs:
            assert torch.equal(s[name], f[name][b:b + nb]), f"{name} block {b}"
