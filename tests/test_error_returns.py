"""A call that returns an error leaves no work behind that still reads or writes what the caller, or the thread's next
call, may free or overwrite: every HIP call of an entry is made to fail in turn.  No GPU needed."""
import pytest

from tests import fake_device

BLOCK = """
flags = {flags}
klon, klev, prec = {klon}, 91, {prec!r}
p = C.default_params(900.0, klev)
p.lcldbud = flags
b = C.synth_host(p, 3, klon, klon, klev, prec)
kf = C.budget_fields(flags)
a = C.allocate_block(klon, klev, prec, kfldx=kf, fill=0.0)
for k, x in b.items():
    a[k][...] = x[0].T if x[0].ndim < 3 else x[0].transpose(2, 1, 0)
if flags:
    for n, kind in C.BUDGET_ARRAYS:
        shape = (klon,) if kind == "1di" else (klon, klev)
        a[n] = np.zeros(shape, np.int32 if kind == "1di" else a["pt"].dtype, order="F")

def call():
    C.CLOUDSC(p, 1, klon, klon, klev, 900.0, a, prec, kfldx=kf)

arm()
call()
arm()
call()
res = [["", 0, True, fake.fake_pending(None)]]
for name in ("hipLaunchKernel", "hipMemcpyAsync", "hipHostMalloc", "hipMalloc", "hipGetDevice"):
    arm()
    call()
    for i in range(1, calls(name) + 1):
        arm(name, i)
        try:
            call()
            ok = True
        except C.CloudscError:
            ok = False
        res.append([name, i, ok, fake.fake_pending(None)])
print(json.dumps(res))
"""

HYBRID = """
klev, ngptot, nproma, batch = 3, 300, 64, 128
p = C.default_params(900.0, 91)
p.ncldtop = 2
from openifs_amd import surrogate as S

L = S._lib()
arm()
h = ctypes.c_void_p()
rc = L.cloudsc_surrogate_create(ctypes.byref(h), klev, 128, 1, batch, ctypes.c_uint64(1))
assert rc == 0, L.cloudsc_last_error()
ngpblks = (ngptot + nproma - 1) // nproma
arr = {n: np.ones(C.blocked_shape(kind, nproma, klev, ngpblks), np.int32 if kind == "1di" else np.float32)
       for n, kind, _ in C.BLOCKED_ARRAYS}
n = ctypes.c_int()

def call():
    return L.cloudsc_hybrid_sp_c(h, ctypes.c_float(0.5), ctypes.c_uint64(1), ctypes.c_float(1e30), ctypes.byref(n),
                                 ctypes.byref(p), ngptot, nproma, klev, ngpblks, ctypes.c_float(900.0),
                                 *C.blocked_args(arr, lambda x: x.ctypes.data), ctypes.c_void_p(0))

res = []
for sel in (0, 40):
    fake.fake_select(sel)
    arm()
    assert call() == 0 and n.value == sel, L.cloudsc_last_error()
    for name in ("hipLaunchKernel", "hipMemcpyAsync", "hipEventRecord", "hipStreamWaitEvent", "hipEventSynchronize"):
        arm()
        call()
        for i in range(1, calls(name) + 1):
            arm(name, i)
            ok = call() == 0
            res.append([name, i, ok, fake.fake_pending(None) if not ok else 0])
print(json.dumps(res))
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fake_device.build(str(tmp_path_factory.mktemp("fake")))


# FP64, 1,300 columns x L91: beyond the page-locked image's 64 MiB, array by array
@pytest.mark.parametrize("prec,klon,flags", [("sp", 16, 0), ("dp", 1300, 0), ("mixed", 16, 16 | 1)])
def test_per_block_entry_waits_for_its_stream(fake, prec, klon, flags):
    res = fake_device.run(fake, BLOCK.format(prec=prec, klon=klon, flags=flags))
    assert any(not ok for _, _, ok, _ in res)
    for name, nth, ok, pending in res:
        assert pending == 0, f"call {nth} of {name} failed, {pending} operations left"
        assert ok or name != "hipHostMalloc"  # without page-locked memory: array by array


def test_hybrid_waits_for_its_side_stream(fake):
    """The caller's stream is the caller's to wait for; the object's own is not."""
    res = fake_device.run(fake, HYBRID)
    assert sum(not ok for _, _, ok, _ in res) > 10
    for name, nth, ok, pending in res:
        assert pending == 0, f"call {nth} of {name} failed, {pending} operations left on the side stream"
