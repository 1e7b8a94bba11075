"""Which kernel a CLOUDSC launch takes, decided on the host by its size, blocks, arithmetic and constants.  No GPU needed."""
import re

import pytest

from tests import fake_device

SCRIPT = """
from openifs_amd import autotune, satadj

L = C.lib()
some = np.ones(8, np.float64)  # nothing runs
ptr = ctypes.c_void_p(some.ctypes.data)
arm()
res = []
for step in {steps}:
    if step[0] == "set":
        autotune.set_launch(*step[1:])
        continue
    kind, prec, ncol, nproma, klev, default = step
    p = C.default_params(900.0, klev)
    if not default:
        p.rcldiff *= 1.5
    fn = ("cloudsc_blocked_" if kind == "plain" else "cloudsc_satadj_cloudsc_blocked_") + prec + "_c"
    n = len(C.BLOCKED_ARRAYS) + (0 if kind == "plain" else {extra})
    arm()
    rc = getattr(L, fn)(ctypes.byref(p), ncol, nproma, klev, -(-ncol // nproma),
                        (ctypes.c_double if prec == "dp" else ctypes.c_float)(900.0), *([ptr] * n), ctypes.c_void_p(0))
    res.append([rc, log()])
print(json.dumps(res))
"""


@pytest.fixture(scope="module")
def routes(tmp_path_factory):
    from openifs_amd import satadj as A

    lib = fake_device.build(str(tmp_path_factory.mktemp("fake")))

    def run(*steps):
        out = []
        for rc, log in fake_device.run(lib, SCRIPT.format(steps=list(steps), extra=len(A.SATADJ_EXTRA_INPUTS) + len(A.SATADJ_TENDENCY_OUT))):
            log = [line for line in log if "clear" not in line]  # the padding columns' PRAINFRAC_TOPRFZ
            assert rc == 0 and len(log) == 1, (rc, log)
            if "pipeline" in log[0]:
                out.append("three waves")
            else:
                block, wpe, kl = re.search(r"Li(\d+)ELb[01]ELb[01]ELb[01]ELi(\d+)ELi(\d+)E", log[0]).groups()
                out.append((int(block), int(wpe), int(kl)))
        return out

    return run


def test_fp64_at_two_waves_per_simd(routes):
    """More waves than SIMDs (65,536 columns; padding counts for nothing), but never with the saturation adjustment."""
    one, two = (256, 0, 0), (256, 2, 0)
    assert routes(("plain", "dp", 65536, 64, 91, True), ("plain", "dp", 65537, 64, 91, True),
                  ("plain", "dp", 65536, 100, 91, True), ("plain", "dp", 65537, 100, 91, True),
                  ("plain", "dp", 65536, 100, 91, False), ("plain", "dp", 70000, 128, 91, False),
                  ("plain", "dp", 20000, 100, 91, False)) == [one, two, one, two, one, two, one]
    assert routes(*[("fused", "dp", 131072, n, 137, d) for n in (64, 100) for d in (True, False)]) == [one] * 4
    assert routes(("plain", "mixed", 200000, 64, 91, False), ("plain", "sp", 200000, 100, 91, True)) == [one] * 2


def test_a_launch_that_is_set_is_used_at_every_size(routes):
    """cloudsc_tune_set_launch holds for small launches too, and waves 0 is the compiler's choice beyond 65,536 FP64
    columns; a recorded launch (autotune.apply, at the library's loading) leaves both choices to the library."""
    small, big = ("plain", "sp", 2000, 64, 91, True), ("plain", "sp", 100000, 64, 91, True)
    dp = ("plain", "dp", 100000, 128, 137, True)
    assert routes(small, big, dp, ("set", "sp", 91, 128, 0, 0), small, big, ("set", "sp", 91, 0), small, big,
                  ("set", "dp", 137, 256, 0, 0), dp, ("plain", "dp", 100000, 100, 137, True), ("set", "dp", 137, 128, 2, 1),
                  dp, ("plain", "dp", 500, 128, 137, True)) == [
        "three waves", (256, 4, 91), (256, 2, 0), (128, 0, 0), (128, 0, 0), "three waves", (256, 0, 0), (256, 0, 0),
        (256, 0, 0), (128, 2, 137), (128, 2, 137)]


@pytest.mark.gpu
def test_timing_launches_leaves_the_settings_as_they_were():
    pytest.importorskip("torch")
    from openifs_amd import autotune as A
    from openifs_amd import cloudsc as C

    scope = lambda: C.lib().cloudsc_tune_get_scope(A.VARIANTS["sp"], 91)  # noqa: E731
    was = scope(), A.get_launch("sp", 91)
    try:
        for prepare, want in ((lambda: A.set_launch("sp", 91, 0), 0), (lambda: A.set_recorded("sp", 91, 128, 4, 1), 1),
                              (lambda: A.set_launch("sp", 91, 64), 2)):
            prepare()
            before = A.get_launch("sp", 91)
            A.time_launches("sp", 91, 2048, 64, [(256, 0, 0), (128, 4, 1)], reps=1)
            assert scope() == want and A.get_launch("sp", 91) == before
    finally:
        (A.set_recorded if was[0] == 1 else A.set_launch)("sp", 91, *(was[1] if was[0] else (0,)))


def test_three_wave_launches_by_size(routes):
    """One round of work-groups: 49,152 columns in FP32, 16,384 in FP64; 45,056 in blocks that are no multiple of 64."""
    steps = []
    for prec in ("sp", "mixed"):
        for nproma, line in ((64, 49152), (32, 45056)):
            for default in (True, False):
                for kind in ("plain", "fused"):
                    steps += [(kind, prec, line, nproma, 91, default), (kind, prec, line + nproma, nproma, 91, default)]
    for nproma in (64, 32):
        steps += [("plain", "dp", 16384, nproma, 91, True), ("plain", "dp", 16384 + nproma, nproma, 91, True)]
    assert [r == "three waves" for r in routes(*steps)] == [True, False] * (len(steps) // 2)
