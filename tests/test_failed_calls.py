"""What a call that runs out of memory leaves behind, on a HIP runtime without a
device (tests/emu/hipfake.c, preloaded in a process of its own): every allocation,
stream and event in turn refused, the next calls made on what is left."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

HEAD = """
import ctypes, sys
import numpy as np
fake = ctypes.CDLL(sys.argv[1])
fake.fake_log.restype = ctypes.c_char_p
fake.fake_armed.restype = fake.fake_live.restype = ctypes.c_long
fake.fake_fail.argtypes = [ctypes.c_long]
import bluecrunch_amd as bc
L = bc.lib()
def operands():
    # both magnitudes end at 0: the words decide the order
    a = bc.DeviceBigfloat((np.arange(1, 3001, dtype=np.uint32), -3000, 1))
    b = bc.DeviceBigfloat((np.arange(2, 3002, dtype=np.uint32), -3000, 1))
    t = bc.DeviceBigfloat()
    return a, b, t
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    if not shutil.which("gcc"):
        pytest.skip("gcc not available")
    if not os.path.exists(os.path.join(ROOT, "bluecrunch_amd", "libbluecrunch.so")):
        pytest.fail("libbluecrunch.so is not built")
    so = tmp_path_factory.mktemp("fake") / "hipfake.so"
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", os.path.join(HERE, "emu", "hipfake.c"), "-o", str(so)], check=True)
    return str(so)


def _run(fake, body):
    env = dict(os.environ, LD_PRELOAD=fake, PYTHONPATH=ROOT)
    r = subprocess.run([sys.executable, "-c", HEAD + body, fake], env=env, cwd=ROOT, capture_output=True, text=True)
    assert r.returncode == 0, (r.returncode, r.stdout[-500:], r.stderr[-1500:])
    return r.stdout


def test_failed_initialisation(fake):
    out = _run(fake, """
failed = 0
for nth in range(1, 400):
    fake.fake_fail(nth)
    rc = L.bcg_init(0)
    reached = fake.fake_armed() == 0
    fake.fake_fail(0)
    assert rc == 0 or reached, nth
    failed += rc != 0
    # whatever is left: a product of several passes and a difference
    a = bc.DeviceWords.from_host(np.arange(1, 20001, dtype=np.uint32))
    c = bc.DeviceWords(40000)
    bc.mul_dev(c.ptr, 40000, a.ptr, 20000, a.ptr, 20000)
    x, y, t = operands()
    bc.bf_op("sub", t, x, y, 0)
    del a, c, x, y, t
    bc.check(L.bcg_shutdown(), "shutdown")
    assert fake.fake_live() == 0, (nth, fake.fake_live())
    if not reached:
        break
assert failed >= 10 and not reached
print("done", failed)
""")
    assert out.startswith("done")


def test_failed_difference_leaves_no_order_behind(fake):
    # the search for the word that decides the order leaves it to the difference behind
    # it, which clears it: the search must not run if the difference cannot
    out = _run(fake, """
failed = 0
for nth in range(1, 50):
    bc.check(L.bcg_init(0), "init")
    x, y, t = operands()
    fake.fake_log_clear()
    fake.fake_fail(nth)
    rc = L.bcg_bf_sub(ctypes.byref(t.bf), ctypes.byref(x.bf), ctypes.byref(y.bf), 0)
    reached = fake.fake_armed() == 0
    fake.fake_fail(0)
    log = fake.fake_log().decode()
    assert log.count("k_ucmp_diff") == log.count("k_addsub"), (nth, rc, log)
    del x, y, t
    bc.check(L.bcg_shutdown(), "shutdown")
    if not reached:
        break
    failed += rc != 0
assert failed >= 2 and rc == 0 and "k_ucmp_diff" in log
print("done", failed)
""")
    assert out.startswith("done")
