"""Key-switching key loads that fail, on the CPU: the library runs against a
host stand-in for the HIP runtime (cpp/fake_hip.cpp) in which one call fails.
A key that did not arrive whole is never in service; one that was not touched
stays.  Each case runs in a process of its own, where the stand-in is loaded
before the library.
"""

import os
import subprocess
import sys

import pytest

TESTS = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(TESTS)

HEAD = """
import ctypes, sys
import numpy as np
fake = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
import cufhedb_amd as F
L = F.lib()
N0 = 2
p = F.preset(F.PRESET_CFG636)
p.n0 = N0
sk = F.SecretKeys(p, 1)
ctx = F.Context(p)
fail = lambda name, after: fake.fake_fail(name.encode(), after)
loaded = lambda kind: L.fhe_ksk_loaded(ctx.h, kind)
# never read by the stand-in's copies, so never backed by memory
key = {k: np.zeros(F.ksk_shape(p, k), np.uint32) for k in (10, 20, 21)}
def load(kind):
    return L.fhe_load_ksk(ctx.h, kind, F._ptr(key[kind]))
def keygen(kind):
    return L.fhe_keygen_ksk_dev(ctx.h, kind, 7, F._ptr(sk.s1 if kind == 10 else sk.s2),
                                F._ptr(sk.s1 if kind == 21 else sk.s0), None)
def switch(kind):
    return L.fhe_iks_dev(ctx.h, kind, 64, 64, 1, None)
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", os.path.join(TESTS, "cpp", "fake_hip.cpp"), "-o", so],
                   check=True)
    return so


def run(fake, body):
    r = subprocess.run([sys.executable, "-c", HEAD + body, fake], cwd=ROOT, text=True,
                       capture_output=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("kind", [10, 20, 21])
@pytest.mark.parametrize("how", ["load", "keygen"])
def test_failed_first_load_is_not_loaded(fake, kind, how):
    run(fake, f"""
fail("hipMemcpy" if "{how}" == "load" else "hipMemcpyAsync", 0)
assert {how}({kind}) == F.FHE_ERR_DEVICE and not fake.fake_pending()
assert loaded({kind}) == 0 and switch({kind}) == F.FHE_ERR_NOT_LOADED
assert {how}({kind}) == F.FHE_OK and loaded({kind}) == 1 and switch({kind}) == F.FHE_OK
ctx.close()
assert fake.fake_live() == 0
""")


@pytest.mark.parametrize("kind", [10, 20, 21])
@pytest.mark.parametrize("how", ["load", "keygen"])
def test_failed_reload(fake, kind, how):
    """Kinds 10 and 20 arrive where the old key was, so it is gone once the
    first write is under way; kind 21 arrives beside it, so it stays, and so
    does any key when the device generator's inputs do not arrive."""
    run(fake, f"""
assert {how}({kind}) == F.FHE_OK
fail("hipMemcpy" if "{how}" == "load" else "hipMemcpyAsync", 0)
assert {how}({kind}) == F.FHE_ERR_DEVICE and not fake.fake_pending()
stays = {kind} == 21 or "{how}" == "keygen"
assert loaded({kind}) == stays
assert switch({kind}) == (F.FHE_OK if stays else F.FHE_ERR_NOT_LOADED)
ctx.close()
assert fake.fake_live() == 0
""")


@pytest.mark.parametrize("kind", [10, 20])
def test_failed_generation(fake, kind):
    run(fake, f"""
assert keygen({kind}) == F.FHE_OK
fail("hipGetLastError", 0)  # of the kernel that writes the key
assert keygen({kind}) == F.FHE_ERR_DEVICE and not fake.fake_pending()
assert loaded({kind}) == 0 and switch({kind}) == F.FHE_ERR_NOT_LOADED
""")


@pytest.mark.parametrize("kind", [10, 20, 21])
def test_failed_layout_is_not_loaded(fake, kind):
    """The kernel that puts an arrived key into its layout fails, on a first
    load and on a reload."""
    run(fake, f"""
for again in (False, True):
    fail("hipGetLastError", 0)
    assert load({kind}) == F.FHE_ERR_DEVICE and not fake.fake_pending()
    assert loaded({kind}) == 0 and switch({kind}) == F.FHE_ERR_NOT_LOADED
    if not again:
        assert load({kind}) == F.FHE_OK and loaded({kind}) == 1
ctx.close()
assert fake.fake_live() == 0
""")


@pytest.mark.parametrize("kind", [10, 20, 21])
def test_file_that_cannot_be_read_whole(fake, kind, tmp_path):
    """A key file whose upload stops after the first of its chunks."""
    path = str(tmp_path / "ksk.key")
    run(fake, f"""
from cufhedb_amd import keyio as K
member = {{10: K.IKSKLVL10, 20: K.IKSKLVL20, 21: K.IKSKLVL21}}[{kind}]
p.n0 = N0 if {kind} == 21 else 16  # more than one chunk of 64 MB
ctx = F.Context(p)
K.write_key({path!r}, member, p, np.zeros(F.ksk_shape(p, {kind}), np.uint32))
fail("hipMemcpyAsync", 1)
try:
    K.load_key(ctx, {path!r}, member)
    assert False
except F.FheError:
    assert not fake.fake_pending()
assert loaded({kind}) == 0 and switch({kind}) == F.FHE_ERR_NOT_LOADED
ctx.close()
""")


@pytest.mark.parametrize("kind", [10, 20, 21])
def test_reload_without_memory_keeps_the_key(fake, kind):
    """No room for what the reload needs beside the key's own memory."""
    run(fake, f"""
assert load({kind}) == F.FHE_OK
for how in (load, keygen):
    fail("hipMalloc", 0)
    assert how({kind}) == F.FHE_ERR_ALLOC and not fake.fake_pending()
    assert loaded({kind}) == 1 and switch({kind}) == F.FHE_OK
ctx.close()
assert fake.fake_live() == 0
""")


@pytest.mark.parametrize("kind", [10, 21])
def test_refused_during_capture(fake, kind):
    run(fake, f"""
assert load({kind}) == F.FHE_OK and L.fhe_graph_begin(ctx.h) == F.FHE_OK
assert load({kind}) == F.FHE_ERR_ARG and keygen({kind}) == F.FHE_ERR_ARG
assert loaded({kind}) == 1 and switch({kind}) == F.FHE_OK
""")
