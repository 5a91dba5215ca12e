"""The library's host side on a HIP runtime without a device
(tests/fake_hip.c): what it allocates, and how long the sources of its
asynchronous uploads live."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes, sys
sys.path.insert(0, {root!r})
fake = ctypes.CDLL({fake!r}, mode=ctypes.RTLD_GLOBAL)
from hydro3d_amd import _lib as L
lib = L.load()
def handle(blocks, **kw):
    from hydro3d_amd import MultigridSolver
    return MultigridSolver([dict(n=n, h=(0.1,) * 3, bc=(0,) * 6, nlev=q) for n, q in blocks], **kw)
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", so, os.path.join(HERE, "fake_hip.c")],
                   check=True)

    def run(code):
        r = subprocess.run([sys.executable, "-c", PRELUDE.format(root=ROOT, fake=so) + code],
                           capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr
        return r.stdout.split()
    return run


@pytest.mark.parametrize("blocks", [1, 3])
def test_uploads_outlive_their_copy(fake, blocks):
    """Every host-to-device copy's source holds its data until the stream is
    waited for, over the velocity loop's begin (its tables) and steps."""
    out = fake(f"""
S = handle([((8, 8, 8), 2)] * {blocks})
mem = ctypes.create_string_buffer(16 * 9 * 8 * 8 * 8)
at = lambda q: ctypes.addressof(mem) + q * 9 * 8 * 8 * 8
arr = lambda q: (ctypes.c_void_p * {blocks})(*[at(q)] * {blocks})
rm = ctypes.c_double(0.0)
before = fake.fake_late_sources()
for _ in range(2):
    L.check(lib.h3dmg_velocity_begin(S.h, arr(0), arr(1), arr(2), arr(3), arr(4), arr(5), 1.0,
                                     ctypes.byref(rm)))
    L.check(lib.h3dmg_velocity_step(S.h, ctypes.byref(rm)))
print(before, fake.fake_late_sources())
""")
    assert out == ["0", "0"]
