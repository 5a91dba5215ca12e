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


def test_line_workspace_is_optional(fake):
    """A line-TDMA block's region is what its levels, p, f and tables take
    (the line passes' workspace is not in it), and a handle is made where
    memory suffices for everything but that workspace."""
    out = fake("""
from hydro3d_amd.solver import block_bytes
al = lambda x: (x + 255) // 256 * 256
def expect(n, nlev):
    tot = 0
    for g in range(nlev):
        ni, nj, nk = (x >> g for x in n)
        tot += 6 * al((((ni + 1) // 2 + 1) & ~1) * nj * nk * 8) + al(32 * (ni + nj + nk) * 8)
    return tot + 4 * al((((n[0] + 1) // 2 + 1) & ~1) * n[1] * n[2] * 8)
ok = True
for n, nlev in (((64, 64, 64), 5), ((32, 32, 32), 1), ((48, 16, 130), 2)):
    spec = dict(n=n, h=(0.1,) * 3, bc=(0,) * 6, nlev=nlev)
    ok = ok and block_bytes(spec, smoother="tdma") == expect(n, nlev)
fake.fake_set_room.argtypes = [ctypes.c_size_t]
fake.fake_room.restype = ctypes.c_size_t
fake.fake_set_room(1 << 30)
blocks = [((32, 32, 32), 3), ((16, 24, 20), 2)]
S = handle(blocks, smoother="tdma")
used = (1 << 30) - fake.fake_room()
assert S.device_bytes == used, (S.device_bytes, used)
S.close()
fake.fake_set_room(used - 1)  # either allocation fits, not both
S = handle(blocks, smoother="tdma")
small = S.device_bytes
assert small == used - 1 - fake.fake_room()
S.close()
fake.fake_set_room(small)
handle(blocks, smoother="tdma").close()
fake.fake_set_room(small - 1)
try:
    handle(blocks, smoother="tdma")
except L.H3dError as e:
    print(ok, e.status == L.ERR_NOMEM)
""")
    assert out == ["True", "True"]


@pytest.mark.parametrize("kw,before", [(dict(precision="mixed", coarse="exact"), 564736),
                                       (dict(), 550656), (dict(smoother="tdma"), 488960)],
                         ids=["mixed", "fp64", "tdma"])
def test_pooled_tables_have_not_grown(fake, kw, before):
    """The pool piece of a pooled handle's tables, for one large block and
    many small ones: no more than before the projection had partials and
    tables for every block (a pooled handle has no velocity loop)."""
    out = fake(f"""
from hydro3d_amd import MultigridSolver
from hydro3d_amd.solver import DevicePool, block_bytes
kw = {kw!r}
specs = [dict(n=n, h=(0.1,) * 3, bc=(0,) * 6, nlev=q)
         for n, q in [((256, 256, 32), 4)] + [((16, 16, 16), 3)] * 20]
P = DevicePool(1 << 28, 64)
offs = [P.alloc(block_bytes(s, **kw)) for s in specs]
S = MultigridSolver(specs, pool=P, offsets=offs, **kw)
print(S.device_bytes)
""")
    assert int(out[0]) <= before
