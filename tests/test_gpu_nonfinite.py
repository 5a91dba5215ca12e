"""Infinities and NaN through the V-cycle: a wall's coefficient is zero, but
its product with the ghost (the cell's own value before the sweep) is NaN
where that value is not finite, in the reference and in the oracle.  Every
route of a level (the tail in LDS, pairs of sweeps, half-sweeps) gives the
oracle's infinities and NaN at the oracle's cells.  Needs an MI355X.
Bitwise, NaN equal to NaN."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

H = (0.02, 0.03, 0.011)
BCS = [(0,) * 6, (1, 1, 0, 0, 0, 0), (0, 0, 1, 1, 1, 1)]


def _pp(n, nlev, bc, f, nu, tail, march, **kw):
    from hydro3d_amd import MultigridSolver
    with MultigridSolver([dict(n=n, h=H, bc=bc, nlev=nlev)], nu1=nu[0], nu2=nu[1], **kw) as S:
        S.set_tail(tail)
        for g in range(1, nlev + 1):
            S.set_march(g, march)
        S.set_rhs(0, f)
        S.vcycle()
        return S.get_pp(0)[1:-1, 1:-1, 1:-1]


def _rhs(n, seed, value, at):
    f = np.random.default_rng(seed).standard_normal(n[::-1])
    f[tuple({"low": 0, "high": d - 1, "mid": d // 3}[at] for d in f.shape)] = value
    return f


@pytest.mark.parametrize("value", [np.inf, np.nan, 1e300], ids=str)
@pytest.mark.parametrize("n,nlev,routes", [
    ((16, 16, 16), 3, "tail"), ((20, 8, 12), 3, "tail"), ((16, 16, 16), 5, "tail"),
    ((32, 24, 16), 1, "pairs"), ((16, 18, 20), 2, "pairs"), ((16, 36, 52), 2, "half"), ((20, 24, 16), 3, "half"),
    ((16, 16, 16), 5, "pairs"), ((16, 16, 16), 5, "half"),
])
def test_gpu_nonfinite_values_equal_oracle(gpu_lib, n, nlev, routes, value):
    from oracle import oracle as O
    for bc in BCS:
        for at in ("low", "mid", "high"):
            f = _rhs(n, 16, value, at)
            for nu in ((2, 2), (1, 0), (0, 1), (2, 1), (0, 3), (4, 0)):
                print(f"case: {n} x {nlev} bc {bc} {value} at {at} nu {nu} {routes}", flush=True)
                want = O.vcycle(O.Block(n, H, bc, nlev), f, *nu)[1:-1, 1:-1, 1:-1]
                tail = 1 if routes == "tail" else nlev + 1
                got = _pp(n, nlev, bc, f, nu, tail, 1 if routes == "half" else 0)
                assert np.array_equal(got, want, equal_nan=True), (bc, at, nu)


@pytest.mark.parametrize("value", [np.inf, np.nan, 1e38], ids=str)
@pytest.mark.parametrize("n,nlev", [((16, 16, 16), 3), ((18, 20, 28), 2)])
def test_gpu_nonfinite_values_mixed_routes_agree(gpu_lib, n, nlev, value):
    for bc in BCS:
        for at in ("low", "mid", "high"):
            f = _rhs(n, 17, value, at)
            for nu in ((2, 2), (0, 1), (2, 1), (0, 3), (4, 0)):
                print(f"case: mixed {n} bc {bc} {value} at {at} nu {nu}", flush=True)
                ref = _pp(n, nlev, bc, f, nu, nlev + 1, 1, precision="mixed")
                for tail, march in ((1, 0), (nlev + 1, 0)):
                    if tail == 1 and max(n) > 16:
                        continue
                    got = _pp(n, nlev, bc, f, nu, tail, march, precision="mixed")
                    assert np.array_equal(got, ref, equal_nan=True), (bc, at, nu, tail, march)
