"""Whole sweeps of one mid-size level in a launch (k_rb_tile) against the
half-sweep kernels: sizes around the tiles of 8 and 12 cells, odd extents,
walls and periodic faces, one to five sweeps, from zero and not.  Needs an
MI355X.  Bitwise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [((32, 32, 32), 2), ((16, 16, 16), 1), ((18, 20, 26), 2), ((16, 24, 70), 1),
          ((13, 9, 7), 1), ((1, 2, 3), 1), ((8, 12, 40), 2), ((64, 64, 64), 3)]
BCS = [(0,) * 6, (1,) * 6, (1, 1, 0, 0, 1, 1), (0, 0, 1, 1, 0, 0)]


@pytest.mark.parametrize("kw", [dict(), dict(precision="mixed", coarse="exact")], ids=str)
@pytest.mark.parametrize("n,nlev", SHAPES)
def test_gpu_rb_tile_equals_half_sweeps(gpu_lib, n, nlev, kw):
    from hydro3d_amd import MultigridSolver
    if kw and nlev == 1:
        nlev, n = 2, tuple(2 * q for q in n)
    rng = np.random.default_rng(8)
    f, p0 = rng.standard_normal(n[::-1]), rng.standard_normal(n[::-1])
    f -= f.mean()
    for q, bc in enumerate(BCS):
        for nu in [(2, 2), (1, 2), (3, 1), (0, 5)]:
            ps = []
            for march in (0, 1):
                print(f"case: {n} x {nlev} bc {bc} nu {nu} march {march} {kw}", flush=True)
                with MultigridSolver([dict(n=n, h=(0.02, 0.03, 0.011), bc=bc, nlev=nlev)],
                                     nu1=nu[0], nu2=nu[1], tol=0.0, maxcy=2, **kw) as S:
                    S.set_tail(nlev + 1)
                    for g in range(1, nlev + 1):
                        S.set_march(g, march)
                    S.set_rhs(0, f)
                    S.set_p(0, p0)
                    S.solve()
                    ps.append(S.get_p(0))
            assert np.isfinite(ps[0]).all()
            assert np.array_equal(ps[0], ps[1]), (bc, nu)
