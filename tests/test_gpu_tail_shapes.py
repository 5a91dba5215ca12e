"""The V-cycle tail in one workgroup (k_vtail) against the same levels on
their own kernels, at the sizes where a thread's entries, a wavefront or the
workgroup end.  Needs an MI355X.  Bitwise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (cells, levels): both entries of every thread; one entry; entries past the
# registers' (marched); odd rows; odd coarsest cells; a wavefront's edges;
# single cells
SHAPES = [((16, 16, 16), 3), ((16, 16, 8), 3), ((16, 16, 20), 2), ((18, 10, 14), 2),
          ((12, 20, 4), 3), ((6, 22, 2), 2), ((4, 8, 16), 2), ((2, 2, 2), 2), ((26, 2, 34), 2)]
BCS = [(1, 1, 1, 1, 0, 0), (0,) * 6, (1,) * 6, (0, 0, 1, 1, 1, 1)]


@pytest.mark.parametrize("kw", [dict(), dict(coarse="exact"),
                                dict(precision="mixed", coarse="exact"),
                                dict(precision="mixed")], ids=str)
@pytest.mark.parametrize("n,nlev", SHAPES)
def test_gpu_tail_shapes_keep_results(gpu_lib, n, nlev, kw):
    from hydro3d_amd import MultigridSolver
    from hydro3d_amd import _lib as L
    rng = np.random.default_rng(8)
    f = rng.standard_normal(n[::-1])
    f -= f.mean()
    for q, bc in enumerate(BCS):
        nu = [(2, 2), (1, 0), (3, 1), (2, 1)][q]
        ps = {}
        for tail in (nlev + 1, 1, 2):
            print(f"case: tail {tail} of {n} x {nlev} bc {bc} {kw}", flush=True)
            with MultigridSolver([dict(n=n, h=(0.02, 0.03, 0.011), bc=bc, nlev=nlev)], nu1=nu[0],
                                 nu2=nu[1], tol=0.0, maxcy=3, **kw) as S:
                S.set_tail(tail)
                S.set_rhs(0, f)
                try:
                    S.solve()
                    ps[tail] = S.get_p(0)
                    assert np.isfinite(ps[tail]).all()
                except L.H3dError as e:  # one cell between walls: no smoothed coarsest value
                    assert n == (2, 2, 2) and e.status == L.ERR_DIVERGED
                    ps[tail] = e.status
        for tail in (1, 2):
            assert np.array_equal(ps[tail], ps[nlev + 1]), (bc, tail)
