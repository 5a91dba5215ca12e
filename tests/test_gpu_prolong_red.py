"""The prolongation that leaves interior red cells to the red half-sweep after
it: every mix of walls and periodic faces, short and long rows, with and
without a sweep to follow, against the oracle.  Needs an MI355X.  Bitwise."""
import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(4, 4, 4), (260, 4, 8), (12, 20, 4)])
@pytest.mark.parametrize("nu", [(2, 1), (1, 2), (2, 0)])
def test_gpu_prolong_red_cells(gpu_lib, n, nu):
    from hydro3d_amd import MultigridSolver
    from oracle import oracle as O
    rng = np.random.default_rng(9)
    f = rng.standard_normal(n[::-1])
    f -= f.mean()
    h = (0.02, 0.03, 0.011)
    for per in itertools.product((0, 1), repeat=3):
        bc = tuple(p for p in per for _ in (0, 1))
        print(f"case: {n} nu {nu} bc {bc}", flush=True)
        with MultigridSolver([dict(n=n, h=h, bc=bc, nlev=2)], nu1=nu[0], nu2=nu[1], tol=0.0,
                             maxcy=3) as S:
            S.set_tail(3)
            S.set_rhs(0, f)
            S.solve()
            p = S.get_p(0)[1:-1, 1:-1, 1:-1]
        po, _ = O.solve(O.Block(n, h, bc, 2), f, 3, 0.0, nu1=nu[0], nu2=nu[1])
        assert np.array_equal(p, po[1:-1, 1:-1, 1:-1]), bc
