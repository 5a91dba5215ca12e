"""The device's stopping rule (one wavefront, a lane per block) against the
host's loop at the block counts where its reduction changes rounds; the block
that decides is the last, the first or one in between.  Needs an MI355X."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("criterion", ["rel_l2", "ref_rmax"])
@pytest.mark.parametrize("nb", [1, 2, 3, 5, 8, 9, 32, 33, 64, 65, 130])
def test_gpu_stopping_rule_of_many_blocks(gpu_lib, nb, criterion):
    from hydro3d_amd import MultigridSolver
    rng = np.random.default_rng(15)
    spec = dict(n=(8, 8, 8), h=(0.1,) * 3, bc=(0,) * 6, nlev=2)
    f = [rng.standard_normal((8, 8, 8)) for _ in range(nb)]
    f = [x - x.mean() for x in f]
    for worst in sorted({0, nb // 2, nb - 1}):
        print(f"case: {nb} blocks, worst {worst}, {criterion}", flush=True)
        out = []
        for graph in (True, False):
            with MultigridSolver([spec] * nb, criterion=criterion, tol=1e-5, dt=1.0,
                                 use_graph=graph) as S:
                for b in range(nb):
                    S.set_rhs(b, f[b] * (50.0 if b == worst else 1.0))
                st, nc, hist = S.solve()
                out.append((st, nc, hist.tolist(), S.block_stats(),
                            [S.get_p(b) for b in (0, worst, nb - 1)]))
        assert out[0][:4] == out[1][:4]
        assert all(np.array_equal(x, y) for x, y in zip(out[0][4], out[1][4]))
