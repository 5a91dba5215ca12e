"""A velocity loop's projection beside a stepped solve that runs: it replaces
f, and the running block's residual, from which its next V-cycle starts, stays
in the level-1 right-hand side.  Needs an MI355X.  Bitwise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_gpu_projection_keeps_running_residuals(gpu_lib, precision, use_graph):
    import torch
    from hydro3d_amd import MultigridSolver
    n = (16, 24, 32)
    specs = [dict(n=n, h=(0.02, 0.03, 0.011), bc=(1, 1, 0, 0, 1, 1), nlev=3)] * 2
    rng = np.random.default_rng(18)
    vel = [[torch.from_numpy(rng.standard_normal((32 + (a == 2), 24 + (a == 1), 16 + (a == 0)))).cuda()
            for _ in range(2)] for a in range(3)]
    fs = [rng.standard_normal(n[::-1]) for _ in range(2)]
    fs = [f - f.mean() for f in fs]
    p0 = [rng.standard_normal(n[::-1]) for _ in range(2)]
    out = []
    for project in (False, True):
        print(f"case: {precision} graph {use_graph} project {project}", flush=True)
        with MultigridSolver(specs, precision=precision, tol=1e-12, use_graph=use_graph) as S:
            if project:  # a captured step of a loop before the solve
                S.velocity_begin(*vel)
                S.velocity_step()
            for b in range(2):
                S.set_rhs(b, fs[b])
                S.set_p(b, p0[b])
            S.solve_begin([0, 1])
            if project:
                S.velocity_begin(*vel)
            S.solve_step()
            out.append([S.get_p(b) for b in range(2)])
            if project:  # and the loop's own step is what it is without a solve
                p = [S.result_p(b) for b in range(2)]
                S.velocity_begin(*vel)
                S.velocity_step()
                got = [S.get_p(b) for b in range(2)]
    for x, y in zip(*out):
        assert np.array_equal(x, y)
    with MultigridSolver(specs, precision=precision) as R:
        for b in range(2):
            R.set_p(b, p[b])
        R.velocity_begin(*vel)
        R.velocity_step()
        for b in range(2):
            assert np.array_equal(R.get_p(b), got[b])
