"""The correction read back after a solve (h3dmg_get_pp): the residual that
ends a cycle writes the next one's red half-sweep into a level-1 buffer, which
must not be the one the correction lies in, whether level 1 takes its sweeps
in pairs (k_rb_tile, one buffer step a pair) or one by one, or runs in the
tail.  Needs an MI355X.  Bitwise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(n, nlev, f, p0, nu, march, tail):
    from hydro3d_amd import MultigridSolver
    with MultigridSolver([dict(n=n, h=(0.02, 0.03, 0.011), bc=(1, 1, 0, 0, 1, 1), nlev=nlev)],
                         nu1=nu[0], nu2=nu[1], tol=0.0, maxcy=3) as S:
        S.set_tail(tail)
        for g in range(1, nlev + 1):
            S.set_march(g, march)
        S.set_rhs(0, f)
        S.set_p(0, p0)
        S.solve()
        return S.get_p(0), S.get_pp(0)


@pytest.mark.parametrize("nu", [(1, 1), (1, 2), (1, 3), (1, 4), (1, 5), (2, 1), (2, 2), (3, 1)],
                         ids=lambda n: f"V{n[0]}{n[1]}")
@pytest.mark.parametrize("n,nlev", [((32, 32, 32), 2), ((16, 18, 20), 1), ((16, 16, 16), 2)])
def test_gpu_pp_after_solve(gpu_lib, n, nlev, nu):
    rng = np.random.default_rng(12)
    f, p0 = rng.standard_normal(n[::-1]), rng.standard_normal(n[::-1])
    f -= f.mean()
    ref = _run(n, nlev, f, p0, nu, 1, nlev + 1)
    for tail in (nlev + 1, 1):
        if tail == 1 and max(n) > 20:
            continue  # beyond a workgroup's LDS
        print(f"case: {n} x {nlev} nu {nu} tail {tail}", flush=True)
        out = _run(n, nlev, f, p0, nu, 0, tail)
        assert np.array_equal(out[0], ref[0])
        assert np.array_equal(out[1], ref[1])
    # each cycle is p = p + pp: the last correction, not what came after it
    assert np.isfinite(ref[1]).all() and np.abs(ref[1]).max() > 0
