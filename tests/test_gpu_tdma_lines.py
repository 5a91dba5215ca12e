"""The line-TDMA passes in two launches (k_tdma_pre, k_tdma_lines) against
the oracle's sequential sweeps, at the sizes where a wavefront's lanes, the
register-held line or the diagonals end.  Needs an MI355X.  Bitwise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# full lanes and lines; odd axes; single cells; lines a little over a kernel's
# 16 or 32 positions; more steps than lanes; an axis over 64 (the pipelined
# whole-sweep kernel)
SHAPES = [(64, 64, 64), (17, 33, 9), (1, 5, 64), (64, 1, 2), (16, 16, 16), (2, 17, 31),
          (8, 3, 100), (72, 16, 10)]
BCS = [(1, 1, 1, 1, 0, 0), (0,) * 6, (1,) * 6, (0, 0, 1, 1, 1, 1)]


@pytest.mark.parametrize("n", SHAPES)
@pytest.mark.parametrize("bc", BCS)
def test_gpu_tdma_lines_sweeps_equal_oracle(gpu_lib, n, bc):
    from hydro3d_amd import MultigridSolver
    from oracle import oracle as O
    print(f"case: TDMA {n} bc {bc}", flush=True)
    h = (0.02, 0.03, 0.011)
    rng = np.random.default_rng(5)
    f = rng.standard_normal(n[::-1])
    f -= f.mean()
    with MultigridSolver([dict(n=n, h=h, bc=bc, nlev=1)], nu1=2, nu2=1, tol=0.0, maxcy=2,
                         smoother="tdma") as S:
        S.set_rhs(0, f)
        S.solve()
        p = S.get_p(0)[1:-1, 1:-1, 1:-1]
    po, _ = O.solve(O.Block(n, h, bc, 1), f, 2, 0.0, nu1=2, nu2=1, scheme=O.SCHEME_TDMA)
    assert np.array_equal(p, po[1:-1, 1:-1, 1:-1])


def test_gpu_tdma_lines_many_blocks(gpu_lib):
    """Blocks of different sizes share the launches (the longest line of each
    pass sets the kernel)."""
    from hydro3d_amd import MultigridSolver
    from oracle import oracle as O
    rng = np.random.default_rng(6)
    specs = [dict(n=n, h=(0.02,) * 3, bc=BCS[q % 4], nlev=2)
             for q, n in enumerate([(16, 16, 32), (64, 8, 4), (6, 40, 10), (32, 32, 32)])]
    fs = []
    for s in specs:
        f = rng.standard_normal(s["n"][::-1])
        fs.append(f - f.mean())
    with MultigridSolver(specs, tol=0.0, maxcy=2, smoother="tdma") as S:
        for b, f in enumerate(fs):
            S.set_rhs(b, f)
        S.solve()
        ps = [S.get_p(b)[1:-1, 1:-1, 1:-1] for b in range(len(specs))]
    for s, f, p in zip(specs, fs, ps):
        po, _ = O.solve(O.Block(s["n"], s["h"], s["bc"], 2), f, 2, 0.0, scheme=O.SCHEME_TDMA)
        assert np.array_equal(p, po[1:-1, 1:-1, 1:-1])
