"""Blocks of one level beside deeper ones in one handle, where one group's
level 1 may take its sweeps in pairs (k_rb_tile) and the other's does not:
every block's pressure against the oracle's solve of it alone, and its
correction against the half-sweep launches.  Needs an MI355X.  Bitwise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

H = (0.02, 0.03, 0.011)
# (cells, levels) of a handle's blocks: a one-level block that takes pairs beside a deeper level 1
# too large for them; two one-level blocks beside a deeper one that takes
# pairs; both of a size that takes pairs
HANDLES = [[((32, 32, 32), 1), ((64, 64, 64), 4)],
           [((16, 12, 20), 1), ((32, 32, 32), 3), ((24, 16, 18), 1)],
           [((13, 9, 7), 1), ((32, 24, 16), 2)]]
NUS = [(2, 1), (1, 2), (3, 1), (2, 2), (1, 1), (1, 3), (0, 3), (2, 0)]


def _run(blocks, bc, fs, p0, nu, march):
    from hydro3d_amd import MultigridSolver
    nlev = max(q for _, q in blocks)
    with MultigridSolver([dict(n=n, h=H, bc=bc, nlev=q) for n, q in blocks], nu1=nu[0],
                         nu2=nu[1], tol=0.0, maxcy=2) as S:
        S.set_tail(nlev + 1)
        for g in range(1, nlev + 1):
            S.set_march(g, march)
        for b in range(len(blocks)):
            S.set_rhs(b, fs[b])
            S.set_p(b, p0[b])
        S.solve()
        return ([S.get_p(b)[1:-1, 1:-1, 1:-1] for b in range(len(blocks))],
                [S.get_pp(b) for b in range(len(blocks))])


@pytest.mark.parametrize("nu", NUS, ids=lambda n: f"V{n[0]}{n[1]}")
@pytest.mark.parametrize("flip", [False, True])
@pytest.mark.parametrize("which", range(len(HANDLES)))
def test_gpu_one_level_blocks_beside_deeper_ones(gpu_lib, which, flip, nu):
    from oracle import oracle as O
    blocks = HANDLES[which][::-1] if flip else HANDLES[which]
    bc = (1, 1, 0, 0, 1, 1) if which == 1 else (0,) * 6
    print(f"case: {blocks} bc {bc} nu {nu}", flush=True)
    rng = np.random.default_rng(11)
    fs = [rng.standard_normal(n[::-1]) for n, _ in blocks]
    fs = [f - f.mean() for f in fs]
    p0 = [rng.standard_normal(n[::-1]) for n, _ in blocks]
    p, pp = _run(blocks, bc, fs, p0, nu, 0)
    ref_p, ref_pp = _run(blocks, bc, fs, p0, nu, 1)
    for b, (n, nlev) in enumerate(blocks):
        start = np.zeros(tuple(q + 2 for q in n[::-1]))
        start[1:-1, 1:-1, 1:-1] = p0[b]
        po, _ = O.solve(O.Block(n, H, bc, nlev), fs[b], 2, 0.0, nu1=nu[0], nu2=nu[1], p0=start)
        po = po[1:-1, 1:-1, 1:-1]
        assert np.array_equal(ref_p[b], po), b
        assert np.array_equal(p[b], po), b
        assert np.array_equal(pp[b], ref_pp[b]), b
