"""The exact coarsest solve on its routes -- in the V-cycle tail (LDS of one
workgroup), in three launches over planes and columns, one launch per
transform -- at the sizes where planes, columns, tiles of outputs or the LDS
end.  Needs an MI355X.  Bitwise between the routes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BCS = [(1, 1, 1, 1, 0, 0), (0,) * 6, (1,) * 6, (0, 0, 1, 1, 1, 1)]
# two-level blocks: single cells, one plane, ragged columns, planes around
# EXACT_SMALL (512 cells) and of 64 x 64, one column
SHAPES = [(2, 2, 2), (8, 8, 8), (34, 2, 6), (48, 40, 2), (52, 28, 20), (44, 48, 6), (2, 2, 64),
          (128, 128, 4)]
UNFIT = (2, 2, 300)  # coarse 150^2 table over the LDS: one launch per transform


def _solve(specs, fs, tail=None, cycles=3):
    from hydro3d_amd import MultigridSolver
    with MultigridSolver(specs, tol=0.0, maxcy=cycles, coarse="exact") as S:
        if tail is not None:
            S.set_tail(tail)
        for b, f in enumerate(fs):
            S.set_rhs(b, f)
        S.solve()
        return [S.get_p(b) for b in range(len(specs))]


def _rhs(n, seed=3):
    f = np.random.default_rng(seed).standard_normal(n[::-1])
    return f - f.mean()


@pytest.mark.parametrize("n", SHAPES)
@pytest.mark.parametrize("bc", BCS)
def test_gpu_exact_coarse_routes_agree(gpu_lib, n, bc):
    from hydro3d_amd import _lib as L
    print(f"case: exact coarse {n} bc {bc}", flush=True)
    spec, f = dict(n=n, h=(0.02, 0.03, 0.011), bc=bc, nlev=2), _rhs(n)
    split = _solve([spec], [f], tail=3)[0]
    assert np.isfinite(split).all()
    other = dict(n=UNFIT, h=(0.02,) * 3, bc=bc, nlev=2)
    both = _solve([spec, other], [f, _rhs(UNFIT)], tail=3)
    assert np.array_equal(both[0], split)  # k_exact_pass, for both
    try:
        tail = _solve([spec], [f], tail=2)[0]
    except L.H3dError as e:  # does not fit in LDS
        assert e.status == L.ERR_ARG and np.prod(n) > 8 * 3000
        return
    assert np.array_equal(tail, split)


@pytest.mark.parametrize("n", [(64, 64, 32), UNFIT])
def test_gpu_exact_coarse_solves(gpu_lib, n):
    """Two-grid cycles converge at a rate well under 0.25 a cycle only with
    the coarse level solved: 12 cycles, 0.25^12 = 6e-8."""
    import torch
    from hydro3d_amd import MultigridSolver
    f = _rhs(n)
    with MultigridSolver([dict(n=n, h=(0.05,) * 3, bc=(0,) * 6, nlev=2)], tol=0.0, maxcy=12,
                         coarse="exact") as S:
        S.set_rhs(0, f)
        S.solve()
        p = torch.from_numpy(S.get_p(0)[1:-1, 1:-1, 1:-1].copy())
    q = torch.nn.functional.pad(p[None, None], (1,) * 6, mode="replicate")[0, 0]
    lap = (q[2:, 1:-1, 1:-1] + q[:-2, 1:-1, 1:-1] + q[1:-1, 2:, 1:-1] + q[1:-1, :-2, 1:-1]
           + q[1:-1, 1:-1, 2:] + q[1:-1, 1:-1, :-2] - 6 * p) / 0.05**2
    r = (torch.from_numpy(f) - lap).abs().max().item()
    assert r < 0.25**12 * np.abs(f).max()
