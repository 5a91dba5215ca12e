"""A block's arrays in and out of the handle (k_copy_fine, k_set_rhs) and the
stopping rule over many blocks (k_finalize_decide), at the sizes where a row's
lanes, a tile or the workgroup end.  Needs an MI355X."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
SHAPES = [(1, 1, 1), (2, 1, 3), (3, 5, 7), (33, 9, 2), (130, 3, 2), (520, 2, 3), (64, 8, 17)]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_gpu_fine_arrays_round_trip(gpu_lib, precision):
    import torch
    from hydro3d_amd import MultigridSolver
    from hydro3d_amd import _lib as L
    rng = np.random.default_rng(2)
    kw = dict(precision="mixed", coarse="exact") if precision == "mixed" else {}
    if precision == "mixed":  # two levels: the fine one in float
        shapes = [tuple(2 * q for q in n) for n in SHAPES]
    else:
        shapes = SHAPES
    specs = [dict(n=n, h=(0.1,) * 3, bc=(1, 1, 0, 0, 0, 0), nlev=1 if precision == "fp64" else 2)
             for n in shapes]
    with MultigridSolver(specs, **kw) as S:
        for b, n in enumerate(shapes):
            print(f"case: {precision} {n}", flush=True)
            f = rng.standard_normal(n[::-1])
            p = torch.from_numpy(rng.standard_normal(n[::-1])).cuda()
            # a view one element into a buffer: 8-byte alignment only
            buf = torch.empty(f.size + 1, dtype=torch.float64, device="cuda")
            buf[1:] = torch.from_numpy(f).cuda().flatten()
            S.set_rhs(b, buf[1:].view(n[::-1]))
            S.set_p(b, p)
            out = torch.empty(f.size + 1, dtype=torch.float64, device="cuda")[1:].view(n[::-1])
            assert torch.equal(S.get_p(b, out=out), p)
            rhs = S.dbg_get(b, 1, L.ARR_RHS, torch.empty(n[::-1], dtype=torch.float64,
                                                         device="cuda")).cpu().numpy()
            assert np.array_equal(rhs, f if precision == "fp64" else f.astype(np.float32))


@pytest.mark.parametrize("nb", [1, 2, 65, 1100])
@pytest.mark.parametrize("criterion", ["rel_l2", "ref_rmax"])
def test_gpu_stopping_rule_over_blocks(gpu_lib, nb, criterion):
    """Blocks that stop at different cycles: the queued loop (the rule on the
    device) against the host's loop."""
    from hydro3d_amd import MultigridSolver
    print(f"case: {nb} blocks {criterion}", flush=True)
    rng = np.random.default_rng(nb)
    specs = [dict(n=(4, 4, 2 + 2 * (b % 3)), h=(0.1, 0.1, 0.1), bc=(1, 1, 1, 1, 0, 0), nlev=1)
             for b in range(nb)]
    fs = [rng.standard_normal(s["n"][::-1]) * 10.0 ** (b % 5) for b, s in enumerate(specs)]
    res = []
    for graph in (True, False):
        with MultigridSolver(specs, tol=1e-5, maxcy=60, criterion=criterion, use_graph=graph) as S:
            for b, f in enumerate(fs):
                S.set_rhs(b, f - f.mean())
            st, cyc, hist = S.solve()
            res.append((st, cyc, hist, S.block_stats(), [S.get_p(b) for b in range(nb)]))
    a, c = res
    assert a[0] == c[0] and a[1] == c[1] and np.array_equal(a[2], c[2])
    assert np.array_equal(a[3][0], c[3][0]) and np.array_equal(a[3][1], c[3][1])
    assert all(np.array_equal(x, y) for x, y in zip(a[4], c[4]))
