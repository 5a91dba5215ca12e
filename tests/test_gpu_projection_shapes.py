"""calvel + calmas in one launch (k_project) against the per-axis kernels, at
the sizes where its tiles have edges.  Needs an MI355X.

The per-axis kernels serve calls whose outputs overlap their inputs (the
projection in place), so the same projection in place is the reference:
every value is the same expression in both, and the bar is bitwise.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# rows of one entry, odd rows, one lane past a wavefront's 64 entries, single
# rows and planes, more planes than a tile is deep
SHAPES = [(1, 1, 1), (2, 3, 1), (5, 1, 7), (33, 5, 4), (128, 4, 3), (130, 9, 11), (257, 3, 2),
          (64, 64, 40)]


def _faces(n, seed):
    import torch
    ni, nj, nk = n
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(s, generator=g, device="cuda", dtype=torch.float64)
            for s in ((nk, nj, ni + 1), (nk, nj + 1, ni), (nk + 1, nj, ni))]


def _p(n, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(tuple(reversed(n)), generator=g, device="cuda", dtype=torch.float64)


def _project(S, us, outs, su):
    """h3dmg_project_device with the given output arrays; returns rmax."""
    from hydro3d_amd import _lib as L
    import torch
    torch.cuda.synchronize()
    r = ctypes.c_double(0.0)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    L.check(S.lib.h3dmg_project_device(S.h, 0, *[ptr(t) for t in us], *[ptr(t) for t in outs],
                                       ptr(su), 0.75, ctypes.byref(r)))
    return r.value


@pytest.mark.parametrize("n", SHAPES)
@pytest.mark.parametrize("bc", [(0,) * 6, (1,) * 6, (1, 1, 0, 0, 1, 1)])
@pytest.mark.parametrize("density", [False, True])
def test_gpu_projection_equals_per_axis_kernels(gpu_lib, n, bc, density):
    import torch
    from hydro3d_amd import MultigridSolver
    print(f"case: projection {n} bc {bc} density {density}", flush=True)
    us = _faces(n, 3)
    with MultigridSolver([dict(n=n, h=(0.3, 0.7, 0.11), bc=bc, nlev=1)], dt=2e-3) as S:
        if density:
            S.set_density(0, _p(n, 5).abs() + 0.1)
        S.set_p(0, _p(n, 4))
        outs = [torch.empty_like(t) for t in us]
        su = torch.empty(tuple(reversed(n)), device="cuda", dtype=torch.float64)
        rmax = _project(S, us, outs, su)
        ref = [t.clone() for t in us]
        su_ref = torch.empty_like(su)
        rmax_ref = _project(S, ref, ref, su_ref)
    for a, b in zip(outs, ref):
        assert torch.equal(a, b)
    assert torch.equal(su, su_ref)
    assert rmax == rmax_ref


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_gpu_velocity_loop_takes_new_arrays(gpu_lib, precision):
    """The captured step reads the arrays and dt from device memory: a second
    solve with other arrays and another dt equals a fresh handle's."""
    import torch
    from hydro3d_amd import MultigridSolver
    n = (48, 16, 24)
    spec = dict(n=n, h=(1 / 32,) * 3, bc=(1, 1, 0, 0, 0, 0), nlev=3)
    kw = dict(nu1=2, nu2=1, tol=1e-12, maxcy=4, criterion="ref_rmax")
    if precision == "mixed":
        kw.update(precision="mixed", coarse="exact")
    runs = [([t * 1e-3 for t in _faces(n, 10 + q)], 1e-3 * (q + 1)) for q in range(3)]
    p0 = torch.zeros(tuple(reversed(n)), device="cuda", dtype=torch.float64)
    with MultigridSolver([spec], **kw) as S:
        got = []
        for us, dt in runs:
            S.set_p(0, p0)
            S.set_dt(dt)
            _, nc, hist, out = S.solve_velocity(*[[t] for t in us])
            got.append((hist, [x[0] for x in out], S.result_p(0), S.get_su(0)))
    for (us, dt), (hist, out, p, su) in zip(runs, got):
        with MultigridSolver([spec], dt=dt, use_graph=False, **kw) as S:
            _, nc, h2, o2 = S.solve_velocity(*[[t] for t in us])
            assert np.array_equal(hist, h2)
            assert all(torch.equal(a, b[0]) for a, b in zip(out, o2))
            assert torch.equal(p, S.result_p(0)) and torch.equal(su, S.get_su(0))


def test_gpu_velocity_step_after_other_solves(gpu_lib):
    """A step whose level-1 rhs was overwritten in between (by a solve) starts
    from su all the same."""
    import torch
    from hydro3d_amd import MultigridSolver
    n = (32, 16, 16)
    spec = dict(n=n, h=(1 / 32,) * 3, bc=(0,) * 6, nlev=3)
    us = [t * 1e-3 for t in _faces(n, 7)]
    kw = dict(tol=1e-12, maxcy=3)
    res = []
    for between in (False, True):
        with MultigridSolver([spec], **kw) as S:
            S.velocity_begin(*[[t] for t in us])
            if between:
                p = S.result_p(0)
                S.solve()
                S.set_p(0, p)
            rm, keep = S.velocity_step(), S._vel_keep
            res.append((rm, S.result_p(0)))
            del keep
    assert res[0][0] == res[1][0] and torch.equal(res[0][1], res[1][1])
