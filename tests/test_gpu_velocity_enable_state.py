"""A block enabled through h3dmg_set_block_state between h3dmg_velocity_begin
and h3dmg_velocity_step: the begin's projection left it out, so the step's
V-cycle starts from its f, not from what its level-1 right-hand side holds
(a solve's residual).  Needs an MI355X.  Bitwise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_gpu_enabled_block_starts_from_its_f(gpu_lib, precision):
    import torch
    from hydro3d_amd import MultigridSolver
    n = (16, 24, 32)
    spec = dict(n=n, h=(0.02, 0.03, 0.011), bc=(1, 1, 0, 0, 1, 1), nlev=3)
    rng = np.random.default_rng(14)
    vel = [torch.from_numpy(rng.standard_normal((32 + (a == 2), 24 + (a == 1), 16 + (a == 0)))).cuda()
           for a in range(3)]
    kw = dict(precision=precision, tol=0.0, maxcy=2)
    print(f"case: block enabled by its state, {precision}", flush=True)
    with MultigridSolver([spec, spec], **kw) as S:
        _, first = S.velocity_begin(*[[t, t] for t in vel])  # `first`: block 1's outputs live on
        S.set_rhs(1, rng.standard_normal(n[::-1]))
        S.solve()
        S.set_block_enabled(1, False)
        S.velocity_begin(*[[t, None] for t in vel])
        st = S.block_state(1)
        st.enabled = 1
        S.set_block_state(1, st)
        p, f = S.result_p(1), S.get_su(1)
        S.velocity_step()
        out = S.get_p(1)[1:-1, 1:-1, 1:-1]
        assert len(first) == 3
    with MultigridSolver([spec], **kw) as R:
        R.set_rhs(0, f)
        R.vcycle()
        pp = R.get_pp(0)[1:-1, 1:-1, 1:-1]
    assert np.array_equal(out, p.cpu().numpy() + pp)
