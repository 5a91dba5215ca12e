"""Line TDMA in a pooled handle, whose blocks' regions hold no workspace of the
two-launch line passes, against the oracle's sequential sweeps.  Needs an
MI355X.  Bitwise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SPECS = [((32, 32, 32), 3), ((17, 9, 33), 1), ((64, 48, 40), 3)]


@pytest.mark.parametrize("which", [(0,), (0, 2), (1,)])
def test_gpu_tdma_pooled_equals_oracle(gpu_lib, which):
    import torch
    from hydro3d_amd.solver import DevicePool, MultigridSolver, block_bytes
    from oracle import oracle as O
    print(f"case: pooled TDMA {which}", flush=True)
    bc = (1, 1, 0, 0, 1, 1)
    rng = np.random.default_rng(13)
    specs = [dict(n=SPECS[q][0], h=(0.02, 0.03, 0.011), bc=bc, nlev=SPECS[q][1]) for q in which]
    fs = [rng.standard_normal(s["n"][::-1]) for s in specs]
    fs = [f - f.mean() for f in fs]
    with DevicePool(1 << 28, 8) as pool:
        offs = [pool.alloc(block_bytes(s, smoother="tdma")) for s in specs]
        with MultigridSolver(specs, tol=0.0, maxcy=2, smoother="tdma", pool=pool,
                             offsets=offs) as S:
            for b, f in enumerate(fs):
                S.set_rhs(b, torch.from_numpy(f).cuda())
            S.solve()
            ps = [S.result_p(b).cpu().numpy() for b in range(len(specs))]
        for o in offs:
            pool.free(o)
    for s, f, p in zip(specs, fs, ps):
        po, _ = O.solve(O.Block(s["n"], s["h"], bc, s["nlev"]), f, 2, 0.0, scheme=O.SCHEME_TDMA)
        assert np.array_equal(p, po[1:-1, 1:-1, 1:-1])
