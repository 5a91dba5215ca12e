"""The projection of one block of several, pooled and not: its partials lie in
the block's own range or, for blocks of few or short rows, after the last one.
Against the same block alone in a handle.  Needs an MI355X.  Bitwise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NS = [(64, 32, 16), (5, 1, 7), (4, 4, 4), (1, 64, 64), (8, 8, 130), (33, 17, 9)]


@pytest.mark.parametrize("pooled", [False, True])
def test_gpu_projection_of_each_block(gpu_lib, pooled):
    import torch
    from hydro3d_amd.solver import DevicePool, MultigridSolver, block_bytes
    specs = [dict(n=n, h=(0.02, 0.03, 0.011), bc=(0, 0, 1, 1, 0, 0), nlev=1) for n in NS]
    g = torch.Generator(device="cuda").manual_seed(3)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda", dtype=torch.float64)  # noqa: E731
    args = [(rnd(nk, nj, ni + 1), rnd(nk, nj + 1, ni), rnd(nk + 1, nj, ni)) for ni, nj, nk in NS]
    ps = [rnd(*n[::-1]) for n in NS]
    alone = []
    for s, a, p in zip(specs, args, ps):
        with MultigridSolver([s]) as S:
            S.set_p(0, p)
            alone.append(S.project(0, *a))
    pool = DevicePool(1 << 27, 16) if pooled else None
    kw = dict(pool=pool, offsets=[pool.alloc(block_bytes(s)) for s in specs]) if pooled else {}
    with MultigridSolver(specs, **kw) as S:
        for b, p in enumerate(ps):
            S.set_p(b, p)
        for b, a in enumerate(args):
            print(f"case: projection of block {b} {NS[b]} pooled {pooled}", flush=True)
            out = S.project(b, *a)
            for x, y in zip(out[:4], alone[b][:4]):
                assert torch.equal(x, y)
            div = ((out[0][:, :, 1:] - out[0][:, :, :-1]) / 0.02 +
                   (out[1][:, 1:] - out[1][:, :-1]) / 0.03 + (out[2][1:] - out[2][:-1]) / 0.011)
            want = float(div.abs().max()) * 0.02 * 0.03 * 0.011
            assert out[4] == alone[b][4] and abs(out[4] - want) <= 1e-12 * want
    if pooled:
        for o in kw["offsets"]:
            pool.free(o)
        pool.close()
