"""p += pp inside level 1's last half-sweep (k_rb_sweep, k_rb_tile) against the
fused sweeps followed by k_update: planes per tile, odd rows (pad entries),
walls and periodic faces, several blocks, a disabled block.  Needs an MI355X.
Bitwise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BCS = [(0,) * 6, (1,) * 6, (1, 1, 0, 0, 1, 1)]


def _run(specs, fs, p0, march, nu, kw, off=None):
    from hydro3d_amd import MultigridSolver
    nlev = specs[0]["nlev"]
    with MultigridSolver(specs, nu1=nu[0], nu2=nu[1], tol=0.0, maxcy=2, **kw) as S:
        S.set_tail(nlev + 1)
        if march is None:
            S.set_fused(10 ** 9)
        else:
            for g in range(1, nlev + 1):
                S.set_march(g, march)
        for b, f in enumerate(fs):
            S.set_rhs(b, f)
            S.set_p(b, p0[b])
        if off is not None:
            S.set_block_enabled(off, False)
        S.solve()
        return [S.get_p(b) for b in range(len(specs))], [S.get_pp(b) for b in range(len(specs))]


@pytest.mark.parametrize("kw", [dict(), dict(precision="mixed", coarse="exact")], ids=str)
@pytest.mark.parametrize("n", [(16, 16, 16), (6, 10, 4), (262, 4, 8), (50, 22, 36)])
@pytest.mark.parametrize("blocks", [1, 3])
def test_gpu_update_in_sweep(gpu_lib, n, blocks, kw):
    rng = np.random.default_rng(8)
    for bc in BCS:
        specs = [dict(n=n if b != 1 else (4, 4, 8), h=(0.02, 0.03, 0.011), bc=bc, nlev=2)
                 for b in range(blocks)]
        fs = [rng.standard_normal(s["n"][::-1]) for s in specs]
        fs = [f - f.mean() for f in fs]
        p0 = [rng.standard_normal(s["n"][::-1]) for s in specs]
        for nu in [(2, 2), (1, 1), (2, 3)]:
            off = 2 if blocks == 3 and nu == (1, 1) else None
            ref = _run(specs, fs, p0, None, nu, kw, off)
            for march in (0, 1, 2, 4):
                print(f"case: {blocks} x {n} bc {bc} nu {nu} march {march} {kw}", flush=True)
                out = _run(specs, fs, p0, march, nu, kw, off)
                for b in range(blocks):
                    assert np.array_equal(out[0][b], ref[0][b]), (bc, nu, march, b)
                    if b != off:
                        assert np.array_equal(out[1][b], ref[1][b]), (bc, nu, march, b)
