"""The cell-by-cell sweep and restriction (blocks with neighbours, blocks one
cell wide in x, variable density) against a NumPy transcription of the
operators, at uneven and odd sizes: rows over and under a tile's 64 cells,
neighbours of other extents, single cells.  Needs an MI355X.  Bitwise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
WALL, PER, NBR = 0, 1, 2
H = (0.02, 0.03, 0.011)


def _line(axis, ns, wrap, other=(3, 5, 4)):
    """Blocks of extents ns side by side along axis; walls or a wrap at its
    ends, periodic and walls on the two other axes."""
    specs = []
    for b, n in enumerate(ns):
        dims = list(other)
        dims[axis] = n
        bc, nbr = [WALL] * 6, [-1] * 6
        per = (axis + 1) % 3
        bc[2 * per] = bc[2 * per + 1] = PER
        for side, q in ((0, b - 1), (1, b + 1)):
            f = 2 * axis + side
            if 0 <= q < len(ns) or wrap:
                bc[f] = NBR if len(ns) > 1 else PER
                nbr[f] = q % len(ns) if len(ns) > 1 else -1
        specs.append(dict(n=tuple(dims), h=H, bc=tuple(bc), nbr=tuple(nbr), nlev=1))
    return specs


CASES = {"x": _line(0, (5, 67, 130), False), "x wrap": _line(0, (66, 3), True),
         "y": _line(1, (3, 8, 1), True, (70, 0, 3)), "z": _line(2, (2, 7), False, (33, 5, 0)),
         "x ones": _line(0, (1, 2, 1), True), "one wide": _line(0, (1,), False),
         "one wide wrap": _line(0, (1,), True)}


def _padded(specs, arrs, b):
    """arrs[b] with its six face ghosts (walls mirror; then neighbour or
    wrap)."""
    a, s = arrs[b], specs[b]
    p = np.pad(a, 1, mode="edge")
    for ax in range(3):
        for side in range(2):
            f, npax = 2 * ax + side, 2 - ax
            if s["bc"][f] == WALL:
                continue
            o = arrs[s["nbr"][f]] if s["bc"][f] == NBR else a
            dst, src = [slice(1, -1)] * 3, [slice(None)] * 3
            dst[npax] = slice(-1, None) if side else slice(0, 1)
            src[npax] = slice(0, 1) if side else slice(-1, None)
            p[tuple(dst)] = o[tuple(src)]
    return p


def _coefs(s, dens=None):
    n = s["n"]
    shape = n[::-1]
    c = []
    for f in range(6):
        ax, side = f // 2, f % 2
        if dens is None:
            v = np.full(shape, 1.0 / (H[ax] * H[ax]))
        else:
            d = np.pad(dens, 1, mode="edge")
            at = [slice(1, -1)] * 3
            at[2 - ax] = slice(2, None) if side else slice(0, -2)
            mean = 0.5 * (dens + d[tuple(at)])
            edge = [slice(None)] * 3
            edge[2 - ax] = slice(-1, None) if side else slice(0, 1)
            mean[tuple(edge)] = dens[tuple(edge)]
            u, w = [H[q] for q in range(3) if q != ax]
            v = u * w / H[ax] / mean
        if s["bc"][f] == WALL:
            edge = [slice(None)] * 3
            edge[2 - ax] = slice(-1, None) if side else slice(0, 1)
            v[tuple(edge)] = 0.0
        c.append(v)
    return c, -1.0 * (c[0] + c[1] + c[2] + c[3] + c[4] + c[5])


def _sum(c, p):
    m = slice(1, -1)
    v = [p[m, m, :-2], p[m, m, 2:], p[m, :-2, m], p[m, 2:, m], p[:-2, m, m], p[2:, m, m]]
    return c[0] * v[0] + c[1] * v[1] + c[2] * v[2] + c[3] * v[3] + c[4] * v[4] + c[5] * v[5]


def _colour(shape):
    return np.indices(shape).sum(0) & 1


def _sweep(specs, phis, rhss, dens=None):
    out = []
    for b, s in enumerate(specs):
        p = _padded(specs, phis, b)
        c, ap = _coefs(s, dens)
        col = _colour(phis[b].shape)
        for colour in (0, 1):  # ghosts keep the state before the sweep
            new = (rhss[b] - _sum(c, p)) / ap
            p[1:-1, 1:-1, 1:-1] = np.where(col == colour, new, p[1:-1, 1:-1, 1:-1])
        out.append(p[1:-1, 1:-1, 1:-1].copy())
    return out


def _restrict(specs, phis, rhss, dens=None):
    out = []
    for b, s in enumerate(specs):
        p = _padded(specs, phis, b)
        c, ap = _coefs(s, dens)
        r = rhss[b] - (_sum(c, p) + ap * phis[b])
        q = [r[z::2, y::2, x::2] for z in (0, 1) for y in (0, 1) for x in (0, 1)]
        acc = q[0]
        for v in q[1:]:
            acc = acc + v
        out.append(0.125 * acc)
    return out


def _run(specs, op, dens=None):
    import torch
    from hydro3d_amd import MultigridSolver
    from hydro3d_amd import _lib as L
    rng = np.random.default_rng(4)
    phis = [rng.standard_normal(s["n"][::-1]) for s in specs]
    rhss = [rng.standard_normal(s["n"][::-1]) for s in specs]
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    with MultigridSolver(specs, use_graph=False) as S:
        if dens is not None:
            S.set_density(0, dens)
        for b in range(len(specs)):
            S.dbg_put(b, 1, L.ARR_PHI, dev(np.pad(phis[b], 1)))
            S.dbg_put(b, 1, L.ARR_RHS, dev(rhss[b]))
        ref = phis
        if op == "relax":
            S.dbg_relax(1, 2)
            for _ in range(2):
                ref = _sweep(specs, ref, rhss, dens)
        else:
            S.dbg_restrict(2)
            ref = _restrict(specs, phis, rhss, dens)
        for b, s in enumerate(specs):
            n = s["n"][::-1]
            if op == "relax":
                out = S.dbg_get(b, 1, L.ARR_PHI, torch.empty([q + 2 for q in n], dtype=torch.float64,
                                                             device="cuda"))[1:-1, 1:-1, 1:-1]
            else:
                out = S.dbg_get(b, 2, L.ARR_RHS, torch.empty([q // 2 for q in n],
                                                             dtype=torch.float64, device="cuda"))
            assert np.array_equal(out.cpu().numpy(), ref[b]), (op, b)


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("op", ["relax", "restrict"])
def test_gpu_cell_kernels_blocks(gpu_lib, name, op):
    print(f"case: {op} {name}", flush=True)
    specs = CASES[name]
    if op == "restrict":
        specs = [dict(s, n=tuple(2 * q for q in s["n"]), nlev=2) for s in specs]
    _run(specs, op)


@pytest.mark.parametrize("n", [(5, 3, 70), (130, 6, 2), (1, 4, 5), (64, 4, 1), (67, 9, 3)])
@pytest.mark.parametrize("op", ["relax", "restrict"])
def test_gpu_cell_kernels_density(gpu_lib, n, op):
    print(f"case: density {op} {n}", flush=True)
    if op == "restrict":
        n = tuple(2 * q for q in n)
    spec = dict(n=n, h=H, bc=(1, 1, 0, 0, 0, 0), nlev=1 if op == "relax" else 2)
    dens = np.random.default_rng(7).uniform(0.5, 20.0, n[::-1])
    _run([spec], op, dens)
