"""The step with one lane per cell (the large grids' path) against the general
step kernel, which a chosen launch shape selects (16 lanes per cell: the order
of the sums that the mixed path keeps at level 5, FP64 that of 32): every layout and precision
it takes, grids at the smallest size it runs at and with ragged last
workgroups, lists that are empty, one short of a workgroup, full and one over,
tendency and in-place calls, contents below the limits, one NaN cell.

Both paths take the same FP64 sums in other orders (and the same FP32 pair
terms): 2^-53 on some 30 terms, grown over 50 substeps that change a content by
at most 10 % each (1.1^50 = 117) times a conditioning of up to 1e3 near
equilibrium gives 4e-10 of an element; 1e-12 of a row's rms covers elements
that a process empties, and cells at a switch (273 K, saturation) get ten
times what the general kernel itself moves between two launch shapes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RTOL, ATOL_RMS = 1e-9, 1e-12


@pytest.fixture(scope="module")
def capi():
    import torch
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    from salsa_amd import capi as c
    c.lib()
    return c


_MADE = {}


def fields(capi, species, level, grid):
    from salsa_amd import workload as W
    key = (species, level, grid)
    if key not in _MADE:
        desc = capi.bin_desc(species=species)
        kw = dict(W.CONFIGS[5 if level == 5 else 4])
        kw.update(grid=W.Grid(*grid), seed=3, level=level, cloud_frac=0.3)
        _MADE[key] = desc, W.generate(desc, **kw)
    return _MADE[key]


def step(capi, desc, f, prec, n, m, rv, general, inplace):
    g = f.grid
    ctx = capi.Context(desc, capi.params(level=f.level, precision=prec), g.nzp, g.nxp, g.nyp)
    for k in range(3 if general else 0):
        ctx.set_shape(k, general)
    fd = dict(press=f.press, temp=f.temp, rsl=f.rsl, rsi=f.rsi, dn=f.dn, rv=rv.copy())
    n, m = [x.copy() for x in n], [x.copy() for x in m]
    n_t, m_t, rv_t = [np.zeros_like(x) for x in n], [np.zeros_like(x) for x in m], np.zeros_like(rv)
    bad = None
    try:
        if inplace:
            ctx.step_host(fd, n, m, flags=capi.STEP_INPLACE)
        else:
            ctx.step_host(fd, n, m, n_t, m_t, rv_t)
    except capi.SalsaError as e:
        bad = e.code
    fl = ctx.cell_flags()
    ctx.close()
    out = n + m + [fd["rv"][None]] if inplace else \
        [a + b for a, b in zip(n + m, n_t + m_t)] + [(rv + rv_t)[None]]       # dt = 1 s
    return out, fl, bad


CASES = [
    # species, level, grid, cells with hydrometeors (None: as generated)
    (("SO4",), 4, (40, 16, 24), None),               # 15 360 cells: the smallest that runs it
    (("SO4",), 4, (41, 15, 25), 0),
    (("SO4",), 4, (41, 15, 25), 65),
    (("SO4", "DU"), 4, (41, 15, 25), 64),
    (("SO4",), 5, (40, 8, 16), 63),
    (("SO4", "DU"), 5, (32, 8, 16), 63),             # 4 096 cells: the smallest
    (("SO4",), 5, (43, 11, 11), None),
    (("SO4", "DU"), 5, (43, 11, 11), None),
    (("SO4", "DU"), 5, (43, 11, 11), 1),
]


@pytest.mark.parametrize("inplace", [0, 1])
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("species,level,grid,nhyd", CASES)
def test_one_lane_per_cell_matches_general_kernel(capi, species, level, grid, nhyd, prec, inplace):
    print("case %s level %d grid %s hyd %s prec %d inplace %d" % (species, level, grid, nhyd, prec, inplace), flush=True)
    desc, f = fields(capi, species, level, grid)
    ncat = 4 if level == 5 else 3
    idx = f.grid.interior_index()
    n, m, rv = [x.copy() for x in f.n[:ncat]], [x.copy() for x in f.m[:ncat]], f.rv
    nan = None
    if nhyd is not None:
        has = np.zeros(len(idx), bool)
        for c in range(1, ncat):
            has |= (n[c][:, idx] > 0.).any(axis=0)
        off = idx[np.flatnonzero(has)[nhyd:]]        # the others lose theirs, but for contents below the limits
        for c in range(1, ncat):
            n[c][:, off] *= 0.
            m[c][:, off] *= 0.
            n[c][0, off[::3]] = 1.e-12
            m[c][:, off[::3]] = 1.e-24
        nan = 7
        rv = rv.copy()
        rv[idx[nan]] = np.nan
    a, fa, ea = step(capi, desc, f, prec, n, m, rv, 0, inplace)
    b, fb, eb = step(capi, desc, f, prec, n, m, rv, 16, inplace)
    b2, _, _ = step(capi, desc, f, prec, n, m, rv, 32, inplace)
    assert ea == eb and np.array_equal(fa, fb)
    keep = np.ones(len(idx), bool)
    if nan is not None:
        assert ea == capi.SALSA_ERR_NONFINITE and fa[nan] & capi.CELL_NONFINITE
        assert np.flatnonzero(fa & capi.CELL_NONFINITE).tolist() == [nan]
        keep[nan] = False
    halo = np.setdiff1d(np.arange(f.grid.ncell3d), idx)
    for x, y, y2 in zip(a, b, b2):
        assert np.array_equal(x[:, halo], y[:, halo])
        x, y, y2 = x[:, idx[keep]], y[:, idx[keep]], y2[:, idx[keep]]
        rms = np.sqrt(np.mean(y * y, axis=1, keepdims=True))
        bad = ~(np.abs(x - y) <= RTOL * np.abs(y) + ATOL_RMS * rms + 10. * np.abs(y - y2))
        assert not bad.any(), (np.argwhere(bad)[:3], x[bad][:3], y[bad][:3], y2[bad][:3])


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("level,grid", [(4, (1, 1, 1)), (4, (13, 5, 1)), (4, (39, 19, 20)), (5, (1, 1, 1)), (5, (33, 3, 7)),
                                        (5, (31, 11, 11))])
def test_small_grids_match_the_launches_by_class(capi, level, grid, prec):
    """Below the sizes of the one-lane path every cell runs in one launch, 32
    (level 5: 64, above 2 048 cells 16) lanes each: bit for bit what the launches by cost class give
    at those lanes."""
    print("case level %d grid %s prec %d" % (level, grid, prec), flush=True)
    desc, f = fields(capi, ("SO4", "DU"), level, grid)
    ncat = 4 if level == 5 else 3
    lanes = 32 if level == 4 else 64 if f.grid.ncells <= 2048 else 16
    for inplace in (0, 1):
        a, fa, ea = step(capi, desc, f, prec, f.n[:ncat], f.m[:ncat], f.rv, 0, inplace)
        b, fb, eb = step(capi, desc, f, prec, f.n[:ncat], f.m[:ncat], f.rv, lanes, inplace)
        assert ea == eb and np.array_equal(fa, fb)
        for x, y in zip(a, b):
            assert np.array_equal(x, y)
