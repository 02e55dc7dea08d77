"""Properties that the routes of a step share: what a call gives does not depend
on timing, on values that a step takes for empty, or on earlier calls."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    import torch
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    from salsa_amd import capi as c
    c.lib()
    return c


def fields(capi, species, level, grid, **over):
    from salsa_amd import workload as W
    desc = capi.bin_desc(species=species)
    kw = dict(W.CONFIGS[5 if level == 5 else 4])
    kw.update(grid=W.Grid(*grid), seed=5, level=level, cloud_frac=0.4)
    kw.update(over)
    return desc, W.generate(desc, **kw)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("species", [("SO4",), ("SO4", "DU")])
def test_one_lane_step_with_ice_repeats_its_bits(capi, species, prec):
    """Wavefronts of a workgroup share an ice target: its old water and rime feed
    the new rime fraction while other wavefronts replace them.  With ice in
    every cell, two workgroups per compute unit's worth of cells and more, every
    repetition gives the first one's bits."""
    import torch
    print("case ice step repeated, %s prec %d" % (species, prec), flush=True)
    desc, f = fields(capi, species, 5, (40, 24, 40), cloud_mode="random", cloud_frac=1., t_range=(240., 272.))
    g = f.grid
    T = lambda a: torch.from_numpy(np.array(a)).cuda()
    fd = {k: T(getattr(f, k)) for k in ("press", "temp", "rsl", "rsi", "dn", "rv")}
    n, m = [T(x) for x in f.n], [T(x) for x in f.m]
    ctx = capi.Context(desc, capi.params(level=5, precision=prec), g.nzp, g.nxp, g.nyp)
    want = None
    for _ in range(12):
        out = [torch.zeros_like(x) for x in n + m + [fd["rv"]]]
        ctx.step_device(fd, n, m, out[:4], out[4:8], out[8])
        ctx.sync()
        if want is None:
            want = out
            assert want[3].any() and want[7].any()
        for a, b in zip(out, want):
            assert torch.equal(a, b)
    ctx.close()


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("level", [4, 5])
def test_nan_and_negative_masses_of_inactive_bins(capi, level, prec):
    """Masses of a hydrometeor bin below its number limit that are NaN or negative
    are empty after a step and add nothing to a cell's water: the one-lane step
    agrees with the general kernel (at 16 and 32 lanes), which clamps them first.

    The bar is that of the comparison of the two paths elsewhere: 2^-53 on some
    30 terms, grown by 1.1^50 = 117 in the substeps times a conditioning of 1e3,
    1e-9 of an element; 1e-12 of a row's rms for what a process empties; ten
    times what the general kernel moves between two shapes."""
    print("case NaN in inactive bins, level %d prec %d" % (level, prec), flush=True)
    desc, f = fields(capi, ("SO4",), level, (41, 20, 20), rh_range=(0.99, 1.01))
    g, ncat = f.grid, 4 if level == 5 else 3
    idx = g.interior_index()
    n, m = [x.copy() for x in f.n[:ncat]], [x.copy() for x in f.m[:ncat]]
    for c in range(1, ncat):                                # (level 5 has ice in every cell)
        n[c][:, idx[::2]] = 0.
        m[c][:, idx[::2]] = 0.
    has = np.zeros(len(idx), bool)
    for c in range(1, ncat):
        has |= (n[c][:, idx] > 0.).any(axis=0)
    off = idx[~has]
    assert len(off) > 1000
    water = desc.iwa * np.array([desc.nbins, desc.ncld, desc.nprc, desc.nice])
    for c in range(1, ncat):
        m[c][water[c], off[c::4]] = np.nan
        m[c][water[c] + 1, off[c::3]] = -1.e-4
        m[c][water[c] + 2, off[c::5]] = 1.e-9
    res = []
    for shape in (0, 16, 32):
        ctx = capi.Context(desc, capi.params(level=level, precision=prec), g.nzp, g.nxp, g.nyp)
        for k in range(3 if shape else 0):
            ctx.set_shape(k, shape)
        a, b = [x.copy() for x in n], [x.copy() for x in m]
        fd = {k: np.array(getattr(f, k)) for k in ("press", "temp", "rsl", "rsi", "dn", "rv")}
        ctx.step_host(fd, a, b, flags=capi.STEP_INPLACE)        # raises where a cell is not finite
        res.append(([x[:, idx] for x in a + b + [fd["rv"][None]]], ctx.cell_flags()))
        ctx.close()
    assert np.array_equal(res[0][1], res[1][1])
    for x, y, y2 in zip(res[0][0], res[1][0], res[2][0]):
        rms = np.sqrt(np.mean(y * y, axis=1, keepdims=True))
        bad = ~(np.abs(x - y) <= 1e-9 * np.abs(y) + 1e-12 * rms + 10. * np.abs(y - y2))
        assert not bad.any(), (np.argwhere(bad)[:3], x[bad][:3], y[bad][:3], y2[bad][:3])


def test_only_steps_take_the_step_work_space(capi):
    """A context that never steps with one lane per cell (sedimentation, a chosen
    launch shape) holds no work space of that step: what creating and using it
    takes is its cell records, lists and flags, and 32 MB for the runtime's own
    granules.  A context's first step makes the space, another one reuses it."""
    import torch
    desc, f = fields(capi, ("SO4",), 4, (60, 48, 48))
    g = f.grid
    free = lambda: (torch.cuda.synchronize(), torch.cuda.mem_get_info()[0])[1]
    T = lambda a: torch.from_numpy(np.array(a)).cuda()
    fd = {k: T(getattr(f, k)) for k in ("press", "temp", "rsl", "rsi", "dn", "rv")}
    n, m = [T(x) for x in f.n[:3]], [T(x) for x in f.m[:3]]
    out = [torch.zeros_like(x) for x in n + m + [fd["rv"]]]
    step = lambda c: c.step_device(fd, n, m, out[:3], out[3:6], out[6])
    warm = capi.Context(desc, capi.params(level=4), g.nzp, g.nxp, g.nyp)     # code and queues are loaded by now
    step(warm)
    warm.sync()
    warm.close()
    rows = 3 * (desc.nbins + desc.ncld + desc.nprc)                          # number and two masses
    records = 8 * g.ncells * (2 * rows + 7) + 16 * g.ncells
    start = free()
    ctx = capi.Context(desc, capi.params(level=4), g.nzp, g.nxp, g.nyp)
    for k in range(3):
        ctx.set_shape(k, 16)
    step(ctx)
    ctx.sync()
    assert start - free() < records + (32 << 20)
    ctx.close()
    ctx = capi.Context(desc, capi.params(level=4), g.nzp, g.nxp, g.nyp)
    assert start - free() < records + (32 << 20)
    step(ctx)
    ctx.sync()
    after = free()
    step(ctx)
    ctx.sync()
    assert free() >= after                                                   # (other objects may go meanwhile)
    ctx.close()


@pytest.mark.parametrize("level,grid", [(4, (40, 16, 25)), (5, (40, 11, 11)), (4, (30, 8, 8)), (4, (39, 19, 20))])
def test_first_step_of_a_context_within_a_capture(capi, level, grid):
    """The first step makes its work space also within a stream capture, and grids
    that go by cost class otherwise take one launch there; replays, with other
    work between them, give the bits of an eager step."""
    import torch
    print("case first step captured, level %d" % level, flush=True)
    desc, f = fields(capi, ("SO4",), level, grid)
    g, ncat = f.grid, 4 if level == 5 else 3
    T = lambda a: torch.from_numpy(np.array(a)).cuda()
    fd = {k: T(getattr(f, k)) for k in ("press", "temp", "rsl", "rsi", "dn", "rv")}
    n, m = [T(x) for x in f.n[:ncat]], [T(x) for x in f.m[:ncat]]
    out = [torch.zeros_like(x) for x in n + m + [fd["rv"]]]
    step = lambda c: c.step_device(fd, n, m, out[:ncat], out[ncat:2 * ncat], out[-1])
    ctx = capi.Context(desc, capi.params(level=level), g.nzp, g.nxp, g.nyp)
    step(ctx)
    ctx.sync()
    ctx.close()
    want = [x.clone() for x in out]
    ctx = capi.Context(desc, capi.params(level=level), g.nzp, g.nxp, g.nyp)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=torch.cuda.ExternalStream(ctx.stream), capture_error_mode="thread_local"):
        step(ctx)
    for _ in range(3):
        for x in out:
            x.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, want):
            assert torch.equal(a, b)
    ctx.close()


def test_class_counts_of_many_timed_steps(capi):
    """salsa_ctx_phase_time adds up every timed step's own class counts, also past
    the 4 096 steps whose counts travel without a wait: steps without hydrometeors,
    but for twenty on both sides of that number with them in known cells."""
    import torch
    desc, f = fields(capi, ("SO4",), 4, (40, 16, 24))
    g = f.grid
    idx = torch.from_numpy(g.interior_index()).cuda()
    T = lambda a: torch.from_numpy(np.array(a)).cuda()
    fd = {k: T(getattr(f, k)) for k in ("press", "temp", "rsl", "rsi", "dn", "rv")}
    n, m = [T(x) for x in f.n[:3]], [T(x) for x in f.m[:3]]
    out = [torch.zeros_like(x) for x in n + m + [fd["rv"]]]
    dry = [n[0]] + [torch.zeros_like(x) for x in n[1:]]
    nhyd = int(((n[1][:, idx] > 0.).any(0) | (n[2][:, idx] > 0.).any(0)).sum())
    assert 0 < nhyd < g.ncells
    ctx = capi.Context(desc, capi.params(level=4), g.nzp, g.nxp, g.nyp)
    ctx.timing(True)
    steps = 4096 + 40
    for k in range(steps):
        ctx.step_device(fd, n if 4090 <= k < 4110 else dry, m, out[:3], out[3:6], out[6], tstep=0.02)
    ms, cells, nsteps = ctx.phase_time()
    ctx.timing(False)
    ctx.close()
    assert nsteps == steps
    assert cells[2] == 20 * nhyd
    assert sum(cells) == steps * g.ncells


@pytest.mark.parametrize("grid", [(40, 16, 24), (20, 8, 8)])
def test_autotune_keeps_a_chosen_launch_by_class(capi, grid):
    """salsa_set_launch_shape selects launches by cost class for every step of the
    context; salsa_autotune changes the shapes, not that choice: the step gives the
    bits of a context whose shapes were set to what the autotuner found.  Without a
    chosen shape the route stays the context's own."""
    import torch
    desc, f = fields(capi, ("SO4",), 4, grid)
    g = f.grid
    T = lambda a: torch.from_numpy(np.array(a)).cuda()
    fd = {k: T(getattr(f, k)) for k in ("press", "temp", "rsl", "rsi", "dn", "rv")}
    n, m = [T(x) for x in f.n[:3]], [T(x) for x in f.m[:3]]

    def step(shapes, tune):
        ctx = capi.Context(desc, capi.params(level=4), g.nzp, g.nxp, g.nyp)
        for k, s in enumerate(shapes):
            ctx.set_shape(k, s)
        if tune:
            ctx.autotune(fd, n, m)
        out = [torch.zeros_like(x) for x in n + m + [fd["rv"]]]
        ctx.step_device(fd, n, m, out[:3], out[3:6], out[6])
        ctx.sync()
        found = [ctx.shape_of(k) for k in range(3)]
        ctx.close()
        return out, found

    tuned, found = step((64, 64, 64), True)
    by_class, _ = step(found, False)
    for a, b in zip(tuned, by_class):
        assert torch.equal(a, b)
    own, _ = step((), False)
    after, _ = step((), True)
    for a, b in zip(own, after):
        assert torch.equal(a, b)


@pytest.mark.parametrize("prec", [0, 1])
def test_one_lane_step_takes_the_layouts_ice_limit(capi, prec):
    """The number below which an ice bin is empty is the layout's: with a lower one
    than usual, and particles between the two, the one-lane step agrees with the
    general kernel at two shapes (the bar of the comparison of the two paths above)."""
    print("case ice limit of the layout, prec %d" % prec, flush=True)
    desc, f = fields(capi, ("SO4",), 5, (41, 20, 12), t_range=(240., 270.))
    g = f.grid
    idx = g.interior_index()
    ice0 = desc.nbins + desc.ncld + desc.nprc
    for b in range(desc.nice):
        desc.nlim[ice0 + b] = 1.e-12
    n, m = [x.copy() for x in f.n], [x.copy() for x in f.m]
    # every other bin with particles of its own mass, but some 1e-8 per kg of them, and mostly rimed: the others
    # collect them at an efficiency that their rime fraction sets
    water, rime = desc.iwa * desc.nice, desc.irim * desc.nice
    m[3][rime:rime + desc.nice] = 0.1 * m[3][water:water + desc.nice]
    for b in range(0, desc.nice, 2):
        few = 1.e-8 / np.maximum(n[3][b], 1.e-8)
        n[3][b] *= few
        m[3][b::desc.nice] *= few
        m[3][rime + b] = 3. * m[3][water + b]
    res = []
    for shape in (0, 16, 32):
        ctx = capi.Context(desc, capi.params(level=5, precision=prec), g.nzp, g.nxp, g.nyp)
        for k in range(3 if shape else 0):
            ctx.set_shape(k, shape)
        a, b = [x.copy() for x in n], [x.copy() for x in m]
        fd = {k: np.array(getattr(f, k)) for k in ("press", "temp", "rsl", "rsi", "dn", "rv")}
        ctx.step_host(fd, a, b, flags=capi.STEP_INPLACE)
        res.append([x[:, idx] for x in a + b + [fd["rv"][None]]])
        ctx.close()
    for x, y, y2 in zip(*res):
        rms = np.sqrt(np.mean(y * y, axis=1, keepdims=True))
        bad = ~(np.abs(x - y) <= 1e-9 * np.abs(y) + 1e-12 * rms + 10. * np.abs(y - y2))
        assert not bad.any(), (np.argwhere(bad)[:3], x[bad][:3], y[bad][:3], y2[bad][:3])


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("level,grid", [(4, (23, 8, 7)), (5, (23, 8, 7)), (5, (23, 11, 12))])
def test_small_grids_with_nan_in_inactive_bins(capi, level, grid, prec):
    """A cell without active hydrometeors steps the same in the one launch of a small
    grid as in the launch of its cost class, whatever its inactive bins hold: bit
    for bit at the same lanes per cell, NaN and negative masses among them."""
    print("case small grid with NaN in inactive bins, level %d grid %s prec %d" % (level, grid, prec), flush=True)
    desc, f = fields(capi, ("SO4", "DU"), level, grid)
    g, ncat = f.grid, 4 if level == 5 else 3
    idx = g.interior_index()
    n, m = [x.copy() for x in f.n[:ncat]], [x.copy() for x in f.m[:ncat]]
    for c in range(1, ncat):
        n[c][:, idx[::2]] = 0.
        m[c][:, idx[::2]] = 0.
        m[c][0, idx[::4]] = np.nan
        m[c][-1, idx[::6]] = np.nan
        m[c][1, idx[::10]] = -1.e-5
    lanes = 32 if level == 4 else 64 if g.ncells <= 2048 else 16
    res = []
    for shape in (0, lanes):
        ctx = capi.Context(desc, capi.params(level=level, precision=prec), g.nzp, g.nxp, g.nyp)
        for k in range(3 if shape else 0):
            ctx.set_shape(k, shape)
        a, b = [x.copy() for x in n], [x.copy() for x in m]
        fd = {k: np.array(getattr(f, k)) for k in ("press", "temp", "rsl", "rsi", "dn", "rv")}
        ctx.step_host(fd, a, b, flags=capi.STEP_INPLACE)
        res.append(([x[:, idx] for x in a + b + [fd["rv"][None]]], ctx.cell_flags()))
        ctx.close()
    assert np.array_equal(res[0][1], res[1][1])
    for x, y in zip(res[0][0], res[1][0]):
        assert np.array_equal(x, y), np.argwhere(x != y)[:3]
