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
