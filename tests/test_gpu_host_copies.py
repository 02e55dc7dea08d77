"""salsa_step_host where its fields travel in several pieces: the same bits as
the step on device fields, tendency and in-place, with process rates, at a size
whose arrays are one piece and less, and several and a remainder."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level,grid", [(4, (3, 2, 2)), (4, (40, 24, 27)), (5, (37, 21, 24))])
@pytest.mark.parametrize("inplace,rates", [(0, 0), (1, 0), (0, 1)])
def test_host_entry_matches_device_entry(level, grid, inplace, rates):
    import torch
    from salsa_amd import capi, workload as W
    print("case host copies, level %d grid %s inplace %d rates %d" % (level, grid, inplace, rates), flush=True)
    desc = capi.bin_desc(species=("SO4", "DU") if level == 5 else ("SO4",))
    f = W.config_fields(desc, 5 if level == 5 else 4, grid_override=grid)
    g, ncat = f.grid, 4 if level == 5 else 3
    rng = np.random.default_rng(1)
    names = ("press", "temp", "rsl", "rsi", "dn", "rv")
    n, m = [x.copy() for x in f.n[:ncat]], [x.copy() for x in f.m[:ncat]]
    nt, mt = [1e-3 * rng.random(x.shape) * x for x in n], [1e-3 * rng.random(x.shape) * x for x in m]
    rvt = 1e-9 * rng.random(f.rv.shape)
    shape = ((capi.NRATE_L5 if level == 5 else capi.NRATE_L4), g.nyp, g.nxp, g.nzp)
    r = np.full(shape, 3.) if rates else None
    hf = {k: np.array(getattr(f, k)) for k in names}
    T = lambda a: torch.from_numpy(np.array(a)).cuda()
    df = {k: T(v) for k, v in hf.items()}
    dn, dm, dnt, dmt = ([T(a) for a in x] for x in (n, m, nt, mt))
    drv, dr = T(rvt), T(r) if rates else None
    flags = capi.STEP_INPLACE if inplace else capi.STEP_TENDENCY
    ctx = capi.Context(desc, capi.params(level=level), g.nzp, g.nxp, g.nyp)
    for _ in range(2):
        ctx.step_host(hf, n, m, nt, mt, rvt, flags=flags, rates=r)
    ctx.close()
    ctx = capi.Context(desc, capi.params(level=level), g.nzp, g.nxp, g.nyp)
    for _ in range(2):
        ctx.step_device(df, dn, dm, dnt, dmt, drv, flags=flags, rates=dr)
    ctx.sync()
    ctx.close()
    for a, b in zip([hf["rv"], rvt] + n + m + nt + mt + ([r] if rates else []),
                    [df["rv"], drv] + dn + dm + dnt + dmt + ([dr] if rates else [])):
        assert np.array_equal(a, b.cpu().numpy())
