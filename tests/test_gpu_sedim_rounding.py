"""salsa_sedim_device rounds each operation of a tendency as the reference writes
it: particles that leave their level whole take exactly q / dtlt out of it, for
the number and every mass row of precipitation and ice.  (A product with 1 / dtlt
differs in the last bit for about a third of all q at dtlt = 3 s.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtlt", [3., 7.])
@pytest.mark.parametrize("cat", [2, 3])
def test_departures_are_correctly_rounded_quotients(cat, dtlt):
    import torch
    from salsa_amd import capi
    print("case sedimentation rounding, category %d, dtlt %.0f s" % (cat, dtlt), flush=True)
    desc = capi.bin_desc(species=("SO4", "DU"))
    nzp, nxp, nyp, k0, bin_ = 14, 12, 12, 9, 3
    nb = [desc.nbins, desc.ncld, desc.nprc, desc.nice]
    rows = [b * (desc.nspec - 1 + (c == 3)) for c, b in enumerate(nb)]
    rng = np.random.default_rng(cat)
    sh = (nyp, nxp, nzp)
    n = [np.zeros((b,) + sh) for b in nb]
    m = [np.zeros((r,) + sh) for r in rows]
    # particles of about a millimetre, on one level of every column: they fall faster than one 0.5 m level per second
    n[cat][bin_, :, :, k0] = 10. * (1. + rng.random(sh[:2]))
    for s in range(rows[cat] // nb[cat]):
        mass = (5e-7 if s == desc.iwa else 1e-9) * (1. + rng.random(sh[:2]))
        m[cat][s * nb[cat] + bin_, :, :, k0] = mass * n[cat][bin_, :, :, k0]
    D = lambda a: torch.from_numpy(np.ascontiguousarray(a.reshape(a.shape[0], -1) if a.ndim == 4 else a.reshape(-1))).cuda()
    dn, dm = [D(x) for x in n], [D(x) for x in m]
    dnt, dmt = [torch.zeros_like(x) for x in dn], [torch.zeros_like(x) for x in dm]
    one = np.ones(sh)
    f = dict(tk=D(270. * one), th=D(275. * one), adn=D(1.1 * one), ustar=D(0.3 * one[:, :, 0]))
    new = lambda *s: torch.zeros(s, dtype=torch.float64, device="cuda")
    n3, ncol = nzp * nxp * nyp, nxp * nyp
    ctx = capi.Context(desc, capi.params(level=5), nzp, nxp, nyp)
    ctx.sedim_device(dtlt, np.full(nzp, 2.), f, dn, dm, dnt, dmt, new(n3), new(n3), new(ncol), new(nb[2], n3),
                     sed=(1, 1, 1, 1), irate=new(n3), sfcirate=new(ncol), vt_ice=new(nb[3], n3))
    ctx.sync()
    ctx.close()
    inner = (slice(2, -2), slice(2, -2), k0)
    for q, t, r in [(n, dnt, bin_)] + [(m, dmt, s * nb[cat] + bin_) for s in range(rows[cat] // nb[cat])]:
        q0, t0 = q[cat][r][inner], t[cat].cpu().numpy()[r].reshape(sh)[inner]
        assert (q0 > 0.).all()
        np.testing.assert_array_equal(t0, -q0 / dtlt)
