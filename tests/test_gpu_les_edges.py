"""salsa_les_update_device where its layout can go wrong: columns of the fewest
levels, of one level less and more than a wavefront's 128 and several
wavefronts, odd and even shares, domains so small that a column has several
periodic images, one and two dry species.  Bit-exact against the oracle,
as every operation is a comparison, a move or a sum in the reference's order."""
import numpy as np
import pytest

from helpers import les_case

pytestmark = pytest.mark.gpu

ALL = ("SO4", "DU")


@pytest.fixture(scope="module")
def capi():
    import torch
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    from salsa_amd import capi as c
    c.lib()
    return c


@pytest.mark.parametrize("level,grid,dry", [(4, (2, 2, 2), 1), (4, (3, 3, 2), 1), (5, (62, 2, 5), 1), (4, (63, 5, 3), 2),
                                            (4, (125, 3, 4), 1), (4, (126, 4, 4), 1), (5, (127, 2, 3), 2),
                                            (4, (253, 3, 3), 1), (4, (255, 2, 2), 1), (4, (391, 2, 2), 1)])
def test_les_update_at_its_edges(capi, oracle_mod, level, grid, dry):
    import torch
    desc = capi.bin_desc(species=ALL[:dry])
    print("case LES update, level %d, grid %s, %d dry species" % (level, grid, dry), flush=True)
    shape, dzt, f, n_p, n_t, m_p, m_t = les_case(desc, level, grid, 11)
    nzp, nxp, nyp = shape
    n3 = nzp * nxp * nyp
    ct = np.ones((desc.nbins + desc.ncld + desc.nprc, n3))
    L = oracle_mod.make_layout(species=tuple(int(capi.SPECIES[s]) for s in ALL[:dry]))
    on, ont, om, omt = ([a.copy() for a in x] for x in (n_p, n_t, m_p, m_t))
    oct_ = ct.copy()
    four = lambda x: (list(x) + [None] * 4)[:4]
    odiag = oracle_mod.les_update(L, level, shape, 1.0, dzt[nzp - 3] / dzt[nzp - 2], f["temp"], f["rh"], f["rhi"],
                                  f["rp"], four(on), four(ont), four(om), four(omt), oct_)
    dev = torch.device("cuda")
    D = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    dn, dnt, dm, dmt = ([D(a) for a in x] for x in (n_p, n_t, m_p, m_t))
    df = {k: D(v) for k, v in f.items()}
    dct = D(ct)
    ddiag = torch.zeros((6, n3), dtype=torch.float64, device=dev)
    ctx = capi.Context(desc, capi.params(level=level), nzp, nxp, nyp)
    ctx.les_update_device(1.0, dzt, df, dn, dnt, dm, dmt, ddiag, charge_time=dct)
    ctx.sync()
    ctx.close()
    for c in range(len(n_p)):
        np.testing.assert_array_equal(dn[c].cpu().numpy(), on[c], err_msg="numbers, category %d" % c)
        np.testing.assert_array_equal(dm[c].cpu().numpy(), om[c], err_msg="masses, category %d" % c)
        assert not dnt[c].any() and not dmt[c].any()
    np.testing.assert_array_equal(dct.cpu().numpy(), oct_)
    rows = 6 if level == 5 else 4
    np.testing.assert_array_equal(ddiag.cpu().numpy()[:rows], odiag[:rows])
