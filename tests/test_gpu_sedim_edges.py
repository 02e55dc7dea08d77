"""salsa_sedim_device on columns around its wavefronts' edges (the fewest
levels, one less and one more than a wavefront, full workgroups) with falls of
one and of several levels; the bars are those of the other sedimentation tests, 1e-10 of each
quantity's scale."""
import numpy as np
import pytest

from test_gpu_sedim import _compare, _compare5, capi  # noqa: F401
from test_oracle_sedim import sed_fields, sed_fields5

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz,dtlt", [(2, 1.), (61, 9.), (62, 9.), (63, 9.), (126, 1.), (127, 30.), (254, 5.)])
@pytest.mark.parametrize("level,dry", [(4, 1), (5, 2)])
def test_sedim_column_edges(capi, oracle_mod, level, dry, nz, dtlt):  # noqa: F811
    desc = capi.bin_desc(species=("SO4", "DU")[:dry])
    make, check = (sed_fields, _compare) if level == 4 else (sed_fields5, _compare5)
    shape, dzt, fld, n_p, m_p, n_t, m_t = make(desc, (nz, 5, 4), 31)
    dzt = np.full_like(dzt, 1. / 20.)
    print("case sedimentation level %d, %d dry, grid %s, dtlt %.0f s" % (level, dry, shape, dtlt), flush=True)
    check(capi, oracle_mod, desc, shape, dzt, fld, n_p, m_p, n_t, m_t, 31, (1,) * (level - 1), dtlt)
