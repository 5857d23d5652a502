"""Workgroup shapes of the batched and forward-only kernels below 128: the large workgroup at 48 for launches of
at most one position per CU against the default one, and operand staging with partly filled last rounds."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.cases import small_case
from tests.conftest import rel

pytestmark = pytest.mark.gpu

GRAD_TOL, LOSS_TOL = 1e-3, 1e-4


# 48: 300 positions take the default shape, each half of them the large one; 24, 32, 96: butterflies that do not
# fill the workgroup's threads, more positions than CUs
@pytest.mark.parametrize('n,nz,binning,npos', [(48, 5, 2, 300), (24, 3, 1, 300), (32, 3, 2, 270), (96, 2, 1, 258)])
def test_shapes_agree_and_match_oracle(n, nz, binning, npos):
    from mset_amd import lib
    c = small_case(n=n, nz=nz, binning=binning, npos=npos, seed=n, spread=n / 6)
    print('case: shapes', n, nz, binning, npos, flush=True)
    with lib.Context(0) as ctx:
        ctx.upload(c['V'], c['probe'], c['prop'], c['xl'], c['yl'], c['M'], c['sig'], c['dx'], slice_binning=c['bin'],
                   n_scan=(npos, 1))
        whole = ctx.grad()
        parts = [ctx.grad(0, npos // 2), ctx.grad(npos // 2, npos - npos // 2)]
        err = ctx.error_resident()
    oV, op, opos, oep = O.grad_fixed(c['V'], c['probe'], c['prop'], c['bprop'], c['xl'], c['yl'], c['M'], c['bin'],
                                     c['sig'], c['dx'])
    for dV, dp, dpos, e in (whole, (parts[0][0] + parts[1][0], parts[0][1] + parts[1][1],
                                    np.concatenate([parts[0][2], parts[1][2]]), parts[0][3] + parts[1][3])):
        assert rel(dV, oV) < GRAD_TOL and rel(dp, op) < GRAD_TOL and rel(dpos, opos) < GRAD_TOL
        assert abs(e / (oep.sum() / npos) - 1) < LOSS_TOL
    assert abs(err / (oep.sum() / npos) - 1) < LOSS_TOL
