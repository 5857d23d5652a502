"""The small workgroup at 24 x 24 for launches of more positions than the default shape keeps resident: gradient,
checkpointed and recomputed waves and the forward pass against the FP64 oracle, with slabs of several positions."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.cases import small_case
from tests.conftest import rel

pytestmark = pytest.mark.gpu

GRAD_TOL, LOSS_TOL = 1e-3, 1e-4


@pytest.mark.parametrize('npos,waves', [(1700, 'STORE'), (2900, 'STORE'), (2900, 'CHECKPOINT'), (2900, 'RECOMPUTE')])
def test_many_positions_match_oracle(npos, waves):
    from mset_amd import lib
    c = small_case(n=24, nz=5, binning=1, npos=npos, seed=npos, spread=4.0)
    print('case: many positions at 24', npos, waves, flush=True)
    with lib.Context(0) as ctx:
        ctx.upload(c['V'], c['probe'], c['prop'], c['xl'], c['yl'], c['M'], c['sig'], c['dx'], slice_binning=c['bin'],
                   n_scan=(npos, 1))
        ctx.set_exit_waves(getattr(lib, 'EXIT_WAVES_' + waves))
        whole = ctx.grad()
        ctx.set_slot_limit(100)                       # another grid, the same sums
        capped = ctx.grad()
        ctx.set_slot_limit(0)
        ctx.set_engine(lib.ENGINE_GENERAL)
        err = ctx.error_resident()
    for a, b in zip(whole, capped):
        assert np.array_equal(a, b)
    dV, dp, dpos, e = whole
    oV, op, opos, oep = O.grad_fixed(c['V'], c['probe'], c['prop'], c['bprop'], c['xl'], c['yl'], c['M'], c['bin'],
                                     c['sig'], c['dx'])
    assert rel(dV, oV) < GRAD_TOL and rel(dp, op) < GRAD_TOL and rel(dpos, opos) < GRAD_TOL
    assert abs(e / (oep.sum() / npos) - 1) < LOSS_TOL and abs(err / (oep.sum() / npos) - 1) < LOSS_TOL
