"""Sequential path as line passes over the device (line_passes.hip) against the FP64 oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.cases import small_case
from tests.conftest import rel
from tests.test_gpu_parity import GRAD_TOL, LOSS_TOL, assert_update_close

pytestmark = pytest.mark.gpu


# every plane size; odd and even plane counts (the orientation of the exit pass), one plane, a bin above the
# four slices kept in registers, partial last bins, and each step alone (launches left out)
@pytest.mark.parametrize('n,nz,binning,steps', [
    (64, 1, 1, (30.0, 2e-3, 2e-2)), (64, 13, 6, (30.0, 2e-3, 2e-2)), (96, 1, 1, (30.0, 2e-3, 2e-2)),
    (128, 13, 6, (30.0, 2e-3, 2e-2)), (96, 8, 4, (30.0, 2e-3, 2e-2)),
    (96, 5, 3, (30.0, 0.0, 2e-2)), (128, 11, 5, (30.0, 2e-3, 0.0)), (128, 6, 2, (0.0, 0.0, 0.0)),
    (256, 3, 2, (30.0, 2e-3, 2e-2)), (256, 2, 2, (0.0, 2e-3, 2e-2))])
def test_line_passes_vs_oracle(n, nz, binning, steps):
    from mset_amd import lib
    c = small_case(n=n, nz=nz, binning=binning, npos=4, seed=7 * n + nz, spread=n / 8)
    print('case: line passes', n, nz, binning, steps, flush=True)
    with lib.Context(0) as ctx:
        ctx.upload(c['V'], c['probe'], c['prop'], c['xl'], c['yl'], c['M'], c['sig'], c['dx'], slice_binning=c['bin'],
                   step_size=steps, n_scan=(c['npos'], 1))
        V, pr, xl, yl, err = ctx.run()
        # the general routine on the same state
        ctx.set_state(c['V'], c['probe'], c['xl'], c['yl'])
        ctx.set_engine(lib.ENGINE_GENERAL)
        gV, gpr, gxl, gyl, gerr = ctx.run()
    oV, opr, oxl, oyl, oerr, _ = O.run_tilt(c['V'], c['probe'], c['prop'], c['bprop'], c['xl'], c['yl'], c['M'],
                                            c['npos'], 1, c['bin'], c['sig'], c['dx'], steps)
    assert abs(err / oerr - 1) < LOSS_TOL
    for new, onew, old in ((V, oV, c['V']), (pr, opr, c['probe']), (xl, oxl, c['xl']), (yl, oyl, c['yl'])):
        assert_update_close(new, onew, old, c['npos'])
    # two FP32 routines, each within GRAD_TOL of the oracle's update
    assert abs(err / gerr - 1) < 2 * LOSS_TOL
    for new, gnew, old in ((V, gV, c['V']), (pr, gpr, c['probe']), (xl, gxl, c['xl']), (yl, gyl, c['yl'])):
        assert_update_close(new, gnew, old, 2 * c['npos'], 2 * GRAD_TOL)
    if not any(steps):
        assert np.array_equal(V, c['V'].astype(np.float32)) and rel(pr, c['probe']) < 1e-6
