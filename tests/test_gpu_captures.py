"""Captured sequential passes: replays give the eager pass's state bit for bit, with eager passes, error passes and
synchronisations between them, and after an eager batched pass has reallocated the scratch they share."""
import numpy as np
import pytest

from tests.cases import small_case

pytestmark = pytest.mark.gpu


# the on-chip separable kernel, line passes, and the general kernel (exact pairing)
@pytest.mark.parametrize('n,nz,mode', [(24, 16, 0), (64, 16, 0), (96, 16, 0), (128, 16, 0), (48, 16, 1), (256, 16, 0)])
def test_sequential_capture_replays_the_eager_pass(n, nz, mode):
    from mset_amd import lib
    c = small_case(n=n, nz=nz, binning=4, npos=5, seed=n, spread=n / 8)
    print('case: captured sequential pass', n, nz, mode, flush=True)

    def series():
        r = lib.Recon(c['V'], c['prop'], 2, c['sig'], c['dx'], slice_binning=4, step_size=(30.0, 2e-3, 2e-2), grad_mode=mode)
        for j, ang in enumerate(((0, 0, 0), (0, 20, 0))):
            r.set_tilt(j, ang, c['probe'], c['xl'], c['yl'], c['M'])
        return r

    plan = [(lib.PATH_PLAIN, 1)] * 4 + [(lib.PATH_BATCHED, 5)] + [(lib.PATH_PLAIN, 1)] * 3
    state = []
    for graph in (False, True):
        r = series()
        errs = []
        for path, batch in plan:
            errs.append(r.iterate(path, batch, use_graph=graph and path == lib.PATH_PLAIN))
            errs.extend(r.error_pass())
        rec, probes, xs, ys = r.get()
        state.append([np.array(errs), rec, probes] + xs + ys)
        r.close()
    for a, b in zip(*state):
        assert np.array_equal(a, b)
