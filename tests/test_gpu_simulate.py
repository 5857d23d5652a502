"""mset_simulate: intensities and their centring against the FP64 oracle, every size and both routines; many positions
per workgroup."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.cases import small_case
from tests.conftest import rel

pytestmark = pytest.mark.gpu

WAVE_TOL = 1e-4                    # on amplitudes; an intensity has twice that


@pytest.mark.parametrize('n', [16, 24, 32, 48, 64, 96, 128, 256])
@pytest.mark.parametrize('nz,binning,engine', [(5, 2, 'AUTO'), (1, 1, 'AUTO'), (4, 1, 'GENERAL')])
def test_intensities_vs_oracle(n, nz, binning, engine):
    from mset_amd import lib
    c = small_case(n=n, nz=nz, binning=binning, npos=3, seed=n + nz, spread=n / 8)
    print('case: simulate', n, nz, binning, engine, flush=True)
    with lib.Context(0) as ctx:
        ctx.upload(c['V'], c['probe'], c['prop'], c['xl'], c['yl'], c['M'], c['sig'], c['dx'], slice_binning=binning,
                   n_scan=(3, 1))
        ctx.set_engine(getattr(lib, 'ENGINE_' + engine))
        I = ctx.simulate()
        ctx.set_slot_limit(1)                    # one workgroup takes them in turn
        one = ctx.simulate()
    assert np.array_equal(I, one)
    for k in range(3):
        psi0 = O.subpixel_shift(c['probe'], c['xl'][k], c['yl'][k])
        exit_wave = O.forward(c['V'], psi0, c['prop'], c['M'][k], binning, c['sig'], c['dx'])[0][-1]
        assert rel(I[k], np.fft.fftshift(np.abs(np.fft.fft2(exit_wave)) ** 2)) < 2 * WAVE_TOL
