"""A mini-batch update and mset_grad at the same state, which below 128 come from different routines: they agree with
each other and with the FP64 oracle, also where a position's terms cancel (patterns that the state nearly explains)."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.cases import small_case

pytestmark = pytest.mark.gpu

GRAD_TOL = 1e-3


def _terms(c):
    G, P, D, _ = O.grad_fixed(c['V'], c['probe'], c['prop'], c['bprop'], c['xl'], c['yl'], c['M'], c['bin'], c['sig'], c['dx'])
    return np.repeat(G, c['bin'], axis=0)[:c['nz']], P, D


@pytest.mark.parametrize('n', [16, 24, 32, 48, 64, 96, 128])
@pytest.mark.parametrize('cancelling', [False, True])
def test_update_agrees_with_grad(n, cancelling):
    from mset_amd import lib
    c = small_case(n=n, nz=5, binning=2, npos=6, seed=3 * n, spread=n / 8)
    print('case: update and grad', n, cancelling, flush=True)
    full = _terms(c)                             # residuals of the size of the amplitudes
    if cancelling:
        moved = c['xl'] + 0.02
        c['M'] = np.stack([np.fft.fftshift(np.abs(np.fft.fft2(
            O.forward(c['V'], O.subpixel_shift(c['probe'], moved[k], c['yl'][k]), c['prop'], c['M'][k], c['bin'], c['sig'],
                      c['dx'])[0][-1])) ** 2) for k in range(c['npos'])]).astype(np.float32)
    want = _terms(c)
    if cancelling:
        assert all(np.linalg.norm(w) < 0.3 * np.linalg.norm(f) for w, f in zip(want, full))
    # steps so large that the update is all that is left of the state
    steps = [float(1e8 / np.abs(t).max()) for t in want]
    with lib.Context(0) as ctx:
        ctx.upload(c['V'], c['probe'], c['prop'], c['xl'], c['yl'], c['M'], c['sig'], c['dx'], slice_binning=c['bin'],
                   step_size=steps, n_scan=(c['npos'], 1))
        dV, dp, dpos, _ = ctx.grad()
        ctx.run_batched(c['npos'])
        V, pr, xl, yl = ctx.download()
    grad = (np.repeat(dV, c['bin'], axis=0)[:c['nz']], dp, dpos)
    upd = ((V.astype(np.float64) - c['V']) / steps[0], (c['probe'] - pr.astype(np.complex128)) / steps[1],
           np.stack([xl - c['xl'].astype(np.float64), yl - c['yl'].astype(np.float64)], 1) / steps[2])
    for g, u, w, f in zip(grad, upd, want, full):
        # amplitudes are right to a few 1e-6, and so are the terms relative to those of full residuals
        bound = GRAD_TOL * np.linalg.norm(w) + 2e-5 * np.linalg.norm(f)
        err = [np.linalg.norm(np.ravel(x)) for x in (g - w, u - w, g - u)]
        print('  ', [e / np.linalg.norm(w) for e in err], np.linalg.norm(w) / np.linalg.norm(f), flush=True)
        assert max(err) < bound
