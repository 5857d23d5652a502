"""The object step V += s1 G in one rounding, on every route that takes it, and the same for every slice of a bin."""
import numpy as np
import pytest

from tests.cases import small_case

pytestmark = pytest.mark.gpu

# (n, nz, bin): single slices, partial last bins, more slices per bin than are loaded together
SHAPES = [(24, 7, 3), (64, 5, 2), (32, 21, 20), (96, 6, 4), (128, 5, 3), (256, 4, 2)]


@pytest.mark.parametrize('n,nz,binning', SHAPES)
@pytest.mark.parametrize('route', ['sequential', 'sequential general', 'sequential single slice', 'batched',
                                   'batched general', 'batched single slice'])
def test_step_is_one_rounding(n, nz, binning, route):
    from mset_amd import lib
    c = small_case(n=n, nz=nz, binning=binning, npos=1, seed=n + nz, spread=n / 8)
    V = c['V'].astype(np.float32)
    bins = nz if 'single' in route else binning
    V[::bins] = 0.0                          # the first slice of a bin holds s1 G alone after a step
    print('case: object step', n, nz, binning, route, flush=True)
    out = []
    with lib.Context(0) as ctx:
        for _ in range(2):
            # first G itself, then a step of the size of V (most of its roundings show)
            s1 = np.float32(0.37 * np.abs(V).max() / np.abs(out[0][::bins]).max()) if out else np.float32(1.0)
            ctx.upload(V, c['probe'], c['prop'], c['xl'], c['yl'], c['M'], c['sig'], c['dx'], slice_binning=c['bin'],
                       step_size=(s1, 0.0, 0.0), n_scan=(1, 1))
            ctx.set_engine(lib.ENGINE_GENERAL if 'general' in route else lib.ENGINE_AUTO)
            m = lib.METHOD_SSET if 'single' in route else lib.METHOD_MSET
            if 'batched' in route:
                ctx.run_batched(1, method=m)
            else:
                ctx.run_resident(m)
            out.append(ctx.download()[0])
    G = np.repeat(out[0][::bins], bins, axis=0)[:nz]
    assert np.abs(G).max() > 0
    # a product of two floats and its sum with a third, rounded once (long double holds the product exactly)
    want = (V.astype(np.longdouble) + np.longdouble(s1) * G.astype(np.longdouble)).astype(np.float32)
    assert np.array_equal(out[1], want)
