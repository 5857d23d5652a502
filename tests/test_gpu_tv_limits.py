"""TV_method where |q|^2 leaves the float range: q / sqrt(max(1, |q|^2)) of finite q is then 0, as a division by
infinity gives, and the output stays finite."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def tv_single(f, lam, iters):
    """TV_method.m:5-84 in single precision, its operation order (dims x, y, z = axes 2, 1, 0)"""
    f = f.astype(np.float32)
    lam, tau = np.float32(lam), np.float32(1) / np.float32(12)
    P = [np.zeros_like(f) for _ in range(3)]
    ax = (2, 1, 0)

    def div():
        d = P[0] + P[1] + P[2]
        for k in range(3):
            d = d - np.roll(P[k], 1, ax[k])
        return d

    with np.errstate(over='ignore', invalid='ignore'):
        for _ in range(iters):
            D = div() - f / lam
            q = [P[k] + tau * (np.roll(D, -1, ax[k]) - D) for k in range(3)]
            den = np.sqrt(np.maximum(np.float32(1), q[0] * q[0] + q[1] * q[1] + q[2] * q[2]))
            P = [a / den for a in q]
        return f - lam * div()


# one float4 row per thread and single elements; below, across and above the square root of the float range
@pytest.mark.parametrize('nx', [8, 9])
@pytest.mark.parametrize('size', [1e15, 3e19, 1e21, 1e30])
def test_large_arguments_stay_finite(nx, size):
    from mset_amd import lib
    rng = np.random.default_rng(nx)
    v = rng.uniform(-1, 1, (5, 6, nx)).astype(np.float32)
    v[2, 3, 4] = size
    v[0, 0, 0] = -size
    print('case: tv limits', nx, size, flush=True)
    with lib.Context(0) as ctx:
        out, _ = ctx.tv(v, 1.0, 6)
    ref = tv_single(v, 1.0, 6)
    assert np.isfinite(ref).all() and np.isfinite(out).all()
    # every P is within [-1, 1], its 6 terms rounded to float32 per iteration; u adds the rounding of the voxel
    assert (np.abs(out.astype(np.float64) - ref) <= 6 * 6 * 2.0 ** -22 + 2.0 ** -22 * np.abs(ref)).all()


# rows of whole float4s and others, odd and even iteration counts
@pytest.mark.parametrize('shape,iters', [((5, 6, 8), 6), ((9, 17, 33), 11), ((16, 24, 20), 0), ((1, 1, 4), 3)])
def test_small_scratch_gives_the_same(tmp_path, shape, iters):
    """the two-launch iteration on 4 volumes of scratch against the one-launch one on 7 and TV_method"""
    from oracle import oracle as O
    from tests.conftest import rel
    from tests.fake_hip import run_failing_malloc
    v = np.random.default_rng(sum(shape)).uniform(0, 3, shape).astype(np.float32)
    np.save(tmp_path / 'v.npy', v)
    print('case: tv small scratch', shape, iters, flush=True)
    run_failing_malloc(tmp_path, '''
        v = np.load(%r)
        with lib.Context(0) as ctx:
            whole, e = ctx.tv(v, 0.25, %d)
        fail_malloc(7 * v.size * 4)
        with lib.Context(0) as ctx:
            out, e2 = ctx.tv(v, 0.25, %d)
        assert failed() == 1
        np.savez(%r, whole=whole, out=out, e=[e, e2])
    ''' % (str(tmp_path / 'v.npy'), iters, iters, str(tmp_path / 'o.npz')))
    o = np.load(tmp_path / 'o.npz')
    ref, rerr = O.tv(v, 0.25, iters)
    for u, e in ((o['whole'], o['e'][0]), (o['out'], o['e'][1])):
        assert rel(u, ref) < 1e-5 and abs(e - rerr) <= 1e-4 * abs(rerr) + 1e-5
