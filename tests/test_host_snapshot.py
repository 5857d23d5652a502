"""Snapshot and restore of a tilt series, on the CPU with a stand-in HIP runtime: tilts of different lengths, tilts
replaced in between, and snapshots that ran out of memory half way."""
import pytest

from tests import fake_hip


@pytest.fixture(scope='session')
def tmp(tmp_path_factory):
    return tmp_path_factory.mktemp('fake_hip')


def test_restore_brings_back_tilts_of_different_lengths(tmp):
    fake_hip.run(tmp, '''
        r = recon(24, 16, (5, 9, 2), angles=(0., 10., 20.))
        want = r.get()
        r.snapshot()
        for j, k in enumerate((5, 9, 2)):
            t = state(24, 16, k)
            r.set_tilt(j, (0., 0., 0.), t['probe'] * 7, t['x'] + 50, t['y'] - 50, t['M'])
        r.restore()
        got = r.get()
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        for a, b in zip(got[2] + got[3], want[2] + want[3]):
            assert np.array_equal(a, b)
    ''')


def test_restore_after_a_tilt_was_replaced(tmp):
    fake_hip.run(tmp, '''
        r = recon(24, 16, (5, 9, 2), angles=(0., 10., 20.))
        want = r.get()
        r.snapshot()
        t = state(24, 16, 4)
        r.set_tilt(1, (0., 0., 0.), t['probe'] * 7, t['x'] + 50, t['y'] - 50, t['M'])
        r.restore()                              # fewer positions: the first ones come back
        got = r.get()
        assert np.array_equal(got[1], want[1])
        for a, b, k in zip(got[2] + got[3], want[2] + want[3], (5, 4, 2) * 2):
            assert np.array_equal(a, b[:k])
        t = state(24, 16, 10)
        r.set_tilt(1, (0., 0., 0.), t['probe'] * 7, t['x'] + 50, t['y'] - 50, t['M'])
        before = r.get()
        try:
            r.restore()
            raise SystemExit('a tilt with more positions than the snapshot was restored')
        except lib.MsetError as e:
            assert e.code == lib.MSET_EINVAL
        for a, b in zip(before[2] + before[3], (lambda g: g[2] + g[3])(r.get())):
            assert np.array_equal(a, b)
    ''')


# the sizes of the three blocks of a snapshot: volume, probes, positions (x and y of 5 + 9 + 2)
@pytest.mark.parametrize('nbytes', [24 * 24 * 16 * 4, 3 * 24 * 24 * 8, 2 * 16 * 4])
@pytest.mark.parametrize('earlier', [False, True])
def test_no_restore_from_a_snapshot_that_failed(tmp, nbytes, earlier):
    fake_hip.run(tmp, '''
        r = recon(24, 16, (5, 9, 2), angles=(0., 10., 20.))
        if %r:                                   # one of fewer positions, whose buffers are too small for the next
            t = state(24, 16, 3)
            r.set_tilt(1, (0., 0., 0.), t['probe'], t['x'], t['y'], t['M'])
            r.snapshot()
            t = state(24, 16, 9)
            r.set_tilt(1, (0., 0., 0.), t['probe'], t['x'], t['y'], t['M'])
        fake.fake_fail_malloc(%d)
        try:
            r.snapshot()
            failed = False
        except lib.MsetError as e:
            assert e.code == lib.MSET_ENOMEM
            failed = True
        fake.fake_fail_malloc(0)
        try:
            r.restore()
            assert not failed
        except lib.MsetError as e:
            assert failed and e.code == lib.MSET_EINVAL
        r.snapshot()
        r.restore()
    ''' % (earlier, nbytes))
