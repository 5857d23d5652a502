"""Captured update passes and the buffers they hold, on the CPU with a stand-in HIP runtime: a pass captured before a
buffer of its was reallocated is captured again and never replayed."""
import pytest

from tests import fake_hip


@pytest.fixture(scope='session')
def tmp(tmp_path_factory):
    return tmp_path_factory.mktemp('fake_hip')


# sequential kernels in the three routes (line passes, on-chip separable kernel, 256), then batched ones
@pytest.mark.parametrize('n,nz', [(24, 16), (64, 16), (128, 16), (256, 16)])
def test_eager_pass_that_grows_buffers_drops_the_capture(tmp, n, nz):
    fake_hip.run(tmp, '''
        r = recon(%d, %d, 6)
        P, B = lib.PATH_PLAIN, lib.PATH_BATCHED
        r.iterate(P, 1, use_graph=True)          # captured after its eager pass
        r.iterate(P, 1, use_graph=True)
        assert (fake.fake_captures(), fake.fake_replays(), fake.fake_stale_replays()) == (1, 1, 0)
        r.iterate(B, 4, use_graph=False)         # several positions per launch: larger scratch
        r.iterate(P, 1, use_graph=True)
        r.iterate(P, 1, use_graph=True)
        assert fake.fake_stale_replays() == 0
        assert (fake.fake_captures(), fake.fake_replays()) == (2, 2)
    ''' % (n, nz))


def test_sequential_pass_that_grows_the_waves_of_a_captured_batched_one(tmp):
    fake_hip.run(tmp, '''
        r = recon(64, 48, 1)
        r.set_exit_waves(lib.EXIT_WAVES_CHECKPOINT)  # fewer planes of waves than the sequential path's L + 2
        P, B = lib.PATH_PLAIN, lib.PATH_BATCHED
        r.iterate(B, 1, use_graph=True)
        r.iterate(P, 1, use_graph=False)
        r.iterate(B, 1, use_graph=True)
        assert fake.fake_stale_replays() == 0
    ''')


def test_passes_that_grow_nothing_keep_the_capture(tmp):
    fake_hip.run(tmp, '''
        r = recon(64, 16, 6)
        r.iterate(lib.PATH_BATCHED, 4, use_graph=True)
        for _ in range(3):
            r.iterate(lib.PATH_PLAIN, 1, use_graph=False)
            r.iterate(lib.PATH_BATCHED, 4, use_graph=False)
            r.iterate(lib.PATH_BATCHED, 4, use_graph=True)
        r.error_pass()
        r.iterate(lib.PATH_BATCHED, 4, use_graph=True)
        assert fake.fake_stale_replays() == 0 and fake.fake_replays() >= 1
        n = fake.fake_captures()
        r.iterate(lib.PATH_BATCHED, 4, use_graph=True)
        assert fake.fake_captures() == n
    ''')


# 3 launches per position below 96 x 96, 2 L + 6 from there on
@pytest.mark.parametrize('n,nz,limit', [(16, 16, 65536 // 3), (96, 256, 65536 // 518)])
def test_long_sequential_passes_are_issued_eagerly(tmp, n, nz, limit):
    """a graph is asked for on both sides of the limit; the launches of a pass are the same"""
    fake_hip.run(tmp, '''
        n, nz, limit = %d, %d, %d
        counts = []
        for npos in (limit, limit + 1):
            r = recon(n, nz, npos, angles=(0.,))
            fake.fake_reset()
            r.iterate(lib.PATH_PLAIN, 1, use_graph=True)
            first = [row[:4] for row in launches() if not row[4]]
            counts.append(len([row for row in first if 'position' in row[0] or 'plain' in row[0] or 'line_pass' in row[0]
                               or 'trans' in row[0]]))
            assert fake.fake_captures() == (npos == limit), npos
            fake.fake_reset()
            r.iterate(lib.PATH_PLAIN, 1, use_graph=True)
            assert fake.fake_replays() == (npos == limit)
            if npos > limit:
                assert [row[:4] for row in launches()] == first
            r.close()
        assert 0.6 * 65536 < counts[0] <= 65536, counts        # the estimate is at least the launches
    ''' % (n, nz, limit))


def test_profiled_passes_are_issued_eagerly(tmp):
    fake_hip.run(tmp, '''
        r = recon(64, 16, 4)
        r.iterate(lib.PATH_BATCHED, 4, use_graph=True)
        r.profile(True)
        r.iterate(lib.PATH_BATCHED, 4, use_graph=True)
        assert (fake.fake_captures(), fake.fake_replays()) == (1, 0)
        assert r.profile_read('position_batch')[0] == 2
        r.profile(False)
        r.iterate(lib.PATH_BATCHED, 4, use_graph=True)
        assert (fake.fake_captures(), fake.fake_replays()) == (2, 0)
    ''')
