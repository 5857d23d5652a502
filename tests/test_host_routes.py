"""Which routine every call takes, by plane size and engine flags, as include/mset.h states it: on the CPU with a
stand-in HIP runtime."""
import pytest

from tests import fake_hip

SIZES = (16, 24, 32, 48, 64, 96, 128, 256)


@pytest.fixture(scope='session')
def tmp(tmp_path_factory):
    return tmp_path_factory.mktemp('fake_hip')


# separable: the propagator factors; exact: the exact pairing; waves: how the batched calls keep them
@pytest.mark.parametrize('separable', [True, False])
@pytest.mark.parametrize('exact', [False, True])
@pytest.mark.parametrize('waves', ['STORE', 'CHECKPOINT', 'RECOMPUTE'])
def test_routes(tmp, separable, exact, waves):
    fake_hip.run(tmp, '''
        separable, exact, waves = %r, %r, %r

        def kernels(call):
            fake.fake_reset()
            call()
            return {row[0].replace('(anonymous namespace)::', '').split('(')[0].replace('void mset::', '') for row in launches()
                    if any(k in row[0] for k in ('k_sep_', 'k_line_pass', 'k_batch<', 'k_fwd<', 'k_plain<'))}

        def routine(names):
            """sep or gen: what the position kernels of a call are"""
            kinds = set()
            for k in names:
                args = k[k.index('<') + 1:-1].split(', ') if '<' in k else []
                if k.startswith(('k_sep_', 'k_line_pass')):
                    kinds.add('sep')
                elif k.startswith('k_batch'):
                    kinds.add('sep' if args[3] == 'true' else 'gen')     # N, shape, waves, SEP, PFAC
                elif k.startswith('k_fwd'):
                    kinds.add('sep' if args[3] == 'true' else 'gen')     # N, shape, tilts, SEP
                else:
                    kinds.add('gen')
            assert len(kinds) == 1, names
            return kinds.pop()

        for n in %r:
            ctx = lib.Context(0)
            upload(ctx, n, 8, 3, mode=lib.GRAD_EXACT if exact else lib.GRAD_REF, separable=separable)
            ctx.set_exit_waves(getattr(lib, 'EXIT_WAVES_' + waves))
            for engine in (lib.ENGINE_AUTO, lib.ENGINE_GENERAL, lib.ENGINE_ALT_SHAPE,
                           lib.ENGINE_ALT_SHAPE | lib.ENGINE_GENERAL):
                ctx.set_engine(engine)
                alt, sep = bool(engine & lib.ENGINE_ALT_SHAPE), separable and not engine & lib.ENGINE_GENERAL
                want = dict(
                    fwd=sep, plain=sep and not exact,
                    update=sep and not exact and ((n < 128 and waves == 'STORE' and not alt) or (n == 256 and waves != 'RECOMPUTE')),
                    grad=sep and not exact and n == 256 and waves != 'RECOMPUTE', sset=False)
                calls = dict(fwd=ctx.error_resident, plain=ctx.run_resident, update=lambda: ctx.run_batched(2), grad=ctx.grad,
                             sset=lambda: (ctx.error_resident(lib.METHOD_SSET), ctx.run_resident(lib.METHOD_SSET),
                                           ctx.run_batched(2, lib.METHOD_SSET)))
                for name, call in calls.items():
                    got = routine(kernels(call))
                    assert got == ('sep' if want[name] else 'gen'), (n, engine, name, got)
            ctx.close()
    ''' % (separable, exact, waves, SIZES))
