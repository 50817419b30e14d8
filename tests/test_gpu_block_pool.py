"""Device blocks kept between calls: given back by release, bounded, and reused without a trace of what
they held before (a large solve's blocks serve a smaller one, and the other way round)."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rmp2(ctx, s, o, v):
    from jues import _lib
    Co, Cv = _lib.f64(s.C[:, :o]), _lib.f64(s.C[:, s.o:s.o + v])
    eps, E = _lib.f64(np.concatenate([s.eps[:o], s.eps[s.o:s.o + v]])), np.zeros(1)
    ctx.check(ctx.lib.jues_rmp2(ctx.h, _lib.FP64, _lib.ptr(Co), o, _lib.ptr(Cv), v, s.n, _lib.ptr(eps), _lib.ptr(E)))
    return float(E[0])


def test_release_gives_everything_back():
    from jues import _lib, synthetic
    s = synthetic.make_system(40, 8, 32, 120, 3)
    ctx = _lib.Context(0)
    before = ctx.lib.jues_device_bytes(ctx.h)
    ctx.set_ao_factors(s.B)
    E = _rmp2(ctx, s, 8, 32)
    held = ctx.lib.jues_device_bytes(ctx.h)
    assert held > before
    assert _rmp2(ctx, s, 8, 32) == E                       # the same bits from reused blocks
    assert ctx.lib.jues_device_bytes(ctx.h) == held          # and no new ones
    ctx.release()
    assert ctx.lib.jues_device_bytes(ctx.h) == before
    ctx.set_ao_factors(s.B)
    assert _rmp2(ctx, s, 8, 32) == E
    ctx.close()


def test_sizes_in_turn_and_two_contexts_in_threads(cfg1):
    from jues import _lib, synthetic
    systems = [synthetic.make_system(n, o, n - o, 3 * n, n) for n, o in ((24, 5), (61, 10), (40, 8))]

    def energies(passes, out):
        ctx = _lib.Context(0)
        for _ in range(passes):
            for s in systems:
                ctx.set_ao_factors(s.B)
                out.append(_rmp2(ctx, s, s.o, s.v))
                out.append(_rmp2(ctx, s, s.o - 1, s.v - 3))
        ctx.close()

    ref = []
    for s in systems:                                       # each in a context of its own
        ctx = _lib.Context(0)
        ctx.set_ao_factors(s.B)
        ref.append(_rmp2(ctx, s, s.o, s.v))
        ctx.close()
        ctx = _lib.Context(0)
        ctx.set_ao_factors(s.B)
        ref.append(_rmp2(ctx, s, s.o - 1, s.v - 3))
        ctx.close()
    outs = [[], []]
    threads = [threading.Thread(target=energies, args=(3, o)) for o in outs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert outs[0] == ref * 3 and outs[1] == ref * 3
