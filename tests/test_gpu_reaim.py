"""A context re-aimed between runs (sources moved, receiver lists and wavelets
grown and shrunk, a tile or its geometry changed) equals a fresh one bit for
bit, with the chunks captured before kept or dropped."""
import numpy as np
import pytest

from fd23_amd import _lib
from helpers import Problem

pytestmark = pytest.mark.gpu


def aim(ctx, p, sources, rx, rz, nstf):
    for s, (xs, zs) in enumerate(sources):
        ctx.reset_shot(s)
        ctx.set_source(s, p.kind, xs, zs, p.stf[:nstf], p.M)
        for c in range(ctx.ncomp):
            ctx.set_receivers(s, c, rx, rz)


@pytest.mark.parametrize("wave,tile", [(_lib.WAVE_PSV, 0), (_lib.WAVE_PSV, 28), (_lib.WAVE_PSV, 10),
                                       (_lib.WAVE_SH, 0), (_lib.WAVE_SH, 20), (_lib.WAVE_SH, 25)])
def test_reaimed_context_equals_fresh(wave, tile):
    nx, nz, nt = 420, 150, 150
    kind = _lib.SRC_FORCE if wave == _lib.WAVE_SH else _lib.SRC_LINE
    p = Problem(wave, nx, nz, 8, 10.0, 7e-4, nt, seed=5, kind=kind, sources=[(100, 40), (200, 60)], rec_z=30)
    rng = np.random.default_rng(3)
    few = (np.array([30, 210], np.int32), np.array([70, 90], np.int32))
    # receivers and sources in the first rows move the marching step's
    # rectangle, deep ones move it back; more of them outgrow the lists
    many = (rng.integers(0, nx, p.rx.size).astype(np.int32), rng.integers(0, nz, p.rx.size).astype(np.int32))
    aims = [([(100, 40), (200, 60)], *few, 20), ([(110, 44), (390, 61)], *few, 20),
            ([(60, 10), (300, 17)], *few, 150), ([(111, 80), (222, 140)], *many, 150),
            ([(100, 40), (200, 60)], *few, 20)]

    def run(ctx):
        ctx.run(0, 129, 2)
        ctx.run(129, 21, 2)
        ctx.sync()
        return [ctx.get_state(s) for s in range(2)] + [ctx.seismograms(s, c, nt // 2).tobytes() for s in range(2)
                                                       for c in range(ctx.ncomp)]

    with p.context() as ctx:
        ctx.tile = tile
        heard = []  # a source may be out of a receiver's reach in these few steps
        for a in aims + aims[::-1]:
            aim(ctx, p, *a)
            got = run(ctx)
            with p.context() as ref:
                ref.tile = tile
                aim(ref, p, *a)
                want = run(ref)
            assert any(want[0]) and got == want
            heard += [any(b) for b in want[2:]]
        assert any(heard)
