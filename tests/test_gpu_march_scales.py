"""16-bit storage between staged entry points and the marching step: a run that
follows a stress half that has changed the scales reads them as they are."""
import numpy as np
import pytest

from fd23_amd import _lib
from helpers import Problem
from test_gpu_march import march_tile

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", [_lib.STORE_F16, _lib.STORE_BF16])
def test_run_after_a_stress_half(storage):
    p = Problem(_lib.WAVE_PSV, 300, 160, 8, 10.0, 7e-4, 40, seed=3, sources=[(120, 70)], rec_z=60)
    out = []
    for tile in (0, march_tile()):
        with p.context(storage=storage) as ctx:
            ctx.tile = tile
            ctx.run(0, 0, 1)  # the scales from the sources
            before = ctx.get_scales(13)[0] / np.float32(2 ** 12)
            ctx.set_scales(before)  # the next check raises them
            ctx.run(0, 8, 1)
            ctx.step_stress()
            after = ctx.get_scales(13)[0]
            assert (after[2:5] > before[2:5]).any(), (before, after)
            ctx.run(8, 12, 1)
            ctx.sync()
            out.append([ctx.get_state(0), ctx.seismograms(0, 0, 20).tobytes(), after.tobytes()])
    assert np.isfinite(np.frombuffer(out[0][0], np.float32)).all()
    assert out[0] == out[1]
