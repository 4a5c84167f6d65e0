"""Untuned contexts run the shape picked from their size; whatever it is, a run
equals tile 0's bit for bit."""
import pytest

from fd23_amd import _lib
from helpers import Problem

pytestmark = pytest.mark.gpu

# both sides of each line of the rule (wave, nx, nz, shots, storage)
CASES = [
    (_lib.WAVE_SH, 64, 48, 1, _lib.STORE_F32), (_lib.WAVE_SH, 288, 128, 2, _lib.STORE_F32),
    (_lib.WAVE_SH, 289, 128, 2, _lib.STORE_F32), (_lib.WAVE_SH, 468, 380, 1, _lib.STORE_F64),
    (_lib.WAVE_SH, 469, 381, 1, _lib.STORE_F32), (_lib.WAVE_SH, 640, 500, 1, _lib.STORE_F16),
    (_lib.WAVE_SH, 1000, 400, 5, _lib.STORE_F32), (_lib.WAVE_SH, 1000, 400, 3, _lib.STORE_F16),
    (_lib.WAVE_PSV, 500, 300, 2, _lib.STORE_F32), (_lib.WAVE_PSV, 501, 300, 2, _lib.STORE_F32),
    (_lib.WAVE_PSV, 400, 250, 2, _lib.STORE_F16), (_lib.WAVE_PSV, 1000, 500, 10, _lib.STORE_BF16),
    (_lib.WAVE_PSV, 1000, 600, 1, _lib.STORE_F64), (_lib.WAVE_PSV, 1001, 600, 1, _lib.STORE_F64),
    (_lib.WAVE_PSV, 1250, 800, 10, _lib.STORE_F32), (_lib.WAVE_PSV, 1250, 800, 20, _lib.STORE_F16),
    (_lib.WAVE_PSV, 4100, 100, 25, _lib.STORE_F32),
]


@pytest.mark.parametrize("wave,nx,nz,shots,storage", CASES)
def test_default_shape_equals_tile_0(wave, nx, nz, shots, storage):
    kind = _lib.SRC_FORCE if wave == _lib.WAVE_SH else _lib.SRC_LINE
    srcs = [(20 + (k * (nx - 40)) // shots, 6 + 3 * (k % 5)) for k in range(shots)]
    p = Problem(wave, nx, nz, 12, 10.0, 7e-4, 13, seed=nx, kind=kind, sources=srcs, rec_z=3,
                f64=storage == _lib.STORE_F64 and wave == _lib.WAVE_PSV)
    out = []
    for tile in (None, 0):
        with p.context(storage=storage) as ctx:
            if tile is not None:
                ctx.tile = tile
            ctx.run(0, 9, 1)
            ctx.run(9, 4, 1)
            ctx.sync()
            out.append([ctx.get_state(s) for s in (0, shots - 1)] +
                       [ctx.seismograms(s, c, 13).tobytes() for s in (0, shots - 1) for c in range(ctx.ncomp)])
    assert any(any(b) for b in out[1])
    assert out[0] == out[1]
