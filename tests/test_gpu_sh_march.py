"""The marching SH step (two steps per launch over the grid's interior, the two
passes on the frame around it) against the two-pass loop: the same arithmetic
per cell, so states and seismograms are equal bit for bit."""
import numpy as np
import pytest

from fd23_amd import _lib
from helpers import Problem
from test_gpu_march import GRIDS, OWN, march_tile, rectangle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [_lib.SRC_FORCE, _lib.SRC_LINE, _lib.SRC_P])
@pytest.mark.parametrize("nx,nz,npml,top,shots", GRIDS + [(640, 400, 20, False, 1)])
def test_sh_march_equals_two_passes(nx, nz, npml, top, shots, kind):
    x0, x1, z0, z1 = rectangle(nx, nz, npml, top)
    rng = np.random.default_rng(nx + nz)
    spots = [(x0, z0), (x1 - 1, z1 - 1), (min(x0 + OWN, nx - npml - 2), (z0 + z1) // 2), (x0 - 1, z0 - 1),
             (nx // 2, 6 + (npml if top else 0)), (x0 + 1, z0 + 17)]
    srcs = [spots[k % len(spots)] for k in range(shots)]
    p = Problem(_lib.WAVE_SH, nx, nz, npml, 10.0, 7e-4, 180, seed=nx, topabsorb=top, kind=kind, sources=srcs,
                rec_z=npml + 3 if top else 2)
    p.rx = np.concatenate([p.rx, [x0 - 1, x0, x1 - 1, 0, nx - 1], rng.integers(0, nx, 600)]).astype(np.int32)
    p.rz = np.concatenate([p.rz, [z0, z0 - 1, z1 - 1, nz - 1, 0], rng.integers(0, nz, 300),
                           np.full(300, (z0 + z1) // 2)]).astype(np.int32)

    def run(tile):
        with p.context() as ctx:
            ctx.tile = tile
            ctx.run(0, 131, 3)
            ctx.run(131, 1, 3)
            ctx.run(132, 27, 3)
            ctx.step_stress()
            ctx.inject(159)
            ctx.step_velocity()
            ctx.record(159, 3)
            ctx.run(160, 20, 3)
            ctx.sync()
            return [ctx.get_state(s) for s in range(shots)], [ctx.seismograms(s, 0, 60) for s in range(shots)]

    want, got = run(0), run(march_tile())
    assert any(np.abs(x).max() > 0 for x in want[1])
    for s in range(shots):
        assert want[0][s] == got[0][s], s
        assert np.array_equal(want[1][s], got[1][s]), s


@pytest.mark.parametrize("storage", [_lib.STORE_F16, _lib.STORE_BF16, _lib.STORE_F64])
def test_sh_march_leaves_other_storage_to_the_passes(storage):
    p = Problem(_lib.WAVE_SH, 300, 160, 8, 10.0, 7e-4, 40, seed=2, kind=_lib.SRC_FORCE, sources=[(90, 60)], rec_z=50)
    out = []
    for tile in (0, march_tile()):
        with p.context(storage=storage) as ctx:
            ctx.tile = tile
            ctx.run(0, 40, 1)
            ctx.sync()
            out.append((ctx.get_state(0), ctx.seismograms(0, 0, 40).tobytes()))
    assert out[0] == out[1]


@pytest.mark.parametrize("nx,nz,shots", [(1400, 800, 3), (1400, 900, 3), (512, 256, 28)])
def test_default_shape_of_large_sh_equals_tile_0(nx, nz, shots):
    """Both sides of the rule that starts untuned contexts on the marching step."""
    srcs = [(20 + (k * (nx - 40)) // shots, 6 + 90 * (k % 2)) for k in range(shots)]
    p = Problem(_lib.WAVE_SH, nx, nz, 12, 10.0, 7e-4, 13, seed=nx, kind=_lib.SRC_FORCE, sources=srcs, rec_z=3)
    out = []
    for tile in (None, 0):
        with p.context() as ctx:
            if tile is not None:
                ctx.tile = tile
            else:
                assert (ctx.tile == march_tile()) == (nz == 900)
            ctx.run(0, 13, 1)
            ctx.sync()
            out.append([ctx.get_state(s) + ctx.seismograms(s, 0, 13).tobytes() for s in (0, shots - 1)])
    assert out[0] == out[1]
