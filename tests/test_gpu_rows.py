"""Pitched transfers between host arrays and the context's device arrays:
rows are packed on the device and cross the host link in chunks, with the
storage type's conversion on the device.  What comes back is the value the
storage holds, bit for bit."""
import numpy as np
import pytest

from fd23_amd import _lib
from fd23_amd.core import Context

pytestmark = pytest.mark.gpu

# odd widths, one row block, widths over a workgroup, and grids whose fields
# take more than one 4 MiB chunk (with a remainder)
GRIDS = [(16, 16), (63, 17), (257, 40), (1501, 1203)]


def stored(v, storage, scale):
    """The value the storage holds, in the compute type."""
    if storage == _lib.STORE_F16:
        return (v / np.float32(scale)).astype(np.float16).astype(np.float32) * np.float32(scale)
    if storage == _lib.STORE_BF16:
        torch = pytest.importorskip("torch")
        b = torch.from_numpy(v / np.float32(scale)).to(torch.bfloat16).to(torch.float32).numpy()
        return b * np.float32(scale)
    return v


@pytest.mark.parametrize("storage", [_lib.STORE_F32, _lib.STORE_F64, _lib.STORE_F16, _lib.STORE_BF16])
@pytest.mark.parametrize("nx,nz", GRIDS)
def test_fields_state_and_material_come_back(nx, nz, storage):
    rng = np.random.default_rng(nx + 7 * storage)
    npml, shots = 5, 2
    with Context(_lib.WAVE_PSV, nx, nz, npml, nshots=shots, storage=storage) as ctx:
        scale = 1.0
        if storage in (_lib.STORE_F16, _lib.STORE_BF16):
            scale = 2.0 ** -7
            ctx.set_scales(np.full(13, scale, np.float32))
        names = ("U", "W", "Txx", "Txz", "Tzz")
        vals = {}
        for s in range(shots):
            for n in names:
                v = rng.standard_normal((nz, nx)).astype(ctx.cdtype)
                v[0, :3] = (0.0, -0.0, 1e-9)  # zeros and a value below FP16's subnormals
                vals[s, n] = v
                ctx.set_field(n, v, shot=s)
        for s in range(shots):
            for n in names:
                want = stored(vals[s, n], storage, scale)
                assert np.array_equal(ctx.field(n, shot=s), want), (s, n)
        # the checkpoint of shot 1 put into shot 0
        data = ctx.get_state(1)
        flat = np.frombuffer(data, ctx.cdtype)
        assert np.array_equal(flat[:nx * nz].reshape(nz, nx), stored(vals[1, "U"], storage, scale))
        ctx.set_state(data, 0)
        assert ctx.get_state(0) == data
        mat = [rng.random((nz, nx)).astype(ctx.cdtype) for _ in range(5)]
        ctx.set_material(mat)
        for i, m in enumerate(mat):
            assert np.array_equal(ctx.material(i), m), i


@pytest.mark.parametrize("nrec,max_rec,frames", [(1, 1, 3), (5, 9, 7), (300, 700, 2000)])
def test_seismograms_are_the_recorded_velocities(nrec, max_rec, frames):
    """Frames of one shot out of a frame-major buffer of two: a field set by
    hand and recorded through the staged entry point."""
    nx, nz = 64, 48
    rng = np.random.default_rng(nrec)
    with Context(_lib.WAVE_SH, nx, nz, 4, nshots=2, max_frames=frames, max_rec=max_rec) as ctx:
        rx, rz = rng.integers(0, nx, nrec).astype(np.int32), rng.integers(0, nz, nrec).astype(np.int32)
        for s in range(2):
            ctx.set_receivers(s, 0, rx, rz)
        want = {}
        for f in (0, frames // 2, frames - 1):
            for s in range(2):
                v = rng.standard_normal((nz, nx)).astype(np.float32)
                ctx.set_field("V", v, shot=s)
                want[s, f] = v[rz, rx]
            ctx.record(f, 1)
        for s in range(2):
            got = ctx.seismograms(s, 0, frames)
            for f in (0, frames // 2, frames - 1):
                assert np.array_equal(got[f], want[s, f]), (s, f)
            assert np.count_nonzero(np.abs(got).sum(axis=1)) == len({0, frames // 2, frames - 1})


@pytest.mark.parametrize("nx,nz,npml", [(16, 16, 0), (63, 17, 5), (300, 130, 12)])
@pytest.mark.parametrize("storage", [_lib.STORE_F32, _lib.STORE_F64, _lib.STORE_F16])
def test_reset_zeroes_one_shot_alone(nx, nz, npml, storage):
    rng = np.random.default_rng(nx)
    with Context(_lib.WAVE_PSV, nx, nz, npml, nshots=3, storage=storage, max_frames=4, max_rec=3) as ctx:
        if storage == _lib.STORE_F16:
            ctx.set_scales(np.ones(13, np.float32))
        n = ctx.state_bytes() // np.dtype(ctx.cdtype).itemsize
        data = [rng.integers(-9, 9, n).astype(ctx.cdtype).tobytes() for _ in range(3)]
        for s in range(3):
            ctx.set_state(data[s], s)
            for c in range(2):
                ctx.set_receivers(s, c, np.array([1, 2, 3], np.int32), np.array([4, 5, 6], np.int32))
        for f in range(4):
            ctx.record(f, 1)
        seis = [[ctx.seismograms(s, c, 4) for c in range(2)] for s in range(3)]
        ctx.reset_shot(1)
        assert not np.frombuffer(ctx.get_state(1), np.uint8).any()
        assert not any(ctx.seismograms(1, c, 4).any() for c in range(2))
        for s in (0, 2):
            assert ctx.get_state(s) == data[s]
            for c in range(2):
                assert np.array_equal(ctx.seismograms(s, c, 4), seis[s][c])
