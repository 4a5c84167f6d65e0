"""The residual kernels of the box on boxes that don't fill their 32 x 8 tiles:
against the oracle's box loop (FP64, 1e-10 relative L2, the bound of the other
box tests), and runs in chunks, which add the velocities' ring at the end of
the step before, against staged steps, which don't, bit for bit."""
import numpy as np
import pytest

import test_gpu_box as B

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("x0,z0,bx,bz", [(4, 4, 16, 16), (60, 50, 33, 41), (90, 61, 32, 24), (50, 30, 97, 23)])
def test_box_of_any_size(monkeypatch, x0, z0, bx, bz):
    monkeypatch.setattr(B, "BOX", dict(x0=x0, z0=z0, bx=bx, bz=bz))
    nt = 140
    rx = np.arange(2, B.NX - 2, 3, dtype=np.int32)
    rz = np.full(rx.size, 25, np.int32)
    mat, packed, wave = B._setup(True, 0, 20.0)
    sim, box, u, w = B._oracle(mat, packed, wave, True, nt, rx, rz)
    names = ("U", "W", "Txx", "Tzz", "Txz")
    got = []
    for staged in (False, True):
        with B._gpu(mat, packed, wave, True, 0 if not staged else nt, rx, rz, staged) as ctx:
            if not staged:
                ctx.run(0, 1)
                ctx.run(1, 130)
                ctx.run(131, 9)
                ctx.sync()
            got.append({n: (ctx.box_residual()[n], ctx.field(n)) for n in names})
    for n in names:
        kind = ("U", "W") if n in "UW" else names[2:]
        scale = max(np.linalg.norm(box.r[k]) for k in kind)
        assert scale > 0
        for a, b, o in zip(got[0][n], got[1][n], (box.r[n], getattr(sim, n))):
            assert np.array_equal(a, b), n
            assert np.linalg.norm(a - o) < 1e-10 * scale, n
