"""The shape an untuned context starts on (no GPU: the runtime is replaced)."""
from hosthip import run


def test_fp64_sh_starts_on_the_passes():
    """FP64 SH contexts start on the passes, one row per thread on small grids
    and two on larger ones, never on a block shape or four rows."""
    run("""
for nx, nz, shots, rz in ((128, 128, 1, 1), (256, 128, 1, 1), (256, 128, 4, 1), (400, 200, 1, 1), (512, 256, 1, 1),
                          (800, 400, 1, 2), (1024, 512, 4, 2), (2000, 1000, 1, 2), (1400, 900, 2, 2)):
    c = Context(SH, nx, nz, 20, nshots=shots, storage=F64)
    assert c.tile_kind() == _lib.TILE_TILED and c.tile_shape()[:2] == (rz, 1), (nx, nz, shots, c.tile_shape())
    c.close()
c = Context(SH, 400, 200, 20)
assert c.tile_kind() == _lib.TILE_BLOCK
""")
