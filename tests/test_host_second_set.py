"""A context that needs a second buffer set where there is no room for it (no
GPU: the runtime is replaced)."""
from hosthip import run


def test_untuned_context_goes_on_in_place():
    """The default shape falls back to the passes; a shape that the caller set
    is refused, before and after."""
    run("""
for wave, nx, nz, shots, storage in ((PSV, 1250, 800, 10, F32), (PSV, 1250, 800, 20, F16), (SH, 1400, 900, 3, F32),
                                     (SH, 256, 128, 1, F32)):
    for call in ("run", "prepare", "time"):
        c = context(wave, nx, nz, shots, storage)
        first = c.tile
        assert c.tile_kind() != _lib.TILE_TILED
        room, hh.hh_room = hh.hh_room, (4 << 20 if nx > 500 else 1 << 18)
        if call == "run":
            c.run(0, 5, 1)
        elif call == "prepare":
            c.prepare(5, 1)
        else:
            c.time_passes(1)
        assert c.tile_kind() == _lib.TILE_TILED and not c.tile_split(), c.tile_shape()
        c.run(5, 6, 1)
        c.seismograms(0, 0, 6)
        c.tile = first
        raises("-2", c.run, 0, 4, 1)
        assert c.tile == first
        hh.hh_room = room
        c.run(0, 4, 1)
        c.close()
""")


def test_tuning_reports_the_missing_room():
    run("""
c = context(SH, 256, 128)
room, hh.hh_room = hh.hh_room, 1 << 20
first = c.tile
raises("-2", c.autotune, 2)
assert c.tile == first
hh.hh_room = 1 << 18
c.run(0, 5, 1)
assert c.tile_kind() == _lib.TILE_TILED
""")
