"""Captured chunks a context holds (no GPU: the runtime is replaced)."""
import pytest

from hosthip import run


@pytest.mark.parametrize("held", range(10, 17))
def test_prepared_run_captures_nothing(held):
    """fd23_prepare leaves its run no capture, however many graphs of other
    lengths the context holds."""
    run("""
for wave, tile in ((PSV, 0), (SH, 20)):
    c = context(wave, 128, 96)
    c.tile = tile
    for n in range(1, %d + 1):
        c.run(0, 2 * n, 1)
    for nt in (329, 200, 128, 7, 200, 329):
        c.prepare(nt, 1)
        before = hh.hh_graphs
        c.run(0, nt, 1)
        assert hh.hh_graphs == before, (nt, hh.hh_graphs - before)
    c.close()
""" % held)


def test_graphs_are_bounded():
    run("""
c = context(PSV, 128, 96)
for n in range(1, 100):
    c.run(0, n, 1)
assert hh.hh_held <= 16, hh.hh_held
c.close()
assert hh.hh_held == 0
""")
