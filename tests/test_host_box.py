"""The box's set-up (no GPU: the runtime is replaced)."""
from hosthip import run

BOX = """
def box(c, bx=40, incident=0, vs=1100.0, x0=20):
    c.box_configure(x0, 20, bx, 30, incident, 10.0, 8.0, 0.1, 1.0, 2000.0, vs, 2000.0, 10.0, 1e-3)
c = context(PSV, 128, 96, storage=F64)
box(c)
c.run(0, 6, 1)
"""


def test_refused_box_drops_the_captured_one():
    """A box that is refused takes the one before it away, and with it the
    graphs that name its arrays."""
    run(BOX + """
raises("SV incidence", box, c, 40, 1, 0.0)
raises("no box", c.box_residual)
before = hh.hh_graphs
c.run(0, 6, 1)
assert hh.hh_graphs == before + 1
""")


def test_same_box_again_allocates_nothing():
    """The next plane wave on a box of the same size takes over its arrays."""
    run(BOX + """
before = hh.hh_mallocs, hh.hh_room
for incident in (1, 0):
    box(c, incident=incident, x0=30)
    c.run(0, 6, 1)
    c.box_residual()
assert (hh.hh_mallocs, hh.hh_room) == before
box(c, 50)
assert hh.hh_mallocs == before[0] + 2 and hh.hh_room < before[1]
c.close()
""")
