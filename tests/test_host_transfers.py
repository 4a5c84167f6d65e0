"""Host transfers and resets beside other parts of a program (no GPU: the
runtime is replaced)."""
import pytest

from hosthip import run

CALLS = """
c = context(%s, 130, 70, 2, %s, nt=300)
c.run(0, 6, 1)
def calls(c):
    for s in range(2):
        state = c.get_state(s)
        c.set_state(state, s)
        for f in (("U", "Txz") if c.wave == PSV else ("V", "Tz")):
            c.set_field(f, c.field(f, s), s)
        for k in range(c.ncomp):
            c.seismograms(s, k, 300)
        c.reset_shot(s)
    c.set_material([c.material(i) for i in range(5 if c.wave == PSV else 3)])
"""
KINDS = [("PSV", "F32"), ("PSV", "F16"), ("PSV", "F64"), ("SH", "F32"), ("SH", "BF16")]


@pytest.mark.parametrize("kind", KINDS)
def test_errors_of_others_stay_theirs(kind):
    """An error that another call has left (an allocation that failed) is neither
    reported by a transfer or a reset nor taken away."""
    run(CALLS % kind + """
hh.hh_error = 2
calls(c)
assert hh.hh_error == 2
""")


@pytest.mark.parametrize("kind", KINDS)
def test_transfers_need_no_free_memory(kind):
    """A context whose run has filled the device still gives its results."""
    run(CALLS % kind + """
hh.hh_room = 0
calls(c)
""")


@pytest.mark.parametrize("kind", KINDS)
def test_one_or_two_frames_come_in_one_call(kind):
    """Neither packed nor queued: that takes about twice as long as the runtime's
    own copy of one or two rows."""
    run(CALLS % kind + """
for n in (1, 2):
    before = hh.hh_launches, hh.hh_async
    c.seismograms(1, 0, n)
    assert (hh.hh_launches, hh.hh_async) == before, n
before = hh.hh_launches
c.seismograms(1, 0, 3)
assert hh.hh_launches == before + 1
""")
