"""What bench.py's line says of a context set to the marching shape (no GPU: the
runtime is replaced, a timed interval takes 1 ms)."""
import pytest

from hosthip import run


@pytest.mark.parametrize("wave", ["PSV", "SH"])
def test_line_of_the_marching_step(wave):
    run("""
import bench
wl = bench.make_workload("sh400" if %s == SH else "psv2000").build()
c = wl.context(max_frames=8)
c.tile = 28
want = c.bytes_per_step()
r = bench.measure_line(wl, 4, 4, tile=28)
assert r["roofline"]["kernel"] == "march" and "march" in r["roofline"]["kernel_name"][0], r
assert r["roofline"]["stress_ms"] is None and r["roofline"]["velocity_ms"] is None
# 20 launches in 1 ms
assert abs(r["roofline"]["kernel_ms"] - 1 / 20) < 1e-4, r["roofline"]
assert abs(r["bytes_per_step"] - want) < 1e-6 * want, (r["bytes_per_step"], want)
""" % wave)


def test_line_of_passes_on_the_marching_shape():
    """FP64 storage runs the two passes there."""
    run("""
import bench
wl = bench.make_workload("sh400", "f64").build()
c = wl.context(max_frames=8)
c.tile = 28
want = c.bytes_per_step()
r = bench.measure_line(wl, 4, 4, tile=28)
assert r["roofline"]["kernel"] == "stress" and r["roofline"]["kernel_name"] == ["fd23::k_sh_stress<double, 4, 1, false>"], r
assert abs(r["bytes_per_step"] - want) < 1e-6 * want
""")
