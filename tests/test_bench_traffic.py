"""The benchmark's measured HBM traffic is of the kernel it names."""
import bench

PMC = """## mtgp32_items_kernel<351,8,1,4,1> (generation launch)
traffic_kernel: mtgp32_items_kernel<351,8,1,4,1>
traffic_bytes_per_launch: 123456
"""


def test_traffic_of_the_kernel_that_ran(tmp_path):
    path = tmp_path / "pmc.txt"
    path.write_text(PMC)
    assert bench.measured_traffic("mtgp32_items_kernel<351,8,1,4,1>", str(path)) == 123456
    for other in ("mtgp32_items_kernel<351,3,1,1,4>", "", None):
        assert bench.measured_traffic(other, str(path)) is None
    path.write_text("traffic_bytes_per_launch: 123456\n")  # of an unnamed kernel
    assert bench.measured_traffic("mtgp32_items_kernel<351,8,1,4,1>", str(path)) is None
    assert bench.measured_traffic("mtgp32_items_kernel<351,8,1,4,1>", str(tmp_path / "none")) is None


def test_the_committed_summary_names_its_kernel():
    assert bench.measured_traffic("mtgp32_items_kernel<351,8,1,4,1>") > 18666339120
