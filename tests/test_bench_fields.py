"""The bench line's roofline fields: every stage is one launch for both grids."""
import bench


def test_roofline_counts_launches_as_they_are():
    stages = {"deposit": 2.4, "z_r2c": 3.8, "y_fft": 3.0, "x_fft_bin": 2.5}
    r = bench.roofline(stages, 1024, 2, 20000000, 0.8)
    b = bench.stage_bytes(1024, 2, 20000000, 0.8)
    assert r["kernel"] == "z_r2c_kernel"
    assert r["bytes_per_launch"] == b["z_r2c"] and r["ms_per_launch"] == 3.8
    assert abs(r["achieved"] - b["z_r2c"] / 3.8e6) < 0.06
    for k, v in r["stages"].items():
        assert v["launches"] == 1
        assert abs(v["GBps"] - b[k] / (stages[k] * 1e6)) < 0.06
