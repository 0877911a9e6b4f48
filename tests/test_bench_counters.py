"""bench.py sets a run's times only against counters of the kernels that it
launches."""
import json

import pytest

import bench

SCHEDULE = {"stages_left": 3, "stages_right": 3, "stages_gram": 3}   # the defaults
PRODUCTS = ("whiten_left", "whiten_right", "gram")


@pytest.mark.parametrize("precision", ["fp64", "bf16x3"])
@pytest.mark.parametrize("kernel", PRODUCTS)
def test_recorded_counters_are_of_the_launched_kernels(kernel, precision):
    name = bench.product_kernel(kernel, precision, SCHEDULE)
    bytes_, src = bench.measured_traffic(kernel, precision, "desi-4096", name)
    assert src and bytes_ > 0
    busy, bsrc = bench.measured_mfma_busy(kernel, precision, "desi-4096", name)
    assert bsrc and 0 < busy < 1


def test_other_kernels_have_no_counters(tmp_path, monkeypatch):
    monkeypatch.setattr(bench, "TRAFFIC_DIR", str(tmp_path))
    (tmp_path / "traffic_gram_fp64_w.json").write_text(json.dumps({"kernel_name": "k_old", "hbm_bytes_per_launch": 1}))
    (tmp_path / "mfma_util_products_w.json").write_text(
        json.dumps({"kernel_name": {"fp64": {"gram": "k_old"}}, "mfma_busy": {"fp64": {"gram": 0.9}}}))
    assert bench.measured_traffic("gram", "fp64", "w", "k_gram64") == (None, None)
    assert bench.measured_mfma_busy("gram", "fp64", "w", "k_gram64") == (None, None)
    assert bench.measured_traffic("gram", "fp64", "w", "k_old")[0] == 1.0
    assert bench.measured_mfma_busy("gram", "fp64", "w", "k_old")[0] == 0.9


@pytest.mark.parametrize("stages,name", [(1, "k_gemm_bf3<0, 1, 3>"), (2, "k_gemm_bf3<0, 2, 3>"),
                                         (3, "k_gemm_bf3d<0, 3, 2, 3>"), (4, "k_gemm_bf3d<0, 3, 3, 3>")])
def test_names_follow_the_staging(stages, name):
    assert bench.product_kernel("whiten_left", "bf16x3", dict(SCHEDULE, stages_left=stages)) == name
