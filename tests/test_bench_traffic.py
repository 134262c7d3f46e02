"""The recorded traffic that bench.py prints beside the level-0 smoother's rate is
that of the kernel it times: 7 coefficients, r, x and the result of a quarter
of 257^3 points a launch, and what a launch reads of the other rows' x besides."""
import json
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_record_is_of_the_timed_kernel():
    rec = json.load(open(os.path.join(ROOT, "profiles", "traffic_gs_pair_f32_257.json")))
    assert rec["kernel"].startswith("k_gs_pair<float, false, true>")
    least = 40 * 257 ** 3 / 4
    whole_x = 4 * 257 ** 3
    assert least <= rec["hbm_bytes_per_launch"] <= 1.1 * (least + whole_x)
    assert os.path.exists(os.path.join(ROOT, rec["source"]))
