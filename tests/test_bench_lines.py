"""What bench.py says about its launches follows from what the engine counted, not
from the precision alone."""
import importlib.util
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def bench():
    spec = importlib.util.spec_from_file_location("bench", os.path.join(ROOT, "bench.py"))
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


def test_launches_follow_the_counts():
    b = bench()
    two = b.launches("f64", 512, 20, 10)
    assert two == {"kernel": "plbamd::fused_two_steps (two steps)", "steps_per_launch": 2, "launches": 10,
                   "bytes_per_cell": 19 * 8}
    assert b.launches("f64", 512, 200, 99)["bytes_per_cell"] == 2 * 19 * 8 * 101 / 200
    one = b.launches("f32", 128, 20, 0)    # in the last-level cache, PLBAMD_FUSED=0, or no room for a second array
    assert one["steps_per_launch"] == 1 and one["bytes_per_cell"] == 2 * 19 * 4 and "bulk_odd_staged" in one["kernel"]
    assert "bulk_pairs" in b.launches("f16", 512, 20, 0)["kernel"]
    assert b.launches("f16", 72, 20, 9)["steps_per_launch"] == 2
    assert b.launches("bf16", 101, 20, 0)["kernel"] == "plbamd::bulk_step"


def test_traffic_is_of_the_launches_that_ran():
    b = bench()
    assert b.traffic_from_profile("f64", 512, 2) > 2e10
    assert b.traffic_from_profile("f64", 512, 1) is None
    assert b.traffic_from_profile("f64", 256, 2) is None
    assert b.traffic_from_profile("f16", 512, 1) > 1e10
