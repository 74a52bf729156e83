"""The autotuner against the library's built-in shape, on the CPU: it is chosen unless
another is clearly faster, and then no entry is kept."""
import json

from rick_amd import FP32, autotune


def result(tile, rpt, ms, unroll=0):
    return {"tile": list(tile), "rows_per_task": rpt, "unroll": unroll, "ms": ms}


def test_builtin_shape_is_kept_unless_clearly_beaten():
    builtin, a, b = result((0, 0), 0, 1.0), result((64, 64), 4096, 0.95), result((64, 32), 1024, 0.9)
    assert autotune.choose([a, builtin]) is builtin
    assert autotune.choose([a, builtin, b]) is b
    assert autotune.choose([a, b]) is b             # without the built-in one, the fastest


def test_builtin_shape_takes_a_stored_entry_out(tmp_path):
    path = tmp_path / "tuning.json"
    key = autotune.signature(1024, 8, 7, FP32, 100_000)
    autotune.store(key, result((64, 64), 4096, 1.0, 7), path)
    assert autotune.lookup(1024, 8, 7, FP32, 100_000, path) == ((64, 64), 4096, 7)
    autotune.store(key, result((0, 0), 0, 0.9), path)
    assert autotune.lookup(1024, 8, 7, FP32, 100_000, path) is None
    assert json.loads(path.read_text()) == {}
    autotune.store(key, result((0, 0), 0, 0.9), path)    # and again, with nothing stored
