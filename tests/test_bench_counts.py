"""bench.py's count of the gridder's LDS adds: two words a cell in FP64 mode, one in FP32C."""
import ast
import inspect


def test_fp32c_counts_one_add_a_cell():
    import bench
    prof = {"grid_tiles": (4.0, 2)}
    assert bench.lds_atomics(1000, 7, prof)["algorithmic_atomics"] == 2 * 49 * 1000
    one = bench.lds_atomics(1000, 7, prof, per_cell=1)
    assert one["algorithmic_atomics"] == 49 * 1000
    assert one["achieved"] == 49 * 1000 / 2e-3 / 1e9
    calls = [c for c in ast.walk(ast.parse(inspect.getsource(bench.bench_fp32c)))
             if isinstance(c, ast.Call) and getattr(c.func, "id", "") == "lds_atomics"]
    assert len(calls) == 1 and [k.value.value for k in calls[0].keywords
                                if k.arg == "per_cell"] == [1]
