"""The statistics pass over record lists whose grids differ: one block per
record, records of many blocks beside tiny ones, more records than one
descriptor launch carries, calls repeated on the same workspace (the blocks'
counters start over), against fp64 and exact counts."""
import numpy as np
import pytest

import oracle as oc
from tests import datagen as dg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [
    [1], [8191, 8192, 8193], [5_000_001, 3, 40_000], [100 + 37 * k for k in range(97)], [9_000_000] * 2 + [1] * 45,
])
def test_record_lists(sizes, gpu):
    import torch
    import checkers_amd as ck
    rng = np.random.default_rng(len(sizes))
    xs = [(rng.standard_normal(n) * 0.1 + 0.05).astype(np.float32) for n in sizes]
    ts = [torch.from_numpy(x).to(gpu) for x in xs]
    a = ck.Analyzer(ts, [ck.F32] * len(ts), 256)
    a.run()
    first = a.results()
    for _ in range(3):
        a.run()
    for x, r, f in zip(xs, a.results(), first):
        ref = oc.tensor_stats(dg.raw_bytes(x), x.size, dg.F32, 256)
        hist, mm, mom64 = ref["histogram"], ref["minmax"], ref["moments64"]
        assert np.array_equal(r["histogram"], hist) and np.array_equal(r["minmax"], mm)
        assert abs(r["moments"][0] - mom64[0]) <= 1e-6 * max(float(mm[1] - mm[0]), 1e-30)
        assert abs(r["moments"][1] - mom64[1]) <= 1e-4 * abs(mom64[1]) + 1e-30
        for k in r:
            assert np.array_equal(r[k], f[k])
