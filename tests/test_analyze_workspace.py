"""ckr_analyze_workspace_bytes: a workspace sized for a list of records serves
every part of the list and smaller records (host arithmetic, no GPU)."""
import random

import pytest

import checkers_amd as ck


def _bytes(recs):
    arr = (ck.StatsRecord * len(recs))()
    for r, (n, dt) in zip(arr, recs):
        r.d_ptr, r.num_elements, r.histogram_bins, r.data_type = 1 << 20, n, 256, dt
    return int(ck.lib().ckr_analyze_workspace_bytes(arr, len(recs)))


@pytest.mark.parametrize("seed", range(6))
def test_parts_and_smaller_records(seed):
    rng = random.Random(seed)
    recs = [(int(10 ** rng.uniform(0, 10.5)), rng.choice([ck.F32, ck.BF16, ck.F16, ck.I8, ck.I32]))
            for _ in range(rng.randint(2, 60))]
    whole = _bytes(recs)
    for _ in range(40):
        part = rng.sample(recs, rng.randint(1, len(recs)))
        assert _bytes(part) <= whole
        assert _bytes([(max(1, int(n * rng.random())), dt) for n, dt in recs]) <= whole


def test_small_records_beside_a_huge_one():
    small = [(15_000_000, ck.F32)] * 10
    assert _bytes(small) <= _bytes(small + [(25_000_000_000, ck.F32)])
