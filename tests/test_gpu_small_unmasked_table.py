"""Small int8 and int32 tensors whose table's correction falls inside a group of equal
fractional parts (the ranks' ambiguity, which most of them have): alone they are
counted once, in a shard counted and coded once; larger ones keep the device table."""
import numpy as np
import pytest

import oracle as oc
from tests import datagen as dg

pytestmark = pytest.mark.gpu


def _ambiguous(n, dt):
    import checkers_amd as ck
    for seed in range(200):
        rng = np.random.default_rng(seed)
        if dt in (dg.F32, dg.BF16):
            x = dg.normal_f32(n, 1e-3, seed) if dt == dg.F32 else dg.normal_bf16(n, 0.02, seed)
            b = dg.raw_bytes(x).reshape(n, -1).copy()
            b[:, : 2 if dt == dg.F32 else 1] = 0
        else:
            x = b = (np.clip(np.round(rng.standard_normal(n) * 32), -127, 127).astype(np.int8) if dt == dg.I8
                     else rng.integers(0, 5000, n).astype(np.int32))
        if ck.build_table_ranked(np.bincount(b.reshape(-1).view(np.uint8), minlength=256).astype(np.uint32))[1]:
            return x
    raise AssertionError("no ambiguous tensor found")


@pytest.mark.parametrize("n,dt", [(2100, dg.I8), (60_000, dg.I8), (262_144, dg.I8), (800, dg.I32), (65_536, dg.I32),
                                  (1000, dg.F32), (3001, dg.BF16)])
def test_counted_once(n, dt, gpu):
    import torch
    import checkers_amd as ck
    x = _ambiguous(n, dt)
    ref = oc.compress_tensor(x, n, dt, 65536)
    src = torch.from_numpy(dg.raw_bytes(x).copy()).to(gpu)
    e = ck.Encoder(n, dt, 65536)
    for _ in range(2):
        ck.profile_begin()
        enc = e.compress(src)
        torch.cuda.synchronize()
        prof = ck.profile_end()
        assert prof["hist_table_kernel"][0] == 1 and "masked_hist_kernel" not in prof
        assert enc.total == ref["data"].size and np.array_equal(enc.data_np(), ref["data"])
        assert np.array_equal(enc.headers_np()[: ref["headers"].size], ref["headers"])


def test_shard(gpu):
    import torch
    import checkers_amd as ck
    parts = [(dg.BF16, dg.normal_bf16(70_001, 0.02, 2)), (dg.I8, _ambiguous(3000, dg.I8)),
             (dg.I32, _ambiguous(5000, dg.I32)), (dg.F32, dg.normal_f32(50_000, 1e-3, 3))]
    srcs = [torch.from_numpy(dg.raw_bytes(a).copy()).to(gpu) for _, a in parts]
    encs = [ck.Encoder(a.size, dt, 65536) for dt, a in parts]
    ck.profile_begin()
    out = ck.compress_many(encs, srcs)
    torch.cuda.synchronize()
    prof = ck.profile_end()
    assert "hist_table_kernel" not in prof and prof["encode_fast_kernel"][0] == len(parts)
    for (dt, a), e in zip(parts, out):
        ref = oc.compress_tensor(a, a.size, dt, 65536)
        assert e.total == ref["data"].size and np.array_equal(e.data_np(), ref["data"])


def test_larger_ones_by_ranks(gpu):
    import torch
    import checkers_amd as ck
    src = torch.zeros(262_145, dtype=torch.int8, device=gpu)
    src[::3] = 5
    e = ck.Encoder(src.numel(), dg.I8, 65536)
    ck.profile_begin()
    enc = e.compress(src)
    torch.cuda.synchronize()
    assert "hist_table_kernel" in ck.profile_end()
    ref = oc.compress_tensor(src.cpu().numpy(), src.numel(), dg.I8, 65536)
    assert enc.total == ref["data"].size and np.array_equal(enc.data_np(), ref["data"])
