"""int8 and int32 units whose lanes outgrow the fast encoder's slots are coded
again by the fast encoder (one slot set that holds any lane), not by the general
kernels: near-uniform bytes that share a table with zero planes, foreign tables
with escapes, minimal slots (mode 3), ragged ends, single tensors and shards."""
import numpy as np
import pytest

import oracle as oc
from tests import datagen as dg

pytestmark = pytest.mark.gpu


def _ids(n, seed):
    return np.random.default_rng(seed).integers(0, 50257, n).astype(np.int32)


def _same(enc, data, hdr, off):
    nu = off.size - 1
    assert enc.total == data.size and np.array_equal(enc.data_np(), data)
    assert np.array_equal(enc.headers_np()[: nu * 256], hdr)
    assert np.array_equal(enc.unit_offsets[: nu + 1].cpu().numpy().view(np.uint64), off)


def _profiled(ck, f):
    import torch
    ck.profile_begin()
    r = f()
    torch.cuda.synchronize()
    return r, ck.profile_end()


def _assert_fast_redo(prof):
    assert "encode_fast_redo_kernel" in prof
    assert "encode_kernel" not in prof and "compact_kernel" not in prof


@pytest.mark.parametrize("n,unit", [(300_000, 65536), (16384 * 3 + 1, 65536), (16384 - 64, 65536), (2_000_003, 65536),
                                    (70_001, 49152)])
def test_ids(n, unit, gpu):
    import torch
    import checkers_amd as ck
    x = _ids(n, n)
    ref = oc.compress_tensor(x, n, dg.I32, unit)
    assert int(ref["headers"]["byte_count"].max()) > (288 if unit == 65536 else 200)
    src = torch.from_numpy(x.copy()).to(gpu)
    e = ck.Encoder(n, dg.I32, unit)
    for _ in range(3):
        enc, prof = _profiled(ck, lambda: e.compress(src))
        _same(enc, ref["data"], ref["headers"], ref["unit_offsets"])
    if unit == 65536:
        _assert_fast_redo(prof)
    dst, bad = ck.decode(enc)
    torch.cuda.synchronize()
    assert bad == 0 and np.array_equal(dst.cpu().numpy(), dg.raw_bytes(x))


def test_shard(gpu):
    import torch
    import checkers_amd as ck
    xs = [_ids(n, n) for n in (100_000, 250_001, 70_000)] + [np.zeros(5000, np.int32)]
    encs = [ck.Encoder(x.size, dg.I32, 65536) for x in xs]
    srcs = [torch.from_numpy(x.copy()).to(gpu) for x in xs]
    out, prof = _profiled(ck, lambda: ck.compress_many(encs, srcs))
    _assert_fast_redo(prof)
    for x, e in zip(xs, out):
        ref = oc.compress_tensor(x, x.size, dg.I32, 65536)
        _same(e, ref["data"], ref["headers"], ref["unit_offsets"])


@pytest.mark.parametrize("mode", [1, 3])
@pytest.mark.parametrize("dt", [dg.I8, dg.I32])
def test_foreign_table_with_escapes(dt, mode, gpu):
    """Rare symbols at 12 bits and symbols without a slot (raw-byte escapes)."""
    import torch
    import checkers_amd as ck
    rng = np.random.default_rng(11)
    raw = np.minimum(rng.geometric(0.2, 65536 * 5 + 1028), 39).astype(np.uint8)
    m = raw[: raw.size // 256 * 256].reshape(-1, 256)
    m[256:512, 40:90] = rng.integers(40, 60, (256, 50), dtype=np.uint8)  # 50 lanes of unit 1: over 10 bits a symbol
    m[600:700, 7] = rng.integers(60, 250, 100, dtype=np.uint8)           # no slot: raw bytes
    h = np.bincount(np.minimum(rng.geometric(0.2, 1 << 20), 59), minlength=256).astype(np.uint32)
    h[40:60] = 600
    t_ck, s = ck.build_table(h)
    t_oc, s_oc = oc.normalize_histogram(h)
    assert s == s_oc == 4096
    data, hdr, off = oc.encode(raw, t_oc, 65536)
    e = ck.Encoder(raw.size // (4 if dt == dg.I32 else 1), dt, 65536)
    src = torch.from_numpy(raw.copy()).to(gpu)
    old = ck.set_fast_paths(mode)
    try:
        enc, prof = _profiled(ck, lambda: e.encode(src, t_ck))
    finally:
        ck.set_fast_paths(old)
    _same(enc, data, hdr, off)
    assert (hdr["byte_count"][256 + 40: 256 + 90] > 288).all() and off[2] - off[1] < 65536
    _assert_fast_redo(prof)
