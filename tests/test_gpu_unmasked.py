"""int8 and int32 tensors on the fast encoder and decoder (four live lanes per
column): ragged ends, units whose lanes outgrow their slots, units stored raw,
tables with escapes, and a shard that mixes them with masked dtypes, against the
oracle."""
import numpy as np
import pytest

import oracle as oc
from tests import datagen as dg

pytestmark = pytest.mark.gpu


def _bytes(n, seed, hot=None):
    """n skewed bytes (about 3 bits each), uniform random in units [a, b) of 64 KiB."""
    rng = np.random.default_rng(seed)
    x = np.minimum(rng.geometric(0.2, n), 255).astype(np.uint8)
    if hot:
        a, b = hot[0] * 65536, min(hot[1] * 65536, n)
        x[a:b] = rng.integers(0, 256, b - a, dtype=np.uint8)
    return x


def _check(enc, ref, raw, ck):
    import torch
    assert enc.total == ref["data"].size
    nu = ref["unit_offsets"].size - 1
    assert np.array_equal(enc.unit_offsets[: nu + 1].cpu().numpy().view(np.uint64), ref["unit_offsets"])
    assert np.array_equal(enc.headers_np()[: nu * 256], ref["headers"])
    assert np.array_equal(enc.data_np(), ref["data"])
    dst, bad = ck.decode(enc)
    torch.cuda.synchronize()
    assert bad == 0 and np.array_equal(dst.cpu().numpy(), raw)


@pytest.mark.parametrize("dt,nbytes,unit,hot", [
    (dg.I8, 1, 65536, None), (dg.I8, 3, 65536, None), (dg.I8, 2 * 65536 - 1, 65536, None),
    (dg.I8, 65536 + 258, 65536, None), (dg.I8, 3 * 16384 + 255, 16384, None), (dg.I8, 65536 * 2 + 511, 65536, None),
    (dg.I32, 4, 65536, None), (dg.I32, 65536 * 2 + 252, 65536, None), (dg.I32, 65536 * 3 + 260, 32768, None),
    (dg.I8, 65536 * 9 + 777, 65536, (3, 5)),      # two units of random bytes: stored raw or coded again
    (dg.I8, 65536 * 40 + 13, 65536, (0, 4)),
    (dg.I8, 262144 * 2 + 1001, 262144, None),     # above 64 KiB: general encoder, fast decoder
])
def test_edges(dt, nbytes, unit, hot, gpu):
    import torch
    import checkers_amd as ck
    raw = _bytes(nbytes, nbytes % 97, hot)
    n = nbytes // (4 if dt == dg.I32 else 1)
    arr = raw.view(np.int32 if dt == dg.I32 else np.int8)
    ref = oc.compress_tensor(arr, n, dt, unit)
    enc = ck.compress(torch.from_numpy(raw.copy()).to(gpu), dt, unit, n_elems=n)
    _check(enc, ref, raw, ck)


def test_lanes_above_their_slots(gpu):
    """A table priced for other data: every lane of the random units needs about
    12 bits a symbol, more than its slot holds, yet the unit's other lanes keep
    it below its length, so that it is coded again and not stored raw."""
    import torch
    import checkers_amd as ck
    raw = _bytes(65536 * 6, 5)
    m = raw.reshape(-1, 256)
    rng = np.random.default_rng(9)
    m[256 * 2: 256 * 3, 40:90] = rng.integers(120, 150, (256, 50), dtype=np.uint8)  # rare symbols in 50 lanes of unit 2
    h = np.bincount(_bytes(1 << 20, 6), minlength=256).astype(np.uint32)
    h[:100] = np.maximum(h[:100], 300)
    h[100:120] = 0
    h[120:150] = 300
    h[150:] = 0
    assert raw.max() < 150 and not ((raw >= 100) & (raw < 120)).any()
    t_ck, s = ck.build_table(h)
    t_oc, s_oc = oc.normalize_histogram(h)
    assert s == s_oc == 4096
    data, hdr, off = oc.encode(raw, t_oc, 65536)
    assert off[3] - off[2] < 65536
    assert (hdr[2 * 256 + 40: 2 * 256 + 90]["byte_count"] > 320).all()  # above the largest slot
    enc = ck.encode(torch.from_numpy(raw.copy()).to(gpu), dg.I8, t_ck, 65536, n_elems=raw.size)
    torch.cuda.synchronize()
    assert enc.total == data.size and np.array_equal(enc.data_np(), data)
    assert np.array_equal(enc.headers_np()[: hdr.size], hdr)
    dst, bad = ck.decode(enc)
    torch.cuda.synchronize()
    assert bad == 0 and np.array_equal(dst.cpu().numpy(), raw)


def test_shard_with_masked_and_unmasked_tensors(gpu):
    import torch
    import checkers_amd as ck
    rng = np.random.default_rng(3)
    parts = [(dg.I8, _bytes(300_001, 1).view(np.int8)), (dg.BF16, dg.normal_bf16(70_001, 0.02, 2)),
             (dg.I32, rng.integers(0, 5000, 40_000).astype(np.int32)), (dg.F32, dg.normal_f32(50_000, 1e-3, 3)),
             (dg.I8, _bytes(255, 4).view(np.int8))]
    srcs = [torch.from_numpy(dg.raw_bytes(a).copy()).to(gpu) for _, a in parts]
    encs = [ck.Encoder(a.size, dt, 65536) for dt, a in parts]
    out = ck.compress_many(encs, srcs)
    for (dt, a), e in zip(parts, out):
        _check(e, oc.compress_tensor(a, a.size, dt, 65536), dg.raw_bytes(a), ck)
    decs = [ck.Decoder(a.size, dt, 65536) for dt, a in parts]
    dsts = [torch.zeros(s.numel() + 16, dtype=torch.uint8, device=gpu) for s in srcs]
    assert ck.decode_many(decs, out, dsts) == [0] * len(parts)
    for s, d in zip(srcs, dsts):
        assert torch.equal(d[: s.numel()], s)


def test_corrupt_streams_are_counted(gpu):
    import torch
    import checkers_amd as ck
    raw = _bytes(65536 * 3 + 100, 8)
    enc = ck.compress(torch.from_numpy(raw.copy()).to(gpu), dg.I8, 65536)
    hdr = enc.headers_np()
    torch.cuda.synchronize()
    for lane in (5, 256 + 6, 2 * 256 + 255):  # a byte in the middle of three lanes of three units
        u = lane // 256
        at = int(enc.unit_offsets[u].item()) + int(hdr[lane]["buf_offset"]) + int(hdr[lane]["byte_count"]) // 2
        enc.data[at] ^= 0x55
    dst, bad = ck.decode(enc)
    torch.cuda.synchronize()
    assert bad == 3
