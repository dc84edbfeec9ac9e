"""Decode of units above 1 MiB on both sides of its rule: at most one unit per
CU (the kernel with the shorter chain) and more (three blocks per CU), and
lanes that take the most stream bytes a symbol can (two)."""
import numpy as np
import pytest

import oracle as oc
from tests import datagen as dg

pytestmark = pytest.mark.gpu

UNIT = (1 << 20) + 256


@pytest.mark.parametrize("units", [256, 257])  # an MI355X has 256 CUs
def test_unit_counts_around_one_per_cu(units, gpu):
    import torch
    import checkers_amd as ck
    n = (units - 1) * (UNIT // 2) + 5001  # a ragged last unit
    g = torch.Generator(device=gpu)
    g.manual_seed(units)
    x = (torch.randn(n, generator=g, device=gpu) * 0.02).to(torch.bfloat16)
    enc = ck.compress(x, ck.BF16, UNIT)
    assert enc.n_units == units
    dst, bad = ck.decode(enc)
    torch.cuda.synchronize()
    assert bad == 0 and torch.equal(dst, x.view(torch.uint8))


@pytest.mark.parametrize("dt", [dg.F32, dg.BF16])
def test_lanes_of_rare_symbols(dt, gpu):
    """Columns whose live bytes are all rare symbols (a few slots each: 10 to 12 bits a
    symbol) beside columns of one common
    symbol (a fraction of a bit): the widest spread of ring positions."""
    import torch
    import checkers_amd as ck
    es = 4 if dt == dg.F32 else 2
    rows = (5 << 20) // 256 + 13
    rng = np.random.default_rng(7)
    b = np.full((rows, 256), 0x3C, np.uint8)
    b[:, 4 * 9:4 * 9 + 8] = rng.integers(0, 30, (rows, 8), dtype=np.uint8)
    raw = b.reshape(-1)[: (rows * 256 - 6 * es)].copy()
    n = raw.size // es
    raw = raw.view(np.uint32 if es == 4 else np.uint16)
    ref = oc.compress_tensor(raw, n, dt, 0)
    src = torch.from_numpy(dg.raw_bytes(raw).copy()).to(gpu)
    enc = ck.compress(src, dt, 0, n_elems=n)
    torch.cuda.synchronize()
    assert enc.total == ref["data"].size and np.array_equal(enc.data_np(), ref["data"])
    dst, bad = ck.decode(enc)
    torch.cuda.synchronize()
    assert bad == 0 and np.array_equal(dst.cpu().numpy(), dg.raw_bytes(raw))


def test_more_units_than_cus_fp32_with_raw_units(gpu):
    """Above one unit per CU (decode_long_kernel), fp32, under a table made for other
    data: units of its frequent bytes are coded, units of rare ones (12 bits each,
    beside zero planes at 5) are stored raw, the ragged last one among them."""
    import torch
    import checkers_amd as ck
    units = 259
    n = (units - 1) * (UNIT // 4) + 70_003
    h = np.full(256, 1, np.uint32)
    h[0] = 128
    h[0x30:0x40] = 232
    t, s = ck.build_table(h)
    assert s == 4096
    g = torch.Generator(device=gpu)
    g.manual_seed(5)
    b = torch.randint(0, 256, (n, 4), generator=g, device=gpu, dtype=torch.uint8)
    cheap = torch.randint(0x30, 0x40, (n, 2), generator=g, device=gpu, dtype=torch.uint8)
    raw_unit = torch.arange(n, device=gpu) // (UNIT // 4) % 3 == 0  # (unit 258 is one)
    b[:, 2:] = torch.where(raw_unit[:, None], (b[:, 2:] & 63) + 0x80, cheap)
    src = b.reshape(-1)
    e = ck.Encoder(n, ck.F32, UNIT)
    enc = e.encode(src, t)
    torch.cuda.synchronize()
    off = enc.unit_offsets[: units + 1].cpu().numpy()
    size = np.diff(off)
    length = np.full(units, UNIT)
    length[-1] = n * 4 - (units - 1) * UNIT
    assert (size[::3] == length[::3]).all() and (size[1::3] < UNIT).all() and (size[2::3] < UNIT).all()
    d = ck.Decoder(n, ck.F32, UNIT)
    dst = torch.zeros(n * 4, dtype=torch.uint8, device=gpu)
    ck.profile_begin()
    bad = d.decode(enc.data, enc.headers, enc.unit_offsets, enc.table, enc.sidecar, dst)
    prof = ck.profile_end()
    assert "decode_long_kernel" in prof and "decode_chain_kernel" not in prof
    assert bad == 0 and torch.equal(dst, src)
