"""int8 and int32 in short units: which coder and decoder take them, on both sides
of the rules (rows per unit, units per tensor), bytes and headers against the
oracle's."""
import numpy as np
import pytest

import oracle as oc
from tests import datagen as dg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [dg.I8, dg.I32])
@pytest.mark.parametrize("unit,units,fast_enc,fast_dec", [
    (256, 40, False, False), (256, 3000, False, False), (1024, 300, False, False), (1792, 90, False, False),
    (2048, 512, True, False), (2048, 513, False, False), (2816, 100, True, False), (3072, 100, True, True),
    (4096, 1024, True, True), (4096, 1025, False, True), (7936, 1985, False, True), (8192, 2100, True, True),
    (65536, 0, True, False), (1024, 0, True, False), (768, 0, False, False),  # one unit of a few bytes
])
def test_routes(dt, unit, units, fast_enc, fast_dec, gpu):
    import torch
    import checkers_amd as ck
    nb = max(units - 1, 0) * unit + (unit // 2 + 4 if units else min(unit, 1252))
    rng = np.random.default_rng(units)
    raw = np.minimum(rng.geometric(0.1, nb), 255).astype(np.uint8)
    n = nb // (4 if dt == dg.I32 else 1)
    ref = oc.compress_tensor(raw.view(np.int32 if dt == dg.I32 else np.int8), n, dt, unit)
    src = torch.from_numpy(raw.copy()).to(gpu)
    e = ck.Encoder(n, dt, unit)
    ck.profile_begin()
    enc = e.compress(src)
    torch.cuda.synchronize()
    prof = ck.profile_end()
    assert ("encode_fast_kernel" in prof) == fast_enc and ("encode_kernel" in prof) != fast_enc
    assert enc.total == ref["data"].size and np.array_equal(enc.data_np(), ref["data"])
    nu = ref["unit_offsets"].size - 1
    assert np.array_equal(enc.headers_np()[: nu * 256], ref["headers"])
    d = ck.Decoder(n, dt, unit)
    dst = torch.zeros(nb, dtype=torch.uint8, device=gpu)
    ck.profile_begin()
    bad = d.decode(enc.data, enc.headers, enc.unit_offsets, enc.table, None, dst)
    prof = ck.profile_end()
    assert ("decode_fast_kernel" in prof) == fast_dec and ("decode_kernel" in prof) != fast_dec
    assert bad == 0 and torch.equal(dst, src)
