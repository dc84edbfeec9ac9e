"""ckr_encode of int8 and int32 without a total only queues work: it can be captured
into a graph and replayed."""
import numpy as np
import pytest

import oracle as oc
from tests import datagen as dg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,n,unit", [(dg.I8, 200_003, 65536), (dg.I32, 50_001, 16384), (dg.I8, 3000, 65536),
                                       (dg.I8, 400_000, 262144)])
def test_captured_encode(dt, n, unit, gpu):
    import torch
    import checkers_amd as ck
    rng = np.random.default_rng(n)
    x = (np.minimum(rng.geometric(0.1, n), 120).astype(np.int8) if dt == dg.I8
         else rng.integers(0, 50257, n).astype(np.int32))
    raw = dg.raw_bytes(x)
    h = np.bincount(raw, minlength=256).astype(np.uint32)
    t_ck, s = ck.build_table(h)
    t_oc, _ = oc.normalize_histogram(h)
    assert s == 4096
    data, hdr, off = oc.encode(raw, t_oc, unit)
    src = torch.from_numpy(raw.copy()).to(gpu)
    e = ck.Encoder(n, dt, unit)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        e.encode(src, t_ck, sync_total=False)
    for _ in range(3):
        e.out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert int(e.unit_offsets[off.size - 1].item()) == data.size
        assert np.array_equal(e.out[: data.size].cpu().numpy(), data)
        assert np.array_equal(e.headers.cpu().numpy().view(ck.HEADER_DTYPE).reshape(-1)[: hdr.size], hdr)
