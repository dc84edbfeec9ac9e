"""Decodes of tensors whose unit counts lie around the number of CUs and of
resident waves, with full and ragged last units: every unit is decoded once,
whichever wave takes it.  Bytes: the decode equals the input.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

UNIT = 4096


@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "int8"])
@pytest.mark.parametrize("units", [1, 2, 255, 256, 257, 1025, 2047, 2049, 4100])
@pytest.mark.parametrize("cut", [0, 4, UNIT - 4])
def test_unit_counts(gpu, dtype, units, cut):
    import torch

    import checkers_amd as ck
    n_bytes = units * UNIT - cut
    rng = np.random.default_rng(units + cut)
    if dtype == "float32":
        raw = rng.normal(0, 1e-3, n_bytes // 4).astype(np.float32).view(np.uint8)
    elif dtype == "bfloat16":
        raw = (rng.normal(0, 0.02, n_bytes // 2).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16).view(np.uint8)
    else:
        raw = np.clip(np.rint(rng.normal(0, 20, n_bytes)), -127, 127).astype(np.int8).view(np.uint8)
    x = torch.from_numpy(raw.copy()).to(gpu).view(getattr(torch, dtype))
    enc = ck.compress(x, {"float32": ck.F32, "bfloat16": ck.BF16, "int8": ck.I8}[dtype], UNIT)
    dst, bad = ck.decode(enc)
    torch.cuda.synchronize()
    assert bad == 0 and torch.equal(dst, x.view(torch.uint8))
