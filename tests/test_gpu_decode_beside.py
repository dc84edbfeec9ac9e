"""ckr_decode_many of shards that go job by job over several streams (an int32
tensor or a destination that is not 4-byte aligned among them): each decode takes
its share of the workgroups, from a few of a small tensor to all of a dominant one."""
import numpy as np
import pytest

from tests import datagen as dg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [
    [("bf16", 40_001), ("i32", 3), ("f32", 9)], [("bf16", 4_000_001)] * 5 + [("i32", 100_000)],
    [("f32", 5_000_003), ("i32", 777)], [("f32", 3_000_000), ("i8", 1_000_001), ("bf16", 70_000), ("i32", 1)],
    [("i8", 3_000_000), ("i8", 200_000), ("i8", 5)],
])
@pytest.mark.parametrize("check", [True, False])
def test_shards(sizes, check, gpu):
    import torch
    import checkers_amd as ck
    g = torch.Generator(device=gpu)
    g.manual_seed(len(sizes))
    make = {"bf16": lambda n: (torch.randn(n, generator=g, device=gpu) * 0.02).to(torch.bfloat16),
            "f32": lambda n: torch.randn(n, generator=g, device=gpu) * 1e-3,
            "i32": lambda n: torch.randint(0, 5000, (n,), generator=g, device=gpu, dtype=torch.int32),
            "i8": lambda n: torch.randint(-9, 9, (n,), generator=g, device=gpu, dtype=torch.int8)}
    tag = {"bf16": dg.BF16, "f32": dg.F32, "i32": dg.I32, "i8": dg.I8}
    xs = [make[t](n) for t, n in sizes]
    encs = [ck.Encoder(n, tag[t], 65536) for t, n in sizes]
    coded = ck.compress_many(encs, xs)
    decs = [ck.Decoder(n, tag[t], 65536) for t, n in sizes]
    dsts = [torch.zeros(x.nbytes + 16, dtype=torch.uint8, device=gpu) for x in xs]
    for _ in range(3):
        for d in dsts:
            d.zero_()
        bad = ck.decode_many(decs, coded, dsts, check=check)
        torch.cuda.synchronize()
        assert bad == ([0] * len(xs) if check else None)
        for x, d in zip(xs, dsts):
            assert torch.equal(d[: x.nbytes], x.view(torch.uint8)) and not d[x.nbytes:].any()
