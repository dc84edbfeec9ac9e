"""ckr_decode_many of small masked tensors around the unit size up to which their
set-ups share a launch (the state chains end at the 256 symbols of a 64 KiB unit):
no bad lane is counted, and the bytes are the sources'."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("unit", [32768, 65536, 65536 + 256, 131072, 262144, 1 << 20])
@pytest.mark.parametrize("sizes", [[300_001, 700_000], [2_000_001, 70_000, 5, 400_000, 33_000]])
def test_small_shards(sizes, unit, gpu):
    import torch
    import checkers_amd as ck
    g = torch.Generator(device=gpu)
    g.manual_seed(unit)
    xs, tags = [], []
    for k, n in enumerate(sizes):
        r = torch.randn(n, generator=g, device=gpu) * 0.02
        xs.append(r if k % 2 else r.to(torch.bfloat16))
        tags.append(ck.F32 if k % 2 else ck.BF16)
    encs = [ck.Encoder(x.numel(), t, unit) for x, t in zip(xs, tags)]
    coded = ck.compress_many(encs, xs)
    decs = [ck.Decoder(x.numel(), t, unit) for x, t in zip(xs, tags)]
    for check in (True, False, True):
        dsts = [torch.zeros(x.nbytes, dtype=torch.uint8, device=gpu) for x in xs]
        print("[case] decode_many", unit, sizes, check, flush=True)
        bad = ck.decode_many(decs, coded, dsts, check=check)
        torch.cuda.synchronize()
        assert bad == ([0] * len(xs) if check else None)
        assert all(torch.equal(d, x.view(torch.uint8)) for d, x in zip(dsts, xs))
