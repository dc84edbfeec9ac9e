"""One or two large records beside the smallest: the statistics pass with four
loads in flight per thread (few blocks of long shares) and with two, on both sides
of that rule, against exact counts and fp64 moments."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,dtype", [
    ([33_554_432 + 5], "float32"), ([33_550_000], "float32"), ([67_108_864 * 2 + 3], "bfloat16"),
    ([34_000_001, 33_999_999], "float32"), ([40_000_000, 5, 5], "float32"), ([9_000_000, 70_000_000], "bfloat16"),
    ([134_300_000] + [77] * 900, "float32"), ([140_000_001], "int8"), ([33_600_003], "int32"),
])
def test_long_shares(sizes, dtype, gpu):
    import torch
    import checkers_amd as ck
    dt = getattr(torch, dtype)
    tag = {"float32": ck.F32, "bfloat16": ck.BF16, "int8": ck.I8, "int32": ck.I32}[dtype]
    g = torch.Generator(device=gpu)
    g.manual_seed(len(sizes))
    scale = 0.1 if dt.is_floating_point else 30.0
    xs = [(torch.randn(n, generator=g, device=gpu) * scale + scale / 2).to(dt) for n in sizes]
    a = ck.Analyzer(xs, [tag] * len(xs), 256)
    for _ in range(2):
        a.run()
    for x, r in zip(xs, a.results()):
        d = x.double()
        assert int(r["histogram"].astype("int64").sum()) == x.numel()
        assert r["minmax"][0] == x.min().float().item() and r["minmax"][1] == x.max().float().item()
        mean, var = d.mean().item(), d.var(unbiased=False).item()
        # fp32 values of fp64 sums over fp32 powers of at most 4 to 8 terms each
        span = float(r["minmax"][1] - r["minmax"][0])
        assert abs(r["moments"][0] - mean) <= 1e-6 * max(span, abs(mean))
        assert abs(r["moments"][1] - var) <= 1e-5 * var + 1e-30
        del d
