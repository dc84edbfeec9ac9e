"""ckr_decode without a bad-lane count under graph capture: its set-up must
queue kernels only, whether or not the library's state chains exist already."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _run():
    import torch
    import checkers_amd as ck
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    x = torch.randn(100_003, generator=g, device="cuda") * 1e-3
    t, s = ck.build_table(ck.byte_histogram(x, ck.F32).cpu().numpy().view("uint32"))
    assert s == 4096
    enc = ck.encode(x, ck.F32, t, 65536)  # (no device table: the chains are not made by it)
    d = ck.Decoder(x.numel(), ck.F32, 65536)
    dst = torch.zeros(x.nbytes, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    for chains_made in (False, True):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            d.decode(enc.data, enc.headers, enc.unit_offsets, enc.table, enc.sidecar, dst, check=False)
        for _ in range(3):
            dst.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(dst, x.view(torch.uint8)), chains_made
        assert d.decode(enc.data, enc.headers, enc.unit_offsets, enc.table, enc.sidecar, dst) == 0


def test_decode_under_capture(gpu):
    """In a process of its own, where no earlier call has made the chains."""
    r = subprocess.run([sys.executable, os.path.abspath(__file__)], cwd=ROOT, timeout=100, capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr


if __name__ == "__main__":
    sys.path.insert(0, ROOT)
    _run()
