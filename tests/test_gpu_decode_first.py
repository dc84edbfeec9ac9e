"""The first decode of a process: without a bad-lane count it queues its work and
returns (no allocation, no wait for the stream's earlier work); with one it makes
the library's state chains."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _run():
    import threading
    import time

    import torch
    import checkers_amd as ck
    x = torch.randn(100_003, device="cuda") * 1e-3
    t, s = ck.build_table(ck.byte_histogram(x, ck.F32).cpu().numpy().view("uint32"))
    assert s == 4096
    enc = ck.encode(x, ck.F32, t, 65536)  # (under a given table: makes no chains)
    d = ck.Decoder(x.numel(), ck.F32, 65536)
    dst = torch.zeros(x.nbytes, dtype=torch.uint8, device="cuda")
    args = (enc.data, enc.headers, enc.unit_offsets, enc.table, enc.sidecar, dst)

    # the decoder's kernels loaded, by the route that uses no chains
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        d.decode(*args, check=False)
    g.replay()
    torch.cuda.synchronize()
    assert torch.equal(dst, x.view(torch.uint8))
    dst.zero_()
    big = torch.ones(1 << 30, device="cuda")
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    for _ in range(200):  # some 2 ms each
        big.mul_(1.0)
    before = torch.cuda.Event()
    before.record()
    d.decode(*args, check=False)
    pending = not before.query()
    torch.cuda.synchronize()
    assert pending, "the call waited for the stream's earlier work"
    assert torch.cuda.mem_get_info()[0] == free, "the call allocated"
    assert torch.equal(dst, x.view(torch.uint8))

    # a counting decode on another thread makes the chains behind long work; one on
    # this thread and another stream neither waits for that nor uses them
    i8 = ck.compress(torch.ones(1000, dtype=torch.int8, device="cuda"), ck.I8, 256)
    dst.zero_()
    out2 = torch.zeros_like(dst)
    d2 = ck.Decoder(x.numel(), ck.F32, 65536)
    busy, other, bad = torch.cuda.Stream(), torch.cuda.Stream(), []
    assert ck.decode(i8)[1] == 0  # (this thread's read-back buffer, by a dtype without chains)
    torch.cuda.synchronize()
    with torch.cuda.stream(busy):
        for _ in range(200):
            big.mul_(1.0)
        before = torch.cuda.Event()
        before.record()
    free = torch.cuda.mem_get_info()[0]
    th = threading.Thread(target=lambda: bad.append(d.decode(*args, stream=busy)), daemon=True)
    th.start()
    while torch.cuda.mem_get_info()[0] == free and not before.query():
        time.sleep(0.001)
    made_early = not before.query()
    assert d2.decode(*args[:-1], out2, stream=other) == 0
    waited = before.query()
    th.join(30)
    assert made_early and not waited, "a call waited for another stream's work"
    torch.cuda.synchronize()
    assert bad == [0] and torch.equal(dst, x.view(torch.uint8)) and torch.equal(out2, x.view(torch.uint8))
    for _ in range(3):
        dst.zero_()
        assert d.decode(*args) == 0 and torch.equal(dst, x.view(torch.uint8))


def test_first_decode(gpu):
    """In a process of its own, where no earlier call has made the chains."""
    r = subprocess.run([sys.executable, os.path.abspath(__file__)], cwd=ROOT, timeout=100, capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr


if __name__ == "__main__":
    sys.path.insert(0, ROOT)
    _run()
