"""Builds on several threads with more workspaces than the library keeps round
graphs: the oldest graphs are dropped while other threads launch theirs."""
import threading

import numpy as np
import pytest

import oracle as oc

pytestmark = pytest.mark.gpu


def test_builds_while_graphs_are_dropped(gpu):
    import torch

    import checkers_amd as ck
    n, max_rules, k = 3000, 13, ck.repair_masked_bits(1, None)
    words = [np.minimum(np.random.default_rng(t).geometric(0.2, n), 300).astype(np.uint16) << 7 for t in range(3)]
    refs = [oc.repair_build(w.view(np.uint8), n, 2, k, max_rules) for w in words]
    srcs = [torch.from_numpy(w.view(np.uint8).copy()).to(gpu) for w in words]
    reps = [[ck.Repairer(n, 1, None, max_rules) for _ in range(12)] for _ in words]
    streams = [torch.cuda.Stream() for _ in words]
    torch.cuda.synchronize()
    before, errors = ck.lib().ckr_repair_graphs_made(), []

    def work(t):
        try:
            with torch.cuda.stream(streams[t]):
                for _ in range(2):
                    for rp in reps[t]:
                        got = rp.build(srcs[t])
                        assert got["rules"] == refs[t]["rules"] and got["out_len"] == refs[t]["out_len"]
        except Exception as e:  # noqa: BLE001 (shown by the main thread)
            errors.append(e)

    threads = [threading.Thread(target=work, args=(t,), daemon=True) for t in range(3)]
    for th in threads:
        th.start()
    for th in threads:
        th.join(60)
    assert not any(th.is_alive() for th in threads) and not errors, errors
    assert ck.lib().ckr_repair_graphs_made() - before > 64  # some were dropped and made again
