"""Two models on two threads of one process, each on its own stream: a prompt
waits for nothing that another model's launches can hold up, and its result is
the one it has alone."""
import threading

import numpy as np
import pytest

from gpu_util import banner
from test_gpu_prefill import _small_model, _spec

pytestmark = pytest.mark.gpu

# 224-block o + FFN launches of one block per CU: two of them fit a GPU of 256
# CUs only one after the other
WIDE = dict(n_layers=1, hidden=512, ffn=14336, n_heads=8, n_kv_heads=2, head_dim=64)


@pytest.mark.parametrize("mode", ["turbo", "precision"])
@pytest.mark.parametrize("n", [1, 40])
def test_prompts_on_two_threads(mode, n):
    banner(f"two models, two threads, prompts of {n}, {mode}")
    models = [_small_model(_spec(mode=mode, kinks_per_row=0, **WIDE))[1] for _ in range(2)]
    ids = np.random.default_rng(n).integers(0, 512, n).astype(np.int32)
    alone = [m.prefill(ids, 0) for m in models]
    start, failures = threading.Barrier(2), [[], []]

    def go(i):
        start.wait()
        for k in range(2000):
            try:
                if not np.array_equal(models[i].prefill(ids, 0), alone[i]):
                    failures[i].append((k, "another result"))
            except Exception as e:   # (collected: the other thread goes on)
                failures[i].append((k, str(e)))
            if len(failures[i]) > 3:
                return

    threads = [threading.Thread(target=go, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for m in models:
        m.close()
    assert failures == [[], []]
