"""What the calls on one grid keep and share: overlapping calls of two host
threads against the same calls one after the other."""
import threading

import numpy as np
import pytest
import torch

import top3d_amd

pytestmark = pytest.mark.gpu


# the radii have sums of weights of different sizes (5^3 and 9^3) and of one
# size (5^3) with other values
@pytest.mark.parametrize("radii", [(2.5, 4.5), (2.5, 2.9)])
def test_filters_of_two_threads(radii):
    print(f"[gpu call state] filters {radii}", flush=True)
    g = top3d_amd.Grid(32, 16, 24, 3)
    rng = np.random.default_rng(7)
    x = g.density(rng.uniform(0.1, 1.0, 32 * 16 * 24))
    torch.cuda.synchronize()
    ref = [(g.filter(r, x).cpu(), g.filter_grad(r, x).cpu()) for r in radii]
    bad = []

    def calls(k):
        for _ in range(50):
            y, w = g.filter(radii[k], x), g.filter_grad(radii[k], x)
            if not (torch.equal(y.cpu(), ref[k][0]) and torch.equal(w.cpu(), ref[k][1])):
                bad.append(radii[k])

    threads = [threading.Thread(target=calls, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    g.close()
