"""GPU tests of the route that a rollout takes: one launch where that takes less time, else a launch per step.

Seen from outside with no re-read allowed and the stand-in's waits given no look: a rollout that the
one launch takes then ends with ids of -1.
"""

import pytest
import torch

from test_gpu_rollout_stand_in import _eager, _runner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,nb,steps,V,one_launch", [
    ("markov", 4, 16, 8191, True), ("markov", 4, 15, 8191, False),
    ("markov", 16, 8, 8192, True), ("markov", 16, 7, 8192, False),
    ("markov", 1, 4, 16384, True), ("markov", 1, 3, 16384, False),
    ("markov", 2, 3, 32768, True), ("markov", 2, 2, 65535, False), ("markov", 2, 2, 65536, True),
    ("markov", 17, 40, 30719, False), ("markov", 17, 8, 30720, True), ("markov", 32, 7, 30720, False),
    ("markov", 20, 4, 65536, True), ("markov", 20, 3, 98303, False), ("markov", 20, 3, 98304, True),
    ("dels", 17, 3, 4099, True), ("dels", 17, 2, 65535, False), ("dels", 17, 2, 65536, True),
    ("dels", 32, 1, 65536, False),
])
def test_route(pkg, dev, kind, nb, steps, V, one_launch):
    print(f"case route {kind} nb={nb} steps={steps} V={V}", flush=True)
    runner = _runner(pkg, dev, kind, nb, steps, V)
    g = torch.Generator().manual_seed(nb)
    first = torch.randint(0, V, (nb, 1), generator=g).to(dev)
    base = torch.randn(nb, steps, V, generator=g).to(torch.bfloat16).to(dev)
    lib = pkg._lib.load()
    limit = lib.dels_debug_set_resident_spin_limit(0)
    lib.dels_debug_set_ordered_wait_limit(0)
    try:
        ids, _ = _eager(runner, first, base)
    finally:
        lib.dels_debug_set_ordered_wait_limit(-1)
        lib.dels_debug_set_resident_spin_limit(limit)
    assert bool((ids == -1).all()) if one_launch else bool((ids >= 0).all())
    runner.close()
