"""GPU tests of the base logits of the one-launch rollouts: quads of columns at every alignment.

The one-launch Markov rollout (code/kernel/markov_dels.py:261-278) combines in the order of the
per-step kernels: ids and scores must equal those of single steps bit for bit.  The DeLS rollout
shares its loads and its argmax.
"""

import pytest
import torch

from test_gpu_markov_resident import _eager, _Head

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.fixture(autouse=True)
def _one_launch_wherever_it_can_run(pkg):
    """Short vocabularies and few steps take the per-step launches by default."""
    lib = pkg._lib.load()
    was = lib.dels_debug_set_rollout_resident(2)
    yield
    lib.dels_debug_set_rollout_resident(was)


# vocabularies that leave 0 to 3 columns of a quad, parts of a tile, and less than a quad
@pytest.mark.parametrize("V", [3, 5, 18, 4100, 4101, 4102, 4103])
@pytest.mark.parametrize("dt", [BF16, F16, F32])
@pytest.mark.parametrize("nb", [5, 21])
def test_rollout_quads_equal_per_step_launches(pkg, dev, V, dt, nb):
    steps, r = 4, 256
    print(f"case rollout quads V={V} dtype={dt} nb={nb}", flush=True)
    g = torch.Generator().manual_seed(V + nb)
    E = torch.randn(V, r, generator=g).to(dt)
    W = (torch.randn(V, r, generator=g) * 0.2).to(dt)
    prior = torch.log_softmax(torch.randn(V, generator=g), 0)
    base = torch.randn(nb, steps, V, generator=g).to(dt)
    base[1, 1] = float("-inf")                      # no candidate
    base[2, 0, : V // 2] = float("nan")             # never taken
    base[nb - 1, 2, V - 1] = 200.0                  # the last column of the last row and quad
    base[3, 3, V - 1] = float("inf")
    prev = torch.randint(0, V, (nb, 1), generator=g).to(dev)
    base = base.to(dev)
    runner = pkg.MarkovDeLSGraphRunner(local_head=_Head(E, W), batch_size=nb, steps=steps, vocab_size=V,
                                       alpha_values=[0.5, 0.6, 0.7, 0.8], beta_values=[0.0, 0.2, 0.0, 0.3],
                                       baseline_logits=prior, device=dev)
    lib = pkg._lib.load()
    was = lib.dels_debug_set_rollout_resident(0)
    try:
        ids, scores = _eager(runner, prev, base)
    finally:
        lib.dels_debug_set_rollout_resident(was)
    assert int(ids[nb - 1, 2]) == V - 1 and int(ids[3, 3]) == V - 1
    got, sc = _eager(runner, prev, base)
    assert torch.equal(got, ids) and torch.equal(sc, scores)
    runner.close()
