"""GPU tests of the launch that stands in for a one-launch rollout that cannot have the whole GPU.

With no re-read allowed the one-launch rollout gives up; what comes out then is the stand-in's.
"""

import pytest
import torch

from test_gpu_markov_resident import _Head as _MarkovHead
from test_gpu_rollout_resident import _Head as _DeLSHead

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _one_launch_wherever_it_can_run(pkg):
    """Short vocabularies and few steps take the per-step launches by default."""
    lib = pkg._lib.load()
    was = lib.dels_debug_set_rollout_resident(2)
    yield
    lib.dels_debug_set_rollout_resident(was)


def _runner(pkg, dev, kind, nb, steps, V):
    sched = dict(batch_size=nb, steps=steps, vocab_size=V, alpha_values=[0.7] * steps, beta_values=[0.0] * steps,
                 baseline_logits=None, device=dev)
    if kind == "markov":
        g = torch.Generator().manual_seed(5)
        head = _MarkovHead(torch.randn(V, 128, generator=g).to(torch.bfloat16),
                           (torch.randn(V, 128, generator=g) * 0.2).to(torch.bfloat16))
        return pkg.MarkovDeLSGraphRunner(local_head=head, **sched)
    head = _DeLSHead(V, 64, 512, 256, "silu", False, seed=6, std=0.05).to(dev)
    return pkg.DeLSGraphRunner(local_head=head, **sched)


@torch.inference_mode()
def _eager(runner, first, base):
    getattr(runner, "static_prev_ids" if hasattr(runner, "static_prev_ids") else "static_prefix_ids").copy_(first)
    runner.static_base_logits.copy_(base)
    runner.static_out.fill_(-7)
    runner.static_scores.fill_(0.5)
    runner.enqueue_eager()
    torch.cuda.synchronize()
    return runner.static_out.clone(), runner.static_scores.clone()


@pytest.mark.parametrize("kind,nb,steps", [("markov", 3, 5), ("markov", 20, 3), ("dels", 18, 1), ("dels", 21, 4)])
def test_stand_in_runs_and_its_waits_end(pkg, dev, kind, nb, steps):
    """The stand-in's waits given no look either: the ids are -1 (so it is that launch that ran), every
    workgroup has ended, and the control area is clean: the next rollouts, by the stand-in and by
    the one launch, are right."""
    V = 4099
    print(f"case stand-in {kind} nb={nb} steps={steps}", flush=True)
    runner = _runner(pkg, dev, kind, nb, steps, V)
    g = torch.Generator().manual_seed(nb)
    first = torch.randint(0, V, (nb, 1), generator=g).to(dev)
    base = torch.randn(nb, steps, V, generator=g).to(torch.bfloat16).to(dev)
    want = _eager(runner, first, base)
    lib = pkg._lib.load()
    limit = lib.dels_debug_set_resident_spin_limit(0)
    try:
        lib.dels_debug_set_ordered_wait_limit(0)
        try:
            ids, scores = _eager(runner, first, base)
        finally:
            lib.dels_debug_set_ordered_wait_limit(-1)
        assert bool((ids == -1).all()) and bool((scores == float("-inf")).all())
        got = _eager(runner, first, base)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    finally:
        lib.dels_debug_set_resident_spin_limit(limit)
    got = _eager(runner, first, base)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    runner.close()
