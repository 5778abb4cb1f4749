"""GPU tests of the one-launch rollout (code/kernel/dels.py:425-467) at 17 to 32 rows, and of the launch
that stands in for it when it cannot have the whole GPU.

Both sum in the order of the one-launch rollout of up to 16 rows, so ids and scores must equal
those of two such rollouts over the same rows bit for bit.
"""

import pytest
import torch

from test_gpu_rollout_resident import _check_against_oracle, _Head

pytestmark = pytest.mark.gpu

CASES = [
    # nb, steps, G, V, prior, act, rank bias, GRU bias
    (24, 14, 1024, 151936, True, "silu", False, False),
    (17, 3, 512, 4099, False, "identity", True, True),   # one row in the second group, few tiles
    (32, 4, 1024, 30011, True, "silu", True, True),
    (18, 1, 1024, 20011, True, "silu", False, True),    # one step: no GRU after it
]


@pytest.fixture(autouse=True)
def _one_launch_wherever_it_can_run(pkg):
    """Short vocabularies and few steps take the per-step launches by default."""
    lib = pkg._lib.load()
    was = lib.dels_debug_set_rollout_resident(2)
    yield
    lib.dels_debug_set_rollout_resident(was)


@torch.inference_mode()
def _eager(runner, prefix, base):
    runner.static_prefix_ids.copy_(prefix)
    runner.static_base_logits.copy_(base)
    runner.static_out.fill_(-7)
    runner.enqueue_eager()
    torch.cuda.synchronize()
    return runner.static_out.clone(), runner.static_scores.clone()


@pytest.mark.parametrize("nb,steps,G,V,with_prior,act,rank_bias,gru_bias", CASES)
def test_two_groups_equal_one_at_a_time(pkg, dev, nb, steps, G, V, with_prior, act, rank_bias, gru_bias):
    print(f"case two-group rollout nb={nb} steps={steps} G={G} V={V}", flush=True)
    head = _Head(V, 64, G, 256, act, rank_bias, seed=40 + V % 97, std=0.02 if G >= 1024 else 0.05,
                 gru_bias=gru_bias).to(dev)
    g = torch.Generator().manual_seed(nb)
    prior = torch.log_softmax(torch.randn(V, generator=g), 0) if with_prior else None
    alphas = [0.8 + 0.05 * i for i in range(steps)]
    betas = [0.1 * (i % 3) for i in range(steps)] if with_prior else [0.0] * steps
    prefix = torch.randint(0, V, (nb, 1), generator=g)
    base = (torch.randn(nb, steps, V, generator=g) * 0.5).to(torch.bfloat16)

    def make(rows):
        return pkg.DeLSGraphRunner(local_head=head, batch_size=rows, steps=steps, vocab_size=V, alpha_values=alphas,
                                   beta_values=betas, baseline_logits=prior, device=dev)

    pd, bd = prefix.to(dev), base.to(dev)
    parts = []
    for lo, hi in ((0, 16), (16, nb)):
        one = make(hi - lo)
        parts.append(_eager(one, pd[lo:hi], bd[lo:hi]))
        one.close()
    want = [torch.cat([p[i] for p in parts]) for i in range(2)]
    runner = make(nb)
    for _ in range(3):
        ids, scores = _eager(runner, pd, bd)
        assert torch.equal(ids, want[0]) and torch.equal(scores, want[1])
    # no wait is given a second look: the launch ends without a result and the ordered one does the work
    lib = pkg._lib.load()
    limit = lib.dels_debug_set_resident_spin_limit(0)
    try:
        ids, scores = _eager(runner, pd, bd)
    finally:
        lib.dels_debug_set_resident_spin_limit(limit)
    assert torch.equal(ids, want[0]) and torch.equal(scores, want[1])
    # the graph replays the one launch on the same workspace
    for _ in range(3):
        assert torch.equal(runner(pd, bd), want[0]) and torch.equal(runner.static_scores, want[1])
    if V <= 40000:
        _check_against_oracle(head, prefix, base, prior, alphas, betas, act, ids, scores, gru_bias, rank_bias)
    runner.close()
