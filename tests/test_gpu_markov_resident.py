"""GPU tests of the Markov rollout (code/kernel/markov_dels.py:261-278) that keeps the low-rank head
on chip, and of the launch that stands in for it when it cannot have the whole GPU.

Both sum the same MFMA steps in the same order as the per-step launches, so ids and scores
must equal theirs bit for bit.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32

CASES = [
    # batch, steps, r, V, dtype of base and prior, prior
    (4, 14, 256, 151936, BF16, True),
    (1, 2, 256, 16, F32, False),          # one tile: all workgroups but one without work
    (5, 3, 128, 4099, F16, True),         # ragged vocabulary
    (16, 5, 256, 30011, BF16, True),
    (17, 4, 256, 100003, F32, True),      # a second group of one row; LDS tiles
    (32, 3, 128, 151936, BF16, False),
    (24, 64, 256, 2048, F16, True),       # the most steps one launch takes
]


@pytest.fixture(autouse=True)
def _one_launch_wherever_it_can_run(pkg):
    """Short vocabularies and few steps take the per-step launches by default."""
    lib = pkg._lib.load()
    was = lib.dels_debug_set_rollout_resident(2)
    yield
    lib.dels_debug_set_rollout_resident(was)


class _Head(torch.nn.Module):
    def __init__(self, E, W):
        super().__init__()
        self.embedding_weight = torch.nn.Parameter(E, requires_grad=False)
        self.lm_head_weight = torch.nn.Parameter(W, requires_grad=False)
        self.vocab_size, self.rank = int(W.shape[0]), int(W.shape[1])


@torch.inference_mode()
def _eager(runner, prev, base):
    runner.static_prev_ids.copy_(prev)
    runner.static_base_logits.copy_(base)
    runner.static_out.fill_(-7)
    runner.enqueue_eager()
    torch.cuda.synchronize()
    return runner.static_out.clone(), runner.static_scores.clone()


@pytest.mark.parametrize("nb,steps,r,V,dt,with_prior", CASES)
def test_resident_and_ordered_equal_per_step_launches(pkg, dev, nb, steps, r, V, dt, with_prior):
    print(f"case markov resident nb={nb} steps={steps} r={r} V={V} dtype={dt} prior={with_prior}", flush=True)
    g = torch.Generator().manual_seed(V + nb)
    E = torch.randn(V, r, generator=g).to(dt)
    W = (torch.randn(V, r, generator=g) * 0.2).to(dt)
    prior = torch.log_softmax(torch.randn(V, generator=g), 0) if with_prior else None
    alphas = [0.5 + 0.01 * i for i in range(steps)]
    betas = [0.2 * (i % 3) for i in range(steps)] if with_prior else [0.0] * steps
    prev = torch.randint(0, V, (nb, 1), generator=g).to(dev)
    base = torch.randn(nb, steps, V, generator=g).to(dt)
    base[nb - 1, 0] = float("-inf")       # no candidate: id 0
    base = base.to(dev)
    runner = pkg.MarkovDeLSGraphRunner(local_head=_Head(E, W), batch_size=nb, steps=steps, vocab_size=V,
                                       alpha_values=alphas, beta_values=betas, baseline_logits=prior, device=dev)
    lib = pkg._lib.load()
    was = lib.dels_debug_set_rollout_resident(0)
    try:
        ids, scores = _eager(runner, prev, base)
    finally:
        lib.dels_debug_set_rollout_resident(was)
    assert int(ids[nb - 1, 0]) == 0 and float(scores[nb - 1, 0]) == float("-inf")
    for _ in range(3):
        got, sc = _eager(runner, prev, base)
        assert torch.equal(got, ids) and torch.equal(sc, scores)
    # no wait is given a second look: the launch ends without a result and the ordered one does the work
    limit = lib.dels_debug_set_resident_spin_limit(0)
    try:
        got, sc = _eager(runner, prev, base)
    finally:
        lib.dels_debug_set_resident_spin_limit(limit)
    assert torch.equal(got, ids) and torch.equal(sc, scores)
    # the control area is clean: the graph (captured with the default limit) replays the resident launch
    for _ in range(3):
        assert torch.equal(runner(prev, base), ids) and torch.equal(runner.static_scores, scores)
    runner.close()


def test_two_resident_rollouts_at_once(pkg, dev):
    """Two rollouts enqueued on two streams: whether they run one after the other or get in each
    other's way, both give their own ids."""
    nb, steps, r, V = 4, 6, 256, 60000
    g = torch.Generator().manual_seed(3)
    head = _Head(torch.randn(V, r, generator=g).to(BF16), (torch.randn(V, r, generator=g) * 0.2).to(BF16))
    made = []
    for i in range(2):
        runner = pkg.MarkovDeLSGraphRunner(local_head=head, batch_size=nb, steps=steps, vocab_size=V,
                                           alpha_values=[1.0] * steps, beta_values=[0.0] * steps,
                                           baseline_logits=None, device=dev)
        prev = torch.randint(0, V, (nb, 1), generator=g).to(dev)
        base = torch.randn(nb, steps, V, generator=g).to(BF16).to(dev)
        made.append((runner, prev, base, runner(prev, base)))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(device=dev) for _ in made]
    for _ in range(4):
        outs = []
        for (runner, prev, base, _), stream in zip(made, streams):
            with torch.cuda.stream(stream):
                outs.append(runner(prev, base))
        torch.cuda.synchronize()
        for (_, _, _, want), got in zip(made, outs):
            assert torch.equal(got, want)
    for runner, *_ in made:
        runner.close()
