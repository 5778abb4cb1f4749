"""GPU tests of rollouts whose rows hold NaN beside -inf.

The rule of every argmax of the path (code/kernel/dels.py:42-138): the lowest column whose score is
the largest, -inf included, NaN never; no such column: id 0 at -inf.  The low-rank head is zero, so a
score is fma(-beta, prior, base) on every route -- one launch, its stand-in, per-step launches -- and
each must give the ids and scores of that rule bit for bit.
"""

import numpy as np
import pytest
import torch

from test_gpu_markov_resident import _Head as _MarkovHead
from test_gpu_rollout_resident import _Head as _DeLSHead
from test_gpu_rollout_stand_in import _eager

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32
BETAS = [0.0, 0.25, 0.0, 0.5]


@pytest.fixture(autouse=True)
def _one_launch_wherever_it_can_run(pkg):
    """Short vocabularies and few steps take the per-step launches by default."""
    lib = pkg._lib.load()
    was = lib.dels_debug_set_rollout_resident(2)
    yield
    lib.dels_debug_set_rollout_resident(was)


def _inputs(nb, V, dt):
    """Rows of a [nb, 4, V] base: NaN up to and past tiles and quads, -inf elsewhere or everywhere, a finite
    or infinite value among them; prior -inf in a column (a -inf base there scores NaN where beta is not 0)."""
    g = torch.Generator().manual_seed(V + nb)
    prior = torch.log_softmax(torch.randn(V, generator=g), 0).to(dt)
    prior[0] = float("-inf")
    base = torch.randn(nb, 4, V, generator=g).to(dt)
    for m in range(nb):
        s = m % 4
        k = [1, 3, V // 2, V - 1, 0, min(V - 1, 530), V][m % 7]      # leading NaN columns
        base[m, s] = float("-inf")
        base[m, s, :k] = float("nan")
        if m % 5 == 4:
            base[m, s, V - 1] = float("inf") if m % 2 else -4.0
        base[m, (s + 1) % 4, V - 1] = 200.0                           # the last column of a row and quad
        base[m, (s + 2) % 4, V // 3] = float("inf")
    return prior, base


def _expected(prior, base):
    """ids, scores of the rule, by float64 (one rounding to float32: a single fma)."""
    with np.errstate(invalid="ignore"):
        x = base.double().numpy()
        p = prior.double().numpy()
        sc = np.stack([x[:, i] - b * p if b else x[:, i] for i, b in enumerate(BETAS)], 1).astype(np.float32)
    ok = ~np.isnan(sc)
    filled = np.where(ok, sc, -np.inf)
    best = filled.max(-1)
    hit = ok & (filled == best[..., None])
    return np.where(hit.any(-1), hit.argmax(-1), 0), best


@pytest.mark.parametrize("V", [3, 5, 18, 4101, 4104])
@pytest.mark.parametrize("dt", [BF16, F16, F32])
@pytest.mark.parametrize("kind,nb", [("markov", 5), ("markov", 21), ("dels", 5), ("dels", 21)])
def test_rollout_rows_of_nan_and_inf(pkg, dev, kind, nb, dt, V):
    print(f"case rollout nan {kind} nb={nb} V={V} dtype={dt}", flush=True)
    prior, base = _inputs(nb, V, dt)
    want_ids, want_sc = _expected(prior, base)
    sched = dict(batch_size=nb, steps=4, vocab_size=V, alpha_values=[0.5, 0.6, 0.7, 0.8], beta_values=BETAS,
                 baseline_logits=prior, device=dev)
    g = torch.Generator().manual_seed(nb)
    if kind == "markov":
        head = _MarkovHead(torch.randn(V, 256, generator=g).to(dt), torch.zeros(V, 256, dtype=dt))
        runner = pkg.MarkovDeLSGraphRunner(local_head=head, **sched)
    else:
        head = _DeLSHead(V, 64, 512, 256, "silu", False, seed=6, std=0.05)
        with torch.no_grad():
            head.low_rank_lm_head.weight.zero_()
        runner = pkg.DeLSGraphRunner(local_head=head.to(dt).to(dev), **sched)
    first = torch.randint(0, V, (nb, 1), generator=g).to(dev)
    based = base.to(dev)

    def check(route):
        ids, scores = _eager(runner, first, based)
        np.testing.assert_array_equal(ids.cpu().numpy(), want_ids, err_msg=route)
        np.testing.assert_array_equal(scores.cpu().numpy(), want_sc, err_msg=route)

    lib = pkg._lib.load()
    was = lib.dels_debug_set_rollout_resident(0)
    try:
        check("per-step launches")
    finally:
        lib.dels_debug_set_rollout_resident(was)
    check("one launch")
    if kind == "markov" or nb > 16:
        limit = lib.dels_debug_set_resident_spin_limit(0)
        try:
            check("stand-in")
        finally:
            lib.dels_debug_set_resident_spin_limit(limit)
    runner.close()
