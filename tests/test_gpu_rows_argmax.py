"""GPU tests of the argmax kernel that shares each tile of B among several 16-row groups.

It takes the fused argmax (code/kernel/dels.py:15-138) for 17 rows and more wherever the
MFMA-tiled kernel does not: fewer than 64 rows, row-major B, or rows the tiled kernel's loads
do not reach.  It sums the same MFMA steps in the same order as the 16-row kernel, so its ids
and scores must equal those of calls on 16 rows at a time bit for bit; one case per family is
also checked against the oracle.
"""

import pytest
import torch

from test_gpu_parity import assert_parity, f

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32

CASES = [
    # M, r, V, base columns (row stride), base dtype, prior dtype, packed
    (17, 512, 4112, 4112, BF16, BF16, True),
    (32, 256, 30000, 30004, F32, F32, True),
    (33, 512, 30000, 30000, F32, F32, True),          # fp32 at r = 512: 48 rows a pass
    (49, 512, 20011, 20011, F32, None, True),         # odd V: element loads
    (64, 512, 4100, 4104, BF16, F32, False),          # row-major, V % 16 = 4, two passes of the prior's own dtype
    (48, 512, 1001, 1001, F16, F16, False),
    (63, 256, 151936, 151936, BF16, BF16, True),
    (40, 128, 16, 16, BF16, None, True),              # one tile for the whole grid
    (20, 128, 5, 5, F16, F32, False),                 # less than a tile
    (130, 512, 9003, 9003, BF16, BF16, True),         # past 64 rows where the tiled kernel does not apply
    (200, 256, 8192, 8200, BF16, BF16, False),
]


def _inputs(pkg, M, r, V, ld, bdt, pdt):
    g = torch.Generator().manual_seed(M * 31 + r + V)
    rank = (torch.randn(M, r, generator=g) * 1.5).to(BF16)
    B = (torch.randn(V, r, generator=g) * 0.05).to(BF16)
    base = (torch.randn(M, ld, generator=g) * 3).to(bdt)[:, :V]
    prior = None if pdt is None else torch.log_softmax(torch.randn(V, generator=g), 0).to(pdt)
    alpha, beta = torch.rand(M, generator=g) * 0.6, torch.rand(M, generator=g) * 0.6
    beta[::5] = 0.0                                   # rows without the prior term
    if pdt is not None and V > 40:
        prior[V // 2] = float("inf")                  # only those rows may still pick it
    base[3] = float("-inf")                           # no candidate: id 0, -inf
    base[5, : min(V, 3)] = 60.0                       # ties: the lowest index
    return rank, B, base, prior, alpha, beta


@pytest.mark.parametrize("M,r,V,ld,bdt,pdt,packed", CASES)
def test_rows_argmax_equals_16_rows_at_a_time(pkg, dev, M, r, V, ld, bdt, pdt, packed):
    print(f"case rows argmax M={M} r={r} V={V} ld={ld} base={bdt} prior={pdt} packed={packed}", flush=True)
    rank, B, base, prior, alpha, beta = _inputs(pkg, M, r, V, ld, bdt, pdt)
    full = torch.empty(M, ld, dtype=bdt, device=dev)
    based = full[:, :V]
    based.copy_(base)
    rd, ad, bd = rank.to(dev), alpha.to(dev), beta.to(dev)
    Bd = B.to(dev)
    Bd = pkg.pack_operand(Bd) if packed else Bd
    pd = None if prior is None else prior.to(dev)
    ids, score = pkg.fused_argmax(rd, Bd, based, pd, ad, bd)
    parts = [pkg.fused_argmax(rd[i:i + 16], Bd, based[i:i + 16], pd, ad[i:i + 16], bd[i:i + 16])
             for i in range(0, M, 16)]
    torch.cuda.synchronize()
    assert torch.equal(ids, torch.cat([p[0] for p in parts]))
    assert torch.equal(score, torch.cat([p[1] for p in parts]))
    assert int(ids[3]) == 0 and float(score[3]) == float("-inf")
    if V <= 40000:
        keep = torch.ones(V, dtype=torch.bool)
        if pdt is not None and V > 40:
            keep[V // 2] = False                      # the oracle check leaves the infinite prior out
            assert not torch.any(ids.cpu()[beta != 0] == V // 2)
        rows = torch.tensor([m for m in range(M) if m != 3 and (pdt is None or beta[m] != 0 or V <= 40)])
        at = torch.full((V,), -1, dtype=torch.int64)
        at[keep] = torch.arange(int(keep.sum()))
        assert_parity(at[ids.cpu()[rows]], score.cpu()[rows], f(rank[rows]), f(B[keep]), f(base[rows][:, keep]),
                      None if prior is None else f(prior[keep]), f(alpha[rows]), f(beta[rows]))


def test_rows_argmax_gathered_rank(pkg, dev):
    """The Markov step's gathered rank (code/kernel/markov_dels.py:216-268) at 24 rows."""
    g = torch.Generator().manual_seed(9)
    M, r, V, rows = 24, 256, 20000, 500
    E = torch.randn(rows, r, generator=g).to(BF16)
    B = (torch.randn(V, r, generator=g) * 0.05).to(BF16)
    base = (torch.randn(M, V, generator=g) * 3).to(BF16)
    tok = torch.randint(0, rows, (M,), generator=g)
    tok[1], tok[2] = -4, rows + 9                      # clamped to the table
    ids, score = pkg.gather_argmax(tok.to(dev), E.to(dev), pkg.pack_operand(B.to(dev)), base.to(dev), None, 0.4, 0.0)
    torch.cuda.synchronize()
    assert_parity(ids, score, f(E)[tok.clamp(0, rows - 1).numpy()], f(B), f(base), None,
                  torch.full((M,), 0.4).numpy(), torch.zeros(M).numpy())
