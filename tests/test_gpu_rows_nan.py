"""GPU tests of the 17-to-64-row argmax kernels on rows that hold NaN beside -inf.

The rule (code/kernel/dels.py:42-138, as the 16-row kernels have it): the lowest column whose score is
the largest, -inf included, NaN never; no such column: id 0 at -inf.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize("fmt", ["packed", "rowmajor", "e4m3"])
@pytest.mark.parametrize("M,V,bdt,pdt", [
    (17, 4112, BF16, BF16),
    (33, 40011, F32, None),           # unaligned rows
    (32, 4097, F16, F32),             # one column in the last tile
    (49, 36867, BF16, BF16),          # less than a quad of columns in the last tile
    (18, 3, BF16, None),              # less than a quad
    (63, 70000, F16, F16),            # several tiles per wave
    (70, 9003, BF16, BF16),           # past 64 rows where the tiled kernel does not apply
    (131, 65540, BF16, F32),          # ... eight groups a pass
])
def test_rows_of_nan_and_inf(pkg, dev, fmt, M, V, bdt, pdt):
    print(f"case rows nan M={M} V={V} base={bdt} prior={pdt} {fmt}", flush=True)
    r = 256
    g = torch.Generator().manual_seed(M + V)
    rank = torch.randn(M, r, generator=g).to(BF16).to(dev)
    B = (torch.randn(V, r, generator=g) * 0.05).to(BF16).to(dev)
    base = (torch.randn(M, V, generator=g) * 3).to(bdt)
    want = {}
    for m in range(0, M, 2):
        k = [1, 3, V // 2, V - 1, 0, min(V - 1, 530), V][(m // 2) % 7]       # leading NaN columns
        base[m] = float("-inf")
        base[m, :k] = float("nan")
        want[m] = k if k < V else 0
    base[1, V - 1] = base[1, V // 3] = float("inf")                          # the lowest of two infinities
    base[3, V // 2] = float("nan")
    based = base.to(dev)
    prior = None if pdt is None else torch.log_softmax(torch.randn(V, generator=g), 0).to(pdt).to(dev)
    alpha, beta = torch.rand(M, generator=g).to(dev), torch.rand(M, generator=g).to(dev)
    if fmt == "e4m3":
        Bq = pkg.quantize_pack_fp8(B, "k128")
        run = lambda lo, hi: pkg.fused_argmax_fp8(rank[lo:hi], Bq, based[lo:hi], prior, alpha[lo:hi], beta[lo:hi])  # noqa: E731
    else:
        Bw = pkg.pack_operand(B) if fmt == "packed" else B
        run = lambda lo, hi: pkg.fused_argmax(rank[lo:hi], Bw, based[lo:hi], prior, alpha[lo:hi], beta[lo:hi])  # noqa: E731
    ids, score = run(0, M)
    parts = [run(i, min(i + 16, M)) for i in range(0, M, 16)]
    torch.cuda.synchronize()
    for m, id_ in want.items():
        assert int(ids[m]) == id_ and float(score[m]) == float("-inf"), (m, int(ids[m]), id_)
    assert int(ids[1]) == V // 3 and float(score[1]) == float("inf")
    assert torch.equal(ids, torch.cat([p[0] for p in parts]))
    assert torch.equal(score, torch.cat([p[1] for p in parts]))
