"""GPU tests of the e4m3 argmax kernel that shares each tile of B among several 16-row groups.

It takes the e4m3 fused argmax for 17 rows and more wherever the MFMA-tiled kernel does not, and
sums the same MFMA steps in the same order as the 16-row kernel: ids and scores must equal those
of calls on 16 rows at a time bit for bit.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize("M,r,V,ld,bdt,pdt", [
    (17, 512, 4112, 4112, BF16, BF16),
    (32, 256, 30000, 30004, F32, F32),
    (33, 512, 20011, 20011, BF16, None),       # odd V: element loads
    (63, 512, 151936, 151936, BF16, F32),
    (64, 256, 1004, 1004, F16, F16),           # V % 8 = 4: past 63 rows where the tiled kernel does not apply
    (40, 512, 16, 16, F32, None),              # one tile for the whole grid
    (20, 256, 5, 5, BF16, BF16),               # less than a tile
    (150, 512, 9003, 9003, F16, F16),          # three passes
])
def test_rows8_argmax_equals_16_rows_at_a_time(pkg, dev, M, r, V, ld, bdt, pdt):
    print(f"case rows8 argmax M={M} r={r} V={V} ld={ld} base={bdt} prior={pdt}", flush=True)
    g = torch.Generator().manual_seed(M * 31 + r + V)
    rank = (torch.randn(M, r, generator=g) * 1.5).to(BF16)
    rank[7] = 0.0                                     # an all-zero row: scale 1
    Bq = pkg.quantize_pack_fp8((torch.randn(V, r, generator=g) * 0.05).to(BF16).to(dev), "k128")
    base = (torch.randn(M, ld, generator=g) * 3).to(bdt)
    base[3] = float("-inf")                           # no candidate: id 0, -inf
    base[5, : min(V, 3)] = 60.0
    prior = None if pdt is None else torch.log_softmax(torch.randn(V, generator=g), 0).to(pdt).to(dev)
    alpha, beta = torch.rand(M, generator=g) * 0.6, torch.rand(M, generator=g) * 0.6
    beta[::5] = 0.0
    rd, based, ad, bd = rank.to(dev), base.to(dev)[:, :V], alpha.to(dev), beta.to(dev)
    ids, score = pkg.fused_argmax_fp8(rd, Bq, based, prior, ad, bd)
    parts = [pkg.fused_argmax_fp8(rd[i:i + 16], Bq, based[i:i + 16], prior, ad[i:i + 16], bd[i:i + 16])
             for i in range(0, M, 16)]
    torch.cuda.synchronize()
    assert torch.equal(ids, torch.cat([p[0] for p in parts]))
    assert torch.equal(score, torch.cat([p[1] for p in parts]))
    assert int(ids[3]) == 0 and float(score[3]) == float("-inf")
