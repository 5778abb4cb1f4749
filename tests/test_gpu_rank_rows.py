"""GPU tests of the rank projection (code/kernel/dels.py:437-443) around the rows and hidden sizes at
which it changes kernels.

Operands are -1, 0 and 1 with few nonzeros per row, so every partial sum is a small integer, exact
in fp32 in any order and in bf16 after the bias: results must equal the integers.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

BF16 = torch.bfloat16


def _ternary(rows, cols, g, keep=0.02):
    x = torch.randint(0, 2, (rows, cols), generator=g) * 2 - 1
    return (x * (torch.rand(rows, cols, generator=g) < keep)).to(BF16)


@pytest.mark.parametrize("layout", ["packed", "rowmajor"])
@pytest.mark.parametrize("M,d,r", [
    (16, 4096, 512), (17, 4096, 512), (33, 2048, 72), (63, 1088, 8), (64, 4096, 256), (65, 2560, 256),
    (17, 1024, 512), (40, 1056, 64),      # short K, and K no multiple of 64: the skinny kernel
    (129, 4096, 512), (300, 2560, 136),
])
def test_rank_proj_exact(pkg, dev, M, d, r, layout):
    print(f"case rank proj M={M} d={d} r={r} {layout}", flush=True)
    g = torch.Generator().manual_seed(M + d + r)
    h, A = _ternary(M, d, g, 0.3), _ternary(r, d, g)
    bias = torch.randint(-3, 4, (r,), generator=g).to(BF16)
    want = h.double() @ A.double().t() + bias.double()
    assert want.abs().max() < 256
    Ad = A.to(dev)
    got = pkg.rank_proj(h.to(dev), pkg.pack_operand(Ad) if layout == "packed" else Ad, bias.to(dev))
    torch.cuda.synchronize()
    assert torch.equal(got.cpu().double(), want)


def test_rank_proj_rows_past_32_bit_offsets(pkg, dev):
    """Rows of h so far apart that a tile's byte offsets pass 32 bits."""
    g = torch.Generator().manual_seed(5)
    M, d, r, ld = 18, 2048, 64, (1 << 24) + 8
    h, A = _ternary(M, d, g, 0.3), _ternary(r, d, g)
    wide = torch.empty((M - 1) * ld + d, dtype=BF16, device=dev)
    view = wide.as_strided((M, d), (ld, 1))
    view.copy_(h)
    got = pkg.rank_proj(view, pkg.pack_operand(A.to(dev)))
    torch.cuda.synchronize()
    assert torch.equal(got.cpu().double(), h.double() @ A.double().t())
