"""Top-k selection and its gate at row widths around the edges of the select
kernel's workgroups (256 threads up to 1024 pages, 1, 2 or 4 scores per
thread; 1024 threads above), against the oracle's selection
(cvsa/backend.py:737-747) and coverage (cvsa/kernels/coverage.py:159-215)."""
import pytest
import torch

from cvsa import ops
from oracle import cvsa_oracle as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W", [1, 2, 63, 65, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025,
                               1026, 2049])
def test_select_at_width_edges(gpu, W):
    """Rows: distinct scores, heavy ties (more than 64 scores in the k-th
    bucket), one value, a -inf tail, a few outliers that crowd the rest into
    one bucket, +inf entries; budgets 1, 3, around half, and the whole row."""
    g = torch.Generator().manual_seed(W)
    rows = torch.randn(6, 1, W, generator=g) * 0.5 + 1.8
    rows[1] = (rows[1] * 2).round()
    rows[2] = 1.25
    nv = max(1, W - W // 3)
    rows[3, :, nv:] = float("-inf")
    rows[4, :, ::97] *= 1e6
    rows[5, :, ::53] = float("inf")
    ctx = torch.full((6,), 16 * W, dtype=torch.int32)
    ctx[3] = 16 * nv
    for k in sorted({1, min(3, W), max(1, W // 2), W}):
        want, n_want = ref.select_topk(rows, k, ctx, 16)
        idx, n, acc, cov = ops.select_topk(rows.to(gpu), k, ctx.to(gpu), 16, 0.9)
        assert torch.equal(n.cpu(), n_want), k
        assert torch.equal(idx.cpu(), want), k
        finite = slice(0, 5)  # a +inf score has no finite normaliser
        acc_w, cov_w = ref.check_coverage(rows[finite], want[finite], n_want[finite], 0.9)
        # Sums of W fp32 exponentials: W ulps of 2^-24 at most, far below 1e-5.
        assert torch.allclose(cov[finite].cpu(), cov_w, rtol=0, atol=1e-5), k
        sure = (cov_w - 0.9).abs() > 1e-5
        assert torch.equal(acc[finite].cpu()[sure], acc_w[sure]), k
