"""Top-k over dense scores whose rows are not 16-B aligned (odd widths), one CTA a row: either side of the widest row
held in registers and of the width from which the candidate list is longer, every score distribution, against
the oracle's selection."""
import numpy as np
import pytest
import torch

from hcu_ops import _C
import workloads as wl
from oracle.topk_c import topk_radix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dist", wl.TOPK_DISTS)
@pytest.mark.parametrize("width", [8191, 8193, 20989, 81919, 81921])
def test_unaligned_rows(gpu, width, dist):
    rows = 5
    x, _, _, pt = wl.topk_scores(rows, width, dist, seed=width)
    x = torch.nan_to_num(x, nan=0.0)
    lens = torch.tensor([width, width - 1, 8192, 2049, max(2048, width - 4097)], dtype=torch.int32)
    cu = torch.arange(rows + 1, dtype=torch.int32)
    out = _C.topk_transform(x.to(gpu), lens.to(gpu), pt.to(gpu), cu.to(gpu), 2048, 1, None)
    want = topk_radix(x.numpy(), None, lens.numpy(), pt.numpy(), width, cu_seqlens_q=cu.numpy())
    assert np.array_equal(out.cpu().numpy(), want)
