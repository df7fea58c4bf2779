"""Rows past the held length whose threshold is +0 or near it: fewer than 2048 positive keys (none, some,
one short of and exactly 2048, one more) filled up with the first zeros, too few zeros to fill (the
threshold negative), zeros only at the row's end or only by the mask, -0.0 beside +0, one CTA a row and
split, aligned and not, either candidate list; against the oracle, order included."""
import numpy as np
import pytest
import torch

import hcu_ops
from oracle.topk_c import topk_radix

pytestmark = pytest.mark.gpu


def _row(n_pos, zeros, length, g):
    """A row of `length` scores: n_pos positive ones, `zeros` zeros (a count, "end": the last 3000, or
    "rest"), the others negative."""
    x = -(torch.rand(length, generator=g) + 1e-3)
    x[torch.rand(length, generator=g) < 0.01] = -0.0
    perm = torch.randperm(length, generator=g)
    x[perm[:n_pos]] = torch.rand(n_pos, generator=g) ** 4 + 1e-30
    rest = perm[n_pos:]
    if zeros == "rest":
        x[rest] = 0.0
    elif zeros == "end":
        tail = rest[rest >= length - 3000]
        x[tail] = 0.0
        x[rest[rest < length - 3000]] = -1.0
    else:
        x[rest[:zeros]] = 0.0
    return x


@pytest.mark.parametrize("length,pad", [(8200, 0), (16384, 0), (16383, 2), (32768, 0), (40000, 0), (65536, 0), (70001, 0),
                                        (90112, 0)])
def test_sparse_rows(gpu, length, pad):
    g = torch.Generator().manual_seed(length)
    # (enough zeros that the sample's threshold falls on +0, and just too few to fill the row)
    shapes = [(0, "rest"), (1, "rest"), (1500, "rest"), (2047, "rest"), (2048, "rest"), (2049, "rest"), (700, length // 2),
              (300, "end"), (1000, 1047), (1000, 1048), (1900, 147), (0, 2048), (0, 2047), (2047, 1), (2048, 0)]
    x = torch.stack([_row(n, z, length, g) for n, z in shapes])
    rows = len(shapes)
    lens = torch.full((rows,), length, dtype=torch.int32)
    lens[1::4] = length - 3
    pt = torch.randperm(length, generator=g).to(torch.int32).repeat(rows, 1).contiguous()
    dev = torch.zeros(rows, length + pad, device=gpu)
    dev[:, :length] = x.to(gpu)
    score = dev[:, :length]
    cu = torch.arange(rows + 1, dtype=torch.int32, device=gpu)
    want = topk_radix(x.numpy(), None, lens.numpy(), pt.numpy(), length)
    for splits in (1, 8):
        got = hcu_ops.topk_transform(score, lens.to(gpu), pt.to(gpu), cu, max_splits=splits).cpu().numpy()
        bad = [shapes[r] for r in range(rows) if not np.array_equal(got[r], want[r])]
        assert not bad, f"rows of (positives, zeros) {bad}, {splits} splits"
    if length % 16:
        return
    keep = torch.rand(rows, length, generator=g) < 0.05  # zeros by the mask: 95% of the row
    m = (keep.view(rows, -1, 16).int() << torch.arange(16, dtype=torch.int32)).sum(-1)
    m = torch.where(m > 32767, m - 65536, m).to(torch.int16).contiguous()
    dense = torch.randn(rows, length, generator=g)
    dense[~keep] = float("nan")
    want = topk_radix(dense.numpy(), m.numpy(), lens.numpy(), pt.numpy(), length)
    got = hcu_ops.sparse_mask_topk_transform(dense.to(gpu), m.to(gpu), lens.to(gpu), pt.to(gpu), cu).cpu().numpy()
    bad = [r for r in range(rows) if not np.array_equal(got[r], want[r])]
    assert not bad, f"masked rows {bad}"
