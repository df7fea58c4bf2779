"""Rows held in registers by the top-k (up to 8192 tokens): row and width edges of every launch shape
(quads past the row, the last token of a shape, rows just past 2048), aligned and unaligned, masked and
dense, on scores that make the threshold search take each of its ends: exactly 2048 positive keys, the
threshold at +0 or -0, heavy ties, values over many octaves, infinities and NaNs of both signs -- the
lowest key of all among them, which tokens past the row hold too -- against the oracle, order included."""
import numpy as np
import pytest
import torch

import hcu_ops
from oracle.topk_c import topk_radix

pytestmark = pytest.mark.gpu

KINDS = ["normal", "uniform", "heavy", "ties", "two_values", "const", "pos2048", "few_pos", "neg", "minus_zero", "inf_nan",
         "lowest_key"]


def _scores(kind, rows, width, lens, g):
    x = torch.randn(rows, width, generator=g)
    if kind == "uniform":
        x = torch.rand(rows, width, generator=g)
    elif kind == "heavy":
        x = x ** 5 * torch.exp(4 * torch.randn(rows, width, generator=g))
    elif kind == "ties":
        x = torch.randint(0, 6, (rows, width), generator=g).float()
    elif kind == "two_values":
        x = torch.where(torch.rand(rows, width, generator=g) < 0.5, 1.0, 1.0 + 2.0 ** -23) * torch.ones(rows, width)
    elif kind == "const":
        x = torch.full((rows, width), -3.5)
    elif kind in ("pos2048", "few_pos"):
        x = -x.abs()
        for r in range(rows):
            n = min(2048 if kind == "pos2048" else 700, lens[r])
            at = torch.randperm(lens[r], generator=g)[:n]
            x[r, at] = torch.rand(n, generator=g) + 1e-6
            x[r, torch.randperm(lens[r], generator=g)[:100]] *= 1.0
        x[:, ::3] = torch.where(x[:, ::3] < 0, torch.zeros(1), x[:, ::3])
    elif kind == "neg":
        x = -x.abs()
    elif kind == "minus_zero":
        x = torch.where(torch.rand(rows, width, generator=g) < 0.3, x.abs(), torch.tensor(-0.0))
    elif kind == "inf_nan":
        p = torch.rand(rows, width, generator=g)
        x = torch.where(p < 0.02, torch.tensor(float("inf")), x)
        x = torch.where((p > 0.3) & (p < 0.6), torch.tensor(-float("inf")), x)
        x = torch.where((p > 0.02) & (p < 0.04), torch.tensor(float("nan")), x)
        x = torch.where((p > 0.96), torch.tensor(-1, dtype=torch.int32).view(torch.float32), x)
    elif kind == "lowest_key":  # all but some tokens hold the float whose key is 0
        low = torch.tensor(-1, dtype=torch.int32).view(torch.float32)
        x = torch.where(torch.rand(rows, width, generator=g) < 0.1, x, low)
    return x.float().contiguous()


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("rows,width,pad", [(5, 2112, 0), (7, 4096, 0), (3, 4093, 0), (6, 8192, 0), (4, 8190, 3), (300, 4096, 0),
                                            (3, 9216, 0), (3, 40000, 0)])
def test_held_rows(gpu, kind, rows, width, pad):
    g = torch.Generator().manual_seed(KINDS.index(kind) * 100 + width)
    top = min(width, 8192)
    lens = torch.randint(2049, top + 1, (rows,), generator=g)
    lens[0], lens[1], lens[2] = top, 2049, min(top, 2048 + 64)
    masked = width % 16 == 0
    x = _scores(kind, rows, width, lens.tolist(), g)
    lens = lens.to(torch.int32)
    pt = torch.randperm(3 * width, generator=g)[:width].to(torch.int32).repeat(rows, 1).contiguous()
    dev = torch.zeros(rows, width + pad, device=gpu)
    dev[:, :width] = x.to(gpu)
    score = dev[:, :width]
    cu = torch.arange(rows + 1, dtype=torch.int32, device=gpu)
    want = topk_radix(x.numpy(), None, lens.numpy(), pt.numpy(), width)
    for splits in (1, 8):
        got = hcu_ops.topk_transform(score, lens.to(gpu), pt.to(gpu), cu, max_splits=splits).cpu().numpy()
        bad = [r for r in range(rows) if not np.array_equal(got[r], want[r])]
        assert not bad, f"{kind}: rows {bad[:5]} (lengths {[int(lens[r]) for r in bad[:5]]}), {splits} splits"
    if masked:
        bits = torch.rand(rows, width, generator=g) < 0.6
        m = (bits.view(rows, -1, 16).int() << torch.arange(16, dtype=torch.int32)).sum(-1)
        m = torch.where(m > 32767, m - 65536, m).to(torch.int16).contiguous()
        want = topk_radix(x.numpy(), m.numpy(), lens.numpy(), pt.numpy(), width)
        got = hcu_ops.sparse_mask_topk_transform(score, m.to(gpu), lens.to(gpu), pt.to(gpu), cu).cpu().numpy()
        bad = [r for r in range(rows) if not np.array_equal(got[r], want[r])]
        assert not bad, f"{kind}, masked: rows {bad[:5]} (lengths {[int(lens[r]) for r in bad[:5]]})"


@pytest.mark.parametrize("rows,width", [(6, 4096), (6, 4090), (6, 8192), (300, 4096)])
@pytest.mark.parametrize("neg", ["normal", "ties", "zeros", "minus_zero", "inf"])
def test_held_rows_threshold_near_zero(gpu, rows, width, neg):
    """2048 positive keys give or take a few up to an eighth of the row, so that the search starts from zero or
    just does not; the others negative, tied, +0, -0 or -inf."""
    g = torch.Generator().manual_seed(width + rows)
    lens = torch.randint(3000, width + 1, (rows,), generator=g, dtype=torch.int32)
    lens[0], lens[1] = width, 2100
    x = -torch.rand(rows, width, generator=g)
    if neg == "ties":
        x = torch.full((rows, width), -0.25)
    elif neg in ("zeros", "minus_zero"):
        x = torch.where(torch.rand(rows, width, generator=g) < 0.05, x, 0.0 if neg == "zeros" else -0.0)
    elif neg == "inf":
        x = torch.where(torch.rand(rows, width, generator=g) < 0.5, x, -float("inf"))
    for r in range(rows):
        n = int(lens[r])
        off = [0, 1, -1, 70, -70, n // 16, -(n // 16), n // 8, -(n // 8)][r % 9]
        at = torch.randperm(n, generator=g)[:max(0, min(n, 2048 + off))]
        x[r, at] = torch.rand(at.numel(), generator=g) * (1e-30 if r % 2 else 3.0) + 1e-38
    pt = torch.randperm(width, generator=g).to(torch.int32).repeat(rows, 1).contiguous()
    cu = torch.arange(rows + 1, dtype=torch.int32, device=gpu)
    want = topk_radix(x.numpy(), None, lens.numpy(), pt.numpy(), width)
    got = hcu_ops.topk_transform(x.to(gpu), lens.to(gpu), pt.to(gpu), cu, max_splits=1).cpu().numpy()
    bad = [r for r in range(rows) if not np.array_equal(got[r], want[r])]
    assert not bad, f"rows {bad[:5]} (lengths {[int(lens[r]) for r in bad[:5]]})"
