"""Decode logits with the rows per CTA left to the library: groups whose rows divide into sets of 2, 3,
4, 6 and 8 either side of the page count from which the larger sets are taken, ragged lengths with an
empty request among them, CTAs of one page and of many; bit-identical to two-row CTAs and within tolerance
of the oracle."""
import numpy as np
import pytest
import torch

import hcu_ops
import workloads as wl
from oracle import indexer as O

from gpu_util import check_logits, check_mask, kv_np, oracle_decode, oracle_q, q_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads", [32, 64])
@pytest.mark.parametrize("group,bt_pages", [(2, 700), (4, 40), (4, 700), (6, 700), (8, 600), (10, 700), (12, 700),
                                             (18, 700)])
def test_open_rows_per_cta(gpu, heads, group, bt_pages):
    case = wl.decode_case(40 + group, [2100, 0, 63, 1], group=group, heads=heads, bt_pages=bt_pages)
    q8, w = hcu_ops.quant_q_fp8(case.q.to(gpu), case.w.to(gpu))
    kv, lens, bt = case.kv.to(gpu), case.context_lens.to(gpu), case.block_table.to(gpu)
    assert hcu_ops.mqa_logits_supported(q8.unsqueeze(1), kv, w, group, lens, bt, case.width)

    def call(rpc):
        lg, mask = hcu_ops.mqa_logits(q8.unsqueeze(1), kv, w, lens, bt, case.width, group, rows_per_cta=rpc)
        return lg.cpu().numpy(), mask.cpu().numpy()

    lg, mask = call(None)
    lg2, mask2 = call(2)
    assert (mask == mask2).all()
    ref, mag, dmag, _ = oracle_decode(case, *oracle_q(case))
    check_mask(mask, lg, ref, mag, case.context_lens.numpy(), "nonzero mask")
    for r in range(case.rows):
        n = int(case.context_lens[r])
        assert (lg[r, :n].view("u4") == lg2[r, :n].view("u4")).all(), f"row {r}: differs from two-row CTAs"
        check_logits(lg[r, :n], ref[r, :n], mag[r, :n], dmag[r, :n], f"row {r}")


POOL = 97  # distinct K pages of the long contexts, so that the oracle scores each once


@pytest.mark.parametrize("heads", [32, 64])
@pytest.mark.parametrize("group", [4, 6, 8, 12])
def test_row_sets_over_many_pages(gpu, heads, group):
    """Contexts of 40-65K tokens: the CTAs resident at once (at most 24 waves a CU, so 6144 / rows of them) stream
    3 to 11 pages each, odd and even counts, first and last pages partly filled."""
    g = torch.Generator().manual_seed(group)
    ctx = [64 * 1000 + 1, 63000, 40037, 64 * 900, 51234, 64 * 1015 - 1]
    req, cap = len(ctx), 1016
    kv = wl.build_kv(g, POOL)
    bt = torch.randint(0, POOL, (req, cap), generator=g, dtype=torch.int32)
    rows = req * group
    lens = torch.tensor([c + j for c in ctx for j in range(-group + 1, 1)], dtype=torch.int32)
    q = torch.randn(rows, heads, 128, generator=g).to(torch.bfloat16)
    w = torch.randn(rows, heads, generator=g) * 0.3
    pages = sum((c + 63) // 64 for c in ctx)
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    assert pages >= 3 * cus * 24 // (4 if group == 4 else 6) // (1 if heads == 32 else 2), "CTAs of a page or two"
    q8, w8 = hcu_ops.quant_q_fp8(q.to(gpu), w.to(gpu))
    kvd, btd, lensd = kv.to(gpu), bt.repeat_interleave(group, 0).contiguous().to(gpu), lens.to(gpu)

    def call(rpc):
        return hcu_ops.mqa_logits(q8.unsqueeze(1), kvd, w8, lensd, btd, cap * 64, group, rows_per_cta=rpc)

    lg, mask = call(None)
    lg2, mask2 = call(2)
    assert torch.equal(mask, mask2)
    lg, lg2 = lg.cpu().numpy(), lg2.cpu().numpy()
    rq8, rw = O.quant_q(q_bits(q), w.numpy())
    ref, mag, dmag, _ = O.mqa_logits_decode(rq8, rw, kv_np(kv), np.full(rows, POOL * 64, dtype=np.int32),
                                            np.arange(POOL, dtype=np.int32)[None, :].repeat(rows, 0), rows, POOL * 64)
    bits = O.unpack_mask(mask.cpu().numpy(), cap * 64)
    for r in range(rows):
        n = int(lens[r])
        at = (bt[r // group].numpy()[:, None].astype(np.int64) * 64 + np.arange(64)).reshape(-1)[:n]
        assert (lg[r, :n].view("u4") == lg2[r, :n].view("u4")).all(), f"row {r}: differs from two-row CTAs"
        check_logits(lg[r, :n], ref[r, at], mag[r, at], dmag[r, at], f"row {r}")
        assert np.array_equal(bits[r, :n], lg[r, :n].view("u4") != 0) and not bits[r, n:].any(), f"row {r}: mask"


def test_explicit_rows_per_cta_unchanged(gpu):
    """The counts a caller may ask for stay the same: six is the library's own choice only."""
    case = wl.decode_case(3, [300], group=6, heads=32)
    q8, w = hcu_ops.quant_q_fp8(case.q.to(gpu), case.w.to(gpu))
    with pytest.raises(RuntimeError, match="rows_per_cta"):
        hcu_ops.mqa_logits(q8.unsqueeze(1), case.kv.to(gpu), w, case.context_lens.to(gpu), case.block_table.to(gpu),
                           case.width, 6, rows_per_cta=6)
