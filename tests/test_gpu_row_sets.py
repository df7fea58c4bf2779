"""Decode logits with the rows per CTA left to the library: groups whose rows divide into sets of 2, 3,
4, 6 and 8 either side of the page count from which the larger sets are taken, ragged lengths with an
empty request among them; bit-identical to two-row CTAs and within tolerance of the oracle."""
import pytest
import torch

import hcu_ops
import workloads as wl

from gpu_util import check_logits, check_mask, oracle_decode, oracle_q

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


def test_explicit_rows_per_cta_unchanged(gpu):
    """The counts a caller may ask for stay the same: six is the library's own choice only."""
    case = wl.decode_case(3, [300], group=6, heads=32)
    q8, w = hcu_ops.quant_q_fp8(case.q.to(gpu), case.w.to(gpu))
    with pytest.raises(RuntimeError, match="rows_per_cta"):
        hcu_ops.mqa_logits(q8.unsqueeze(1), case.kv.to(gpu), w, case.context_lens.to(gpu), case.block_table.to(gpu),
                           case.width, 6, rows_per_cta=6)
