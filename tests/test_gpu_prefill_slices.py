"""Prefill logits where the K slices of the launch can go wrong: keys ending on and either side of a
page and of the 255-page block-table stage, rows of any lengths (none, negative, past the width, not
ascending), and row counts that do not fill a CTA's eight rows; every logit against the oracle and
nothing written at or past a row's length."""
import numpy as np
import pytest
import torch

import hcu_ops
import workloads as wl
from oracle import indexer as O

from gpu_util import check_logits, kv_np, q_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads", [32, 64])
@pytest.mark.parametrize("rows,width,ragged", [(8, 1, False), (9, 64, False), (16, 65, True), (5, 4097, True),
                                               (7, 16320, False), (23, 16321, True), (13, 30016, True),
                                               (130, 2500, True)])
def test_prefill_slices(gpu, heads, rows, width, ragged):
    case = wl.prefill_case(11 * rows + width, rows, max(0, width - rows), heads=heads)
    lens = case.lens.clamp(max=width)
    if ragged:
        g = torch.Generator().manual_seed(rows + width)
        lens = torch.randint(-40, width + 60, (rows,), generator=g, dtype=torch.int32)
        lens[rows // 2] = width
    q8, w = hcu_ops.quant_q_fp8(case.q.to(gpu), case.w.to(gpu))
    kv, bt, lens_d = case.kv.to(gpu), case.block_table.to(gpu), lens.to(gpu)
    # poison the freed block the result is allocated from: what is not written keeps it
    at = torch.full((rows, width), 123.0, device=gpu).data_ptr()
    lg = hcu_ops.mqa_logits_prefill(q8, w, kv, bt, lens_d, width)
    assert lg.data_ptr() == at
    got = lg.cpu().numpy()
    rq8, rw = O.quant_q(q_bits(case.q), case.w.numpy())
    clamped = lens.clamp(0, width)
    ref, mag, dmag = O.mqa_logits_prefill(rq8, rw, kv_np(case.kv), case.block_table.numpy(), clamped.numpy(), width)
    for r in range(rows):
        n = int(clamped[r])
        check_logits(got[r, :n], ref[r, :n], mag[r, :n], dmag[r, :n], f"row {r}")
        assert (got[r, n:] == 123.0).all(), f"row {r}: written past its length"
