"""Prefill logits where the K slices of the launch can go wrong: keys ending on and either side of a
page, rows of any lengths (none, negative, past the width, not ascending), and row counts that do not fill
a CTA's eight rows, in slices of one page or two, every logit against the oracle; and launches whose slices
run from 3 pages to the 255 of the block-table stage, sampled rows against the oracle.  Nothing is written at or past a
row's length."""
import ctypes
import os

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


POISON = 2.0 ** 100
POOL = 61  # distinct K pages of the wide launches, so that the oracle scores each once


@pytest.mark.parametrize("heads,rows,width,least", [(32, 1100, 21000, 12), (64, 1100, 21000, 12), (32, 37, 60064, 3),
                                                    (64, 131, 33000, 4), (32, 2051, 16385, 12), (64, 2061, 130560, 255),
                                                    (64, 2053, 131073, 200), (32, 2061, 130560, 30)])
def test_prefill_long_slices(gpu, heads, rows, width, least):
    """Slices of `least` pages or more: the page loop past its first two slots, the last slice short, rows that end
    within a slice or before it, a last group of 3 to 5 rows."""
    lib = ctypes.CDLL(os.path.join(os.path.dirname(hcu_ops.__file__), "libdsa_indexer.so"))
    lib.dsa_prefill_slice_pages.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    assert lib.dsa_prefill_slice_pages(heads, rows, width, cus) >= least and rows % 8
    g = torch.Generator().manual_seed(rows + width)
    kv = wl.build_kv(g, POOL)
    bt = torch.randint(0, POOL, ((width + 63) // 64,), generator=g, dtype=torch.int32)
    lens = torch.randint(-40, width + 60, (rows,), generator=g, dtype=torch.int32)
    lens[rows // 2], lens[rows - 1], lens[rows - 2] = width, width, 2 * 64 * least + 1
    q = torch.randn(rows, heads, 128, generator=g).to(torch.bfloat16)
    w = torch.randn(rows, heads, generator=g) * 0.3
    q8, w8 = hcu_ops.quant_q_fp8(q.to(gpu), w.to(gpu))
    at = torch.full((rows, width), POISON, device=gpu).data_ptr()
    lg = hcu_ops.mqa_logits_prefill(q8, w8, kv.to(gpu), bt.to(gpu), lens.to(gpu), width)
    assert lg.data_ptr() == at
    clamped = lens.clamp(0, width)
    past = torch.arange(width, device=gpu)[None, :] >= clamped.to(gpu)[:, None]
    for r in range(0, rows, 256):
        assert ((lg[r:r + 256] == POISON) == past[r:r + 256]).all(), "written past a row's length, or not up to it"
    some = sorted({0, 7, 8, rows // 2, *range(rows - 5, rows), *torch.randint(0, rows, (8,), generator=g).tolist()})
    rq8, rw = O.quant_q(q_bits(q[some]), w[some].numpy())
    ref, mag, dmag = O.mqa_logits_prefill(rq8, rw, kv_np(kv), np.arange(POOL, dtype=np.int32),
                                          np.full(len(some), POOL * 64, dtype=np.int32), POOL * 64)
    tok = (bt.numpy()[:, None].astype(np.int64) * 64 + np.arange(64)).reshape(-1)
    for i, r in enumerate(some):
        n = int(clamped[r])
        t = tok[:n]
        check_logits(lg[r, :n].cpu().numpy(), ref[i, t], mag[i, t], dmag[i, t], f"row {r}")
