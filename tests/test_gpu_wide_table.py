"""Decode logits of short requests in block tables far wider than they need (a serving loop's one graph has a
table as wide as the longest context): logits and every mask word against the oracle, the fused top-k
histogram, and the time such a launch takes beside one whose table is as wide as the context."""
import numpy as np
import pytest
import torch

import hcu_ops
from hcu_ops import _C
import workloads as wl
from oracle import indexer as O

from gpu_util import check_logits, check_mask, oracle_decode, oracle_q

pytestmark = pytest.mark.gpu

WIDE = 2048  # pages: 131,072 tokens


def _call(case, gpu, fused=False):
    q8, w = hcu_ops.quant_q_fp8(case.q.to(gpu), case.w.to(gpu))
    kv, lens, bt = case.kv.to(gpu), case.context_lens.to(gpu), case.block_table.to(gpu)
    # the blocks the results are allocated from hold no zeros
    del_me = [torch.full((case.rows, case.width), 7.0, device=gpu),
              torch.full((case.rows, case.width // 16), -1, dtype=torch.int16, device=gpu)]
    del del_me
    if fused:
        return _C.mqa_logits_hist(q8.unsqueeze(1), kv, w, lens, bt, case.width, case.group, 0, 0, lens)
    return hcu_ops.mqa_logits(q8.unsqueeze(1), kv, w, lens, bt, case.width, case.group)


# a group's pages below and above the 16 CTAs that zero its mask, one request and several, and more than 64
# groups (the block-wide assignment)
@pytest.mark.parametrize("heads", [32, 64])
@pytest.mark.parametrize("group,lens", [(1, [4096]), (2, [64, 65, 1, 0]), (4, [900, 0, 5000]), (6, [2100]),
                                        (6, [1000, 1040, 1080]), (8, [1]), (1, [70 + 13 * i for i in range(66)])])
def test_short_requests_in_a_wide_table(gpu, heads, group, lens):
    case = wl.decode_case(70 + group + len(lens), lens, group=group, heads=heads, bt_pages=WIDE)
    lg, mask = (x.cpu().numpy() for x in _call(case, gpu))
    ref, mag, dmag, _ = oracle_decode(case, *oracle_q(case))
    check_mask(mask, lg, ref, mag, case.context_lens.numpy(), "nonzero mask")
    for r in range(case.rows):
        n = int(case.context_lens[r])
        check_logits(lg[r, :n], ref[r, :n], mag[r, :n], dmag[r, :n], f"row {r}")


@pytest.mark.parametrize("group,lens", [(1, [4096, 2049, 3]), (2, [2300])])
def test_fused_histogram_in_a_wide_table(gpu, group, lens):
    case = wl.decode_case(90 + group, lens, group=group, heads=32, bt_pages=WIDE)
    lg, mask, zws = _call(case, gpu, fused=True)
    z, B = zws.cpu().numpy(), case.rows
    ref = O.pass1_hist(lg.cpu().numpy(), mask.cpu().numpy(), case.context_lens.numpy(), case.width)
    assert np.array_equal(z[:B * 4096], ref[:B * 4096]), "histogram differs"
    assert np.array_equal(z[2 * B * 4096:], ref[2 * B * 4096:]), "(positives, zeros) differ"


def _us(call, n=20, reps=9):
    call()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        keep = [call() for _ in range(n)]
    t = []
    for _ in range(reps):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        g.replay()
        b.record()
        torch.cuda.synchronize()
        t.append(a.elapsed_time(b) * 1e3 / n)
    del keep
    return min(t)


def test_wide_table_costs_little_time(gpu):
    """One request of 6 x 8192 tokens, 32 heads: 4.6 us in a table of its own width, 4.9 in one of 131,072 tokens
    (8.1 while every CTA of the launch read the query fragments and the pages fell to one XCD's CTAs)."""
    def timed(bt_pages):
        case = wl.decode_case(5, [8192 - 5], group=6, heads=32, bt_pages=bt_pages)
        q8, w = hcu_ops.quant_q_fp8(case.q.to(gpu), case.w.to(gpu))
        kv, lens, bt = case.kv.to(gpu), case.context_lens.to(gpu), case.block_table.to(gpu)
        return _us(lambda: hcu_ops.mqa_logits(q8.unsqueeze(1), kv, w, lens, bt, case.width, case.group))

    narrow, wide = timed(None), timed(WIDE)
    assert wide < 1.4 * narrow, f"{wide:.2f} us in a wide table, {narrow:.2f} in one as wide as the context"
