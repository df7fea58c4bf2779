"""prefill_indexer's logits slab: rows padded to whole lines when the workspace has room, unpadded in
one of exactly the keys' own size, at key counts of every remainder by 4 (which decide how the top-k may
load the scores); both against the oracle's selection on the same logits."""
import ctypes
import os

import numpy as np
import pytest
import torch

import hcu_ops
import workloads as wl
from oracle.topk_c import topk_radix

pytestmark = pytest.mark.gpu

P, I64, I, SZ = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int, ctypes.c_size_t


@pytest.mark.parametrize("rows,width,splits", [(9, 4096, 1), (9, 4097, 1), (12, 4098, 1), (12, 9003, 1), (3, 33001, 8),
                                               (3, 33003, 1), (2, 81921, 8)])
def test_padded_and_unpadded_slabs(gpu, rows, width, splits):
    lib = ctypes.CDLL(os.path.join(os.path.dirname(hcu_ops.__file__), "libdsa_indexer.so"))
    lib.dsa_last_error.restype = ctypes.c_char_p
    lib.dsa_prefill_indexer.argtypes = [P, P, I, I64, P, I64, P, I64, P, I64, P, I64, I64, I, I, P, SZ, P, P]
    lib.dsa_prefill_indexer_workspace_bytes.argtypes = [I64, I64, I64, I, I]
    lib.dsa_prefill_indexer_workspace_bytes.restype = SZ
    lib.dsa_topk_workspace_bytes.argtypes = [I64, I64, I, I]
    lib.dsa_topk_workspace_bytes.restype = SZ
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    case = wl.prefill_case(rows + width, rows, width - rows, heads=32)
    q8, w = hcu_ops.quant_q_fp8(case.q.to(gpu), case.w.to(gpu))
    kv, bt, lens, pt = case.kv.to(gpu), case.block_table.to(gpu), case.lens.to(gpu), case.slots().to(gpu)
    lg = hcu_ops.mqa_logits_prefill(q8, w, kv, bt, lens, width).cpu().numpy()
    want = topk_radix(lg, None, case.lens.numpy(), case.slots().numpy()[None, :], width,
                      cu_seqlens_q=np.array([0, rows], dtype=np.int32))
    full = lib.dsa_prefill_indexer_workspace_bytes(rows, width, rows, splits, cus)
    own = (rows * width * 4 + 255) // 256 * 256 + lib.dsa_topk_workspace_bytes(rows, width, splits, cus)
    assert own <= full
    for size in {own, full}:
        ws = torch.full((size,), 0x7F, dtype=torch.uint8, device=gpu)
        out = torch.empty(rows, 2048, dtype=torch.int32, device=gpu)
        st = lib.dsa_prefill_indexer(q8.data_ptr(), w.data_ptr(), 32, rows, kv.data_ptr(), kv.stride(0), bt.data_ptr(),
                                     bt.numel(), lens.data_ptr(), width, pt.data_ptr(), width, rows, splits, cus,
                                     ws.data_ptr(), size, out.data_ptr(), torch.cuda.current_stream().cuda_stream)
        assert st == 0, lib.dsa_last_error()
        assert np.array_equal(out.cpu().numpy(), want), f"workspace of {size} bytes (own {own}, full {full})"
