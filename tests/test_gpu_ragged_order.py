"""Workgroup order of ragged prefill batches: every (head count, batch) form of
the order runs each query tile exactly once.

The order depends on heads per kv head, kv heads and batch: units of up to four
heads whose query tiles go round 8, 4, 2 or 1 XCDs (8 / 1 .. 64 / 8 heads, with
batches that are and are not multiples of the XCDs), and the linear order
(one head per kv head, head counts that do not divide 8, under six sequences).  A tile
left out shows as rows that were never written, one run twice is harmless, a wrong
(sequence, head) as wrong rows: outputs against the fp32 oracle, 16-bit rounding
of P and of the output (2e-2) and the fp32 LSE (1e-3) as in the other prefill tests.
"""
import pytest
import torch

from inkling_fa4 import inkling_fa4_rel_attention, testing
from oracle import ref_rel_attn_with_lse


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,batch", [(4, 1, 8), (8, 2, 9), (8, 2, 8), (8, 2, 5), (8, 1, 7),
                                          (16, 4, 7), (32, 4, 6), (64, 16, 6), (64, 8, 7),
                                          (6, 3, 7), (8, 4, 6), (12, 2, 6), (10, 2, 7), (4, 4, 8),
                                          (8, 8, 9)])
def test_ragged_order_runs_every_tile(cuda, hq, hkv, batch):
    lens = [300, 33, 1, 129, 0, 257, 128, 64, 190][:batch]
    case = testing.make_case("order", lens, lens, hq, hkv, 64, torch.bfloat16, seed=hq + batch,
                             scale=0.2)
    print(f"ragged order, {hq}/{hkv} heads, {batch} sequences", flush=True)
    c = case.to(cuda)
    # a freed block of NaN is what the allocator hands out for the outputs
    torch.full((case.q.numel() + 4 * hq * sum(lens),), float("nan"), device=cuda,
               dtype=torch.bfloat16)
    out, lse = inkling_fa4_rel_attention(*c.args(), softmax_scale=c.scale, return_lse=True)
    want_out, want_lse = ref_rel_attn_with_lse(case.q, case.k, case.v, case.rel, case.cu_q,
                                               case.cu_k, case.scale, case.rel_extent)
    torch.testing.assert_close(out.float().cpu(), want_out.float(), atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(lse.cpu(), want_lse, atol=1e-3, rtol=0)
