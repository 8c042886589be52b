"""Workgroup order of ragged prefill batches: every form of the order runs each
query tile exactly once.

The form depends on heads per kv head, kv heads, batch and on how much work the call
has (csrc/workgroup_order.h): FORMS reach units of four heads whose query tiles go
round 8, 4, 2 or 1 XCDs, the turned linear order and the plain one, for the plain kernel
and the fused projection; the host test beside them checks that they do.  A tile left
out shows as rows that were never written, one run twice is harmless, a wrong
(sequence, head) as wrong rows: outputs against the fp32 oracle, 16-bit rounding of P
and of the output (2e-2) and the fp32 LSE (1e-3) as in the other prefill tests.
"""
import pytest
import torch

from inkling_fa4 import (_abi, inkling_fa4_rel_attention, inkling_fa4_rel_attention_rproj,
                         testing)
from oracle import ref_rel_attn_rproj_with_lse, ref_rel_attn_with_lse
from test_workgroup_order import check_order, lib  # noqa: F401 (fixture)

# hq, hkv, batch, fused projection, XCDs of a unit (0: linear), turned
FORMS = [(4, 1, 112, False, 8, 1), (4, 1, 109, False, 8, 1), (8, 2, 56, False, 4, 1),
         (8, 2, 59, False, 4, 1), (8, 1, 54, False, 4, 1), (16, 4, 31, False, 2, 1),
         (32, 8, 16, False, 1, 1), (64, 8, 9, False, 1, 1), (4, 4, 110, False, 0, 1),
         (8, 4, 56, False, 0, 1), (6, 3, 72, False, 0, 1),
         (6, 3, 71, False, 0, 0), (8, 4, 55, False, 0, 0), (8, 2, 60, True, 4, 1),
         (16, 4, 33, True, 2, 1), (8, 4, 64, True, 0, 1), (6, 3, 73, True, 0, 0)]


def _lens(batch, proj):
    # 0 .. 190 tokens, 0 .. 380 for the projection's longer query tiles: up to two tiles
    return [(1 + proj) * ((37 * i) % 191) for i in range(1, batch + 1)]


@pytest.mark.parametrize("hq,hkv,batch,proj,xcds,turn", FORMS)
def test_forms_are_reached(lib, hq, hkv, batch, proj, xcds, turn):  # noqa: F811
    lens = _lens(batch, proj)
    rows, slots = (256, 256) if proj else (128, 512)
    assert 4 * sum(lens) < 3 * batch * max(lens)
    live = (sum(lens) // rows + batch // 2) * hq
    form = check_order(lib, hq, hq // hkv, batch, ragged=2, live=live, slots=slots, proj=int(proj))
    assert (form["xcds"], form["turn"], form["pair_heads"]) == (xcds, turn, 0)
    a = _abi.make_args(q=1 << 20, k=1 << 20, v=1 << 20, out=1 << 20, cu_seqlens_q=1 << 20,
                       cu_seqlens_k=1 << 20, rel=1 << 20, q_stride_t=64 * hq, q_stride_h=64,
                       k_stride_t=64 * hkv, k_stride_h=64, v_stride_t=64 * hkv, v_stride_h=64,
                       out_stride_t=64 * hq, out_stride_h=64, total_q=sum(lens),
                       total_k=sum(lens), batch=batch, n_heads=hq, kv_heads=hkv, head_dim=64,
                       rel_extent=128, rel_width=128, max_seqlen_q=max(lens),
                       max_seqlen_k=max(lens), causal=1, qkv_dtype=_abi.IFA4_BF16,
                       rel_dtype=_abi.IFA4_FP32)
    if proj:
        assert hq * batch >= slots  # one query tile each: not split
    else:  # not split into KV chunks, which keep the order of equal lengths
        assert _abi.lib().ifa4_prefill_workspace_bytes(a) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,batch,proj,xcds,turn", FORMS)
def test_ragged_order_forms(cuda, hq, hkv, batch, proj, xcds, turn):
    lens = _lens(batch, proj)
    case = testing.make_case("order", lens, lens, hq, hkv, 64, torch.bfloat16, seed=hq + batch,
                             scale=0.2)
    print(f"ragged order, {hq}/{hkv} heads, {batch} sequences, projection {proj}", flush=True)
    c = case.to(cuda)
    # a freed block of NaN is what the allocator hands out for the outputs
    torch.full((case.q.numel() + 4 * hq * sum(lens),), float("nan"), device=cuda,
               dtype=torch.bfloat16)
    if proj:
        g = torch.Generator().manual_seed(batch)
        r = 0.3 * torch.randn(case.q.shape[0], hq, 16, generator=g)
        w = 0.3 * torch.randn(16, 128, generator=g)
        out, lse = inkling_fa4_rel_attention_rproj(
            c.q, c.k, c.v, r.to(cuda), w.to(cuda), c.cu_q, c.cu_k, c.max_q, c.max_k, 128,
            softmax_scale=c.scale, return_lse=True)
        want_out, want_lse = ref_rel_attn_rproj_with_lse(case.q, case.k, case.v, r, w, case.cu_q,
                                                         case.cu_k, case.scale, 128)
    else:
        out, lse = inkling_fa4_rel_attention(*c.args(), softmax_scale=c.scale, return_lse=True)
        want_out, want_lse = ref_rel_attn_with_lse(case.q, case.k, case.v, case.rel, case.cu_q,
                                                   case.cu_k, case.scale, case.rel_extent)
    torch.testing.assert_close(out.float().cpu(), want_out.float(), atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(lse.cpu(), want_lse, atol=1e-3, rtol=0)


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
