"""Split KV of the fused relative-logit projection: underfilled grids cut each
256-row query tile's keys into chunks merged by a second pass.

The automatic plan on shapes that split (one to three sequences, masks, alignments,
both head sizes and r types) and forced chunks of two tiles, against the fp32 oracle
(16-bit rounding of P and of the output: 2e-2; LSE 1e-3), pruned against unpruned
launches bit for bit.
"""
import ctypes

import pytest
import torch

from inkling_fa4 import _abi, testing
from inkling_fa4._native import ops
from oracle import ref_rel_attn_rproj_with_lse


def _run(c, r, w, flags):
    return ops().fwd_rproj(c.q, c.k, c.v, r, w.t().contiguous(), c.cu_q, c.cu_k, c.max_q, c.max_k,
                           c.rel_extent, c.causal, c.window_left, c.scale, True, flags)


@pytest.mark.gpu
@pytest.mark.parametrize("lens_q,past,causal,window,bottom_right",
                         [([1000], [0], True, -1, False), ([257, 900], [0, 0], False, -1, False),
                          ([300, 5, 256], [700, 1500, 0], True, -1, True),
                          ([600, 128], [400, 900], True, 200, True)])
@pytest.mark.parametrize("head_dim,r_dtype,extent", [(128, torch.bfloat16, 300),
                                                     (64, torch.float32, 1024)])
def test_rproj_split(cuda, lens_q, past, causal, window, bottom_right, head_dim, r_dtype, extent):
    case = testing.make_case("rproj_split", lens_q, [a + b for a, b in zip(lens_q, past)], 4, 2,
                             head_dim, torch.bfloat16, seed=sum(lens_q), rel_extent=extent,
                             causal=causal, window_left=window, scale=0.1)
    g = torch.Generator().manual_seed(5)
    r = (0.3 * torch.randn(case.q.shape[0], 4, 16, generator=g)).to(r_dtype)
    w = 0.3 * torch.randn(16, extent, generator=g)
    print(f"rproj split: q {lens_q}, past {past}, causal {causal}, window {window}, d {head_dim}",
          flush=True)
    c, flag = case.to(cuda), _abi.IFA4_FLAG_BOTTOM_RIGHT if bottom_right else 0
    rd, wd = r.to(cuda), w.to(cuda)
    want_out, want_lse = ref_rel_attn_rproj_with_lse(
        case.q, case.k, case.v, r, w, case.cu_q, case.cu_k, case.scale, extent, causal=causal,
        window_left=case.window_or_none, bottom_right=bottom_right)
    for extra in (0, _abi.IFA4_FLAG_SPLIT_KV_2):
        out, lse = _run(c, rd, wd, flag | extra)
        torch.testing.assert_close(out.float().cpu(), want_out.float(), atol=2e-2, rtol=2e-2)
        torch.testing.assert_close(lse.cpu(), want_lse, atol=1e-3, rtol=0)
        full = _run(c, rd, wd, flag | extra | _abi.IFA4_FLAG_NO_PRUNE)
        assert torch.equal(full[0], out) and torch.equal(full[1], lse)


def _host_call(**kw):
    a = _abi.make_args(q=1 << 20, k=1 << 20, v=1 << 20, out=1 << 20, cu_seqlens_q=1 << 20,
                       cu_seqlens_k=1 << 20, q_stride_t=1024, q_stride_h=128, k_stride_t=256,
                       k_stride_h=128, v_stride_t=256, v_stride_h=128, out_stride_t=1024,
                       out_stride_h=128, n_heads=8, kv_heads=2, head_dim=128, rel_extent=128,
                       rel_width=128, causal=1, qkv_dtype=_abi.IFA4_BF16,
                       rel_dtype=_abi.IFA4_FP32, **kw)
    pr = _abi.Ifa4RelProj()
    pr.struct_size, pr.d_rel = ctypes.sizeof(_abi.Ifa4RelProj), 16
    pr.r, pr.wt, pr.r_stride_t, pr.r_stride_h = 1 << 20, 1 << 20, 128, 16
    return a, pr


# ranges of eight tiles on split; shorter ones were measured slower split
@pytest.mark.parametrize("batch,q,keys,window,splits", [
    (1, 512, 512, -1, True), (1, 448, 448, -1, False), (10, 200, 200, -1, False),
    (6, 400, 400, -1, False), (2, 60, 500, -1, True), (2, 60, 400, -1, False),
    (6, 400, 1900, 255, True), (6, 60, 1500, 255, False)])
def test_rproj_splits_long_ranges(batch, q, keys, window, splits):
    a, pr = _host_call(total_q=batch * q, total_k=batch * keys, batch=batch, max_seqlen_q=q,
                       max_seqlen_k=keys, window_left=window,
                       flags=_abi.IFA4_FLAG_BOTTOM_RIGHT if keys > q else 0)
    n = _abi.lib().ifa4_prefill_rproj_workspace_bytes(ctypes.byref(a), ctypes.byref(pr))
    assert (n > 0) == splits


def test_rproj_workspace_on_the_host():
    lib = _abi.lib()
    a, pr = _host_call(total_q=1000, total_k=1000, batch=1, max_seqlen_q=1000, max_seqlen_k=1000)
    n = lib.ifa4_prefill_rproj_workspace_bytes(ctypes.byref(a), ctypes.byref(pr))
    assert n > 0
    for ws, size in ((None, 0), (1 << 20, n - 1), ((1 << 20) + 16, n)):
        assert lib.ifa4_prefill_rproj_fwd_ws(ctypes.byref(a), ctypes.byref(pr), ws, size,
                                             None) == _abi.IFA4_EWORKSPACE
    pr.d_rel = 8  # refused as by ifa4_prefill_rproj_fwd
    assert lib.ifa4_prefill_rproj_workspace_bytes(ctypes.byref(a), ctypes.byref(pr)) == 0
    assert lib.ifa4_prefill_rproj_fwd_ws(ctypes.byref(a), ctypes.byref(pr), 1 << 20, n,
                                         None) == _abi.IFA4_EUNSUPPORTED
