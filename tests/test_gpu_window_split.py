"""KV chunks of windowed prefill calls.

A query tile under a causal window sees a short run of keys wherever its queries
sit, so the call gets chunk slots for that run instead of the whole cache; a run cut
by the chunk grid at any alignment must find its slots.  Outputs against the fp32
oracle (16-bit rounding of P and of the output: 2e-2; fp32 LSE: 1e-3), pruned against
unpruned launches (which take slots for every chunk) bit for bit, and against chunks
of two tiles.
"""
import pytest
import torch

from inkling_fa4 import _abi, inkling_fa4_rel_attention, testing
from oracle import ref_rel_attn_with_lse


def _run(c, flags=0, bottom_right=True):
    return inkling_fa4_rel_attention(*c.args(), causal=c.causal, window_size=c.window_size,
                                     softmax_scale=c.scale, return_lse=True,
                                     bottom_right=bottom_right, _flags=flags)


def _check(case, dev, bottom_right=True):
    print(f"{case.name}: q {tuple(case.q.shape)}, k {tuple(case.k.shape)}, causal {case.causal}, "
          f"window {case.window_left}, bottom-right {bottom_right}", flush=True)
    c = case.to(dev)
    out, lse = _run(c, 0, bottom_right)
    want_out, want_lse = ref_rel_attn_with_lse(
        case.q, case.k, case.v, case.rel, case.cu_q, case.cu_k, case.scale, case.rel_extent,
        causal=case.causal, window_left=case.window_or_none, bottom_right=bottom_right)
    rows = ~torch.isnan(want_out).any(-1)  # rows with a visible key
    out, lse = out.cpu(), lse.cpu()
    torch.testing.assert_close(out.float()[rows], want_out.float()[rows], atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(lse.T[rows], want_lse.T[rows], atol=1e-3, rtol=0)
    assert bool((out[~rows] == 0).all()) and bool((lse.T[~rows] == float("-inf")).all())
    full = _run(c, _abi.IFA4_FLAG_NO_PRUNE, bottom_right)
    assert torch.equal(full[0].cpu(), out) and torch.equal(full[1].cpu(), lse)
    two, lse2 = _run(c, _abi.IFA4_FLAG_SPLIT_KV_2, bottom_right)
    torch.testing.assert_close(lse2.cpu(), lse, atol=1e-4, rtol=0)
    torch.testing.assert_close(two.float().cpu(), out.float(), atol=2e-2, rtol=2e-2)


@pytest.mark.gpu
@pytest.mark.parametrize("lens_q,past", [([1000], [777]), ([300, 511, 130], [4000, 64, 1]),
                                         ([128, 128], [1000, 1063])])
@pytest.mark.parametrize("window", [63, 511, 1000])
def test_windowed_chunks_cover_every_alignment(cuda, lens_q, past, window):
    case = testing.make_case("win_split", lens_q, [a + b for a, b in zip(lens_q, past)], 4, 2, 128,
                             torch.bfloat16, seed=window, window_left=window, rel_table=False,
                             rel_extent=200, rel_dtype=torch.bfloat16, scale=0.1)
    _check(case, cuda)


def _splits(batch, q, keys, hq, hkv, window, table):
    a = _abi.make_args(q=1 << 20, k=1 << 20, v=1 << 20, out=1 << 20, cu_seqlens_q=1 << 20,
                       cu_seqlens_k=1 << 20, rel=1 << 20, q_stride_t=hq * 128, q_stride_h=128,
                       k_stride_t=hkv * 128, k_stride_h=128, v_stride_t=hkv * 128,
                       v_stride_h=128, out_stride_t=hq * 128, out_stride_h=128,
                       rel_stride_t=0 if table else hq * 512, rel_stride_h=512,
                       total_q=batch * q, total_k=batch * keys, batch=batch, n_heads=hq,
                       kv_heads=hkv, head_dim=128, rel_extent=512, rel_width=512,
                       max_seqlen_q=q, max_seqlen_k=keys, causal=1, window_left=window,
                       flags=_abi.IFA4_FLAG_BOTTOM_RIGHT, qkv_dtype=_abi.IFA4_BF16,
                       rel_dtype=_abi.IFA4_BF16)
    return _abi.lib().ifa4_prefill_workspace_bytes(a) > 0


# short windows split where few workgroups make the merge pass cheap; (workgroups, tiles)
@pytest.mark.parametrize("batch,q,keys,hq,hkv,window,table,splits", [
    (1, 128, 4128, 8, 2, 255, False, True),     # 8, 7: 17.2 us without the split, 13.3 with it
    (1, 128, 4128, 8, 2, 127, False, True),     # 8, 5
    (1, 128, 4128, 8, 2, 63, False, False),     # 8, 4
    (1, 128, 4128, 8, 2, 127, True, False),     # 8, 5, shared table
    (1, 128, 4128, 8, 2, 255, True, True),      # 8, 7
    (2, 500, 4500, 4, 4, 255, False, True),     # 32, 7
    (2, 500, 4500, 8, 2, 255, False, False),    # 64, 7: 18.7 us without the split, 22.9 with it
    (1, 1000, 5000, 8, 2, 511, False, True),    # 64, 11
    (1, 1000, 5000, 8, 2, 511, True, False),    # 64, 11, shared table
    (20, 128, 6128, 8, 2, 1023, True, False),   # 160, 18, shared table
    (20, 128, 6128, 8, 2, 1023, False, True),   # 160, 18
])
def test_short_windows_split_small_grids(batch, q, keys, hq, hkv, window, table, splits):
    assert _splits(batch, q, keys, hq, hkv, window, table) == splits
