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
