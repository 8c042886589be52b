"""Prefill calls of a few queries per sequence over a cache: packed rows (the
query heads of a kv head share query tiles) and the merge of many chunks.

Rows pack up to 96 queries for groups of four (three quarters of the tiles); sizes sit
on both sides of that, at tile edges and with groups that do not divide the 128 rows
(3, 6, 12).  Within that a call packs by its work (the host test has both sides), and
always under the test flag of two-tile chunks, so every case runs both ways.
Everything is compared with the fp32 oracle (16-bit rounding of P and of the output:
2e-2; fp32 LSE: 1e-3), and pruned with unpruned launches bit for bit.
"""
import ctypes

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
    want_out, want_lse = ref_rel_attn_with_lse(
        case.q, case.k, case.v, case.rel, case.cu_q, case.cu_k, case.scale, case.rel_extent,
        causal=case.causal, window_left=case.window_or_none, bottom_right=bottom_right)
    rows = ~torch.isnan(want_out).any(-1)  # rows with a visible key
    runs = []
    for flags in (0, _abi.IFA4_FLAG_SPLIT_KV_2):
        out, lse = (x.cpu() for x in _run(c, flags, bottom_right))
        torch.testing.assert_close(out.float()[rows], want_out.float()[rows], atol=2e-2, rtol=2e-2)
        torch.testing.assert_close(lse.T[rows], want_lse.T[rows], atol=1e-3, rtol=0)
        assert bool((out[~rows] == 0).all()) and bool((lse.T[~rows] == float("-inf")).all())
        full = _run(c, flags | _abi.IFA4_FLAG_NO_PRUNE, bottom_right)
        assert torch.equal(full[0].cpu(), out) and torch.equal(full[1].cpu(), lse)
        runs.append((out, lse))
    torch.testing.assert_close(runs[1][1], runs[0][1], atol=1e-4, rtol=0)
    torch.testing.assert_close(runs[1][0].float(), runs[0][0].float(), atol=2e-2, rtol=2e-2)


def _host_args(batch, q, keys, hq, hkv, d=128, **kw):
    """A bottom-right call with a per-token bias, for the host-side queries."""
    fields = dict(q=1 << 20, k=1 << 20, v=1 << 20, out=1 << 20, cu_seqlens_q=1 << 20,
                  cu_seqlens_k=1 << 20, rel=1 << 20, q_stride_t=hq * d, q_stride_h=d,
                  k_stride_t=hkv * d, k_stride_h=d, v_stride_t=hkv * d, v_stride_h=d,
                  out_stride_t=hq * d, out_stride_h=d, rel_stride_t=hq * 1024, rel_stride_h=1024,
                  total_q=batch * q, total_k=batch * keys, batch=batch, n_heads=hq, kv_heads=hkv,
                  head_dim=d, rel_extent=1024, rel_width=1024, max_seqlen_q=q, max_seqlen_k=keys,
                  causal=1, flags=_abi.IFA4_FLAG_BOTTOM_RIGHT, qkv_dtype=_abi.IFA4_BF16,
                  rel_dtype=_abi.IFA4_BF16)
    fields.update(kw)
    return _abi.make_args(**fields)


# chunk slots of the plan without packed rows (per head) and with them, and which of
# the two the call takes: packed rows only where they were measured to pay
@pytest.mark.parametrize("batch,q,keys,hq,hkv,slots", [
    (64, 32, 532, 8, 2, 0),      # 512 workgroups of nine tiles, resident at once
    (64, 96, 596, 8, 2, 0),
    (16, 24, 24, 8, 2, 0),       # prompts without a cache
    (4, 64, 4064, 8, 2, 16),     # 32 workgroups in chunks of four tiles (packed: two, 32 slots)
    (12, 5, 8005, 8, 2, 21),     # packed: 24 workgroups in chunks of six (unpacked: 25, six)
    (64, 24, 2024, 8, 2, 4),     # packed: 128 in chunks of eight (unpacked: not split)
    (3, 40, 9040, 8, 2, 36),     # packed: 12 workgroups in chunks of four (unpacked: 21 of seven)
    (16, 32, 8032, 8, 2, 16),    # packed: 32 workgroups in chunks of eight (unpacked: four slots)
])
def test_packed_where_it_pays(batch, q, keys, hq, hkv, slots):
    a = _host_args(batch, q, keys, hq, hkv)
    n = _abi.lib().ifa4_prefill_workspace_bytes(a)
    assert n // (hq * batch * q * (128 + 1) * 4) == slots
    # the tile query reports the chunks that run
    tile = _abi.Ifa4Tile()
    assert _abi.lib().ifa4_prefill_tile(a, ctypes.byref(tile)) == _abi.IFA4_OK
    assert (-(-keys // tile.kv_chunk) if tile.kv_chunk else 0) == slots


def test_count_of_packed_tiles():
    # 200 x 8 queries over 308 keys: more workgroups than fit at once, packed, not split
    a = _host_args(200, 8, 308, 8, 2)
    assert _abi.lib().ifa4_prefill_workspace_bytes(a) == 0
    cu_q = (ctypes.c_int32 * 201)(*range(0, 201 * 8, 8))
    cu_k = (ctypes.c_int32 * 201)(*range(0, 201 * 308, 308))
    vis, tot = ctypes.c_int64(), ctypes.c_int64()
    assert _abi.lib().ifa4_prefill_count_tiles(a, cu_q, cu_k, ctypes.byref(vis),
                                               ctypes.byref(tot)) == _abi.IFA4_OK
    assert vis.value == tot.value == 200 * 2 * 5  # one tile per kv head, five KV tiles


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv", [(8, 2), (6, 2)])
def test_no_workspace_runs_the_same(cuda, hq, hkv):
    # a call that needs no workspace: ifa4_prefill_fwd and ifa4_prefill_fwd_ws bit for bit
    lens_q = [1 + i % 8 for i in range(200)]
    lens_k = [n + (i * 37) % 300 for i, n in enumerate(lens_q)]
    case = testing.make_case("no_ws", lens_q, lens_k, hq, hkv, 128, torch.bfloat16, seed=hq,
                             rel_table=False, rel_extent=200, rel_dtype=torch.bfloat16, scale=0.1)
    print(f"no workspace, {hq}/{hkv} heads", flush=True)
    c = case.to(cuda)
    out, lse = _run(c)
    got, got_lse = torch.empty_like(out), torch.empty_like(lse)
    a = _abi.make_args(
        q=c.q.data_ptr(), k=c.k.data_ptr(), v=c.v.data_ptr(), rel=c.rel.data_ptr(),
        out=got.data_ptr(), lse=got_lse.data_ptr(), cu_seqlens_q=c.cu_q.data_ptr(),
        cu_seqlens_k=c.cu_k.data_ptr(), q_stride_t=c.q.stride(0), q_stride_h=c.q.stride(1),
        k_stride_t=c.k.stride(0), k_stride_h=c.k.stride(1), v_stride_t=c.v.stride(0),
        v_stride_h=c.v.stride(1), rel_stride_t=c.rel.stride(0), rel_stride_h=c.rel.stride(1),
        out_stride_t=got.stride(0), out_stride_h=got.stride(1), lse_stride_h=got_lse.stride(0),
        total_q=sum(lens_q), total_k=sum(lens_k), batch=200, n_heads=hq, kv_heads=hkv,
        head_dim=128, rel_extent=200, rel_width=200, max_seqlen_q=c.max_q, max_seqlen_k=c.max_k,
        causal=1, softmax_scale=c.scale, flags=_abi.IFA4_FLAG_BOTTOM_RIGHT,
        qkv_dtype=_abi.IFA4_BF16, rel_dtype=_abi.IFA4_BF16)
    assert _abi.lib().ifa4_prefill_workspace_bytes(a) == 0
    stream = torch.cuda.current_stream().cuda_stream
    assert _abi.lib().ifa4_prefill_fwd(a, stream) == _abi.IFA4_OK
    torch.cuda.synchronize()
    assert torch.equal(got, out) and torch.equal(got_lse, lse)


# (hq, hkv, longest query length): groups 2, 3, 4, 6, 8, 12, 16, 64; the last two
# lengths of each are the edge of the rule and just past it
@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,top", [(4, 2, 64), (4, 2, 65), (6, 2, 84), (8, 2, 5), (8, 2, 96),
                                        (8, 2, 97), (12, 2, 63), (16, 2, 33), (24, 2, 8),
                                        (16, 1, 96), (64, 1, 3)])
def test_packed_groups_and_lengths(cuda, hq, hkv, top):
    lens_q = [1, top, max(1, top - 1), 2, 0]
    lens_k = [70, 700 + top, 1500, 2, 300]
    case = testing.make_case("packed", lens_q, lens_k, hq, hkv, 128, torch.bfloat16,
                             seed=10 * hq + top, rel_table=False, rel_extent=200,
                             rel_dtype=torch.bfloat16, scale=0.1)
    _check(case, cuda)


@pytest.mark.gpu
@pytest.mark.parametrize("head_dim,dtype", [(128, torch.bfloat16), (64, torch.float16)])
@pytest.mark.parametrize("rel_table,extent,rel_dtype", [(True, 128, torch.float32),
                                                        (True, 1024, torch.bfloat16),
                                                        (False, 300, torch.float16),
                                                        (False, 129, torch.float32)])
def test_packed_bias_forms(cuda, head_dim, dtype, rel_table, extent, rel_dtype):
    # a shared table of 1024 is too long for the packed tables' LDS: unpacked
    case = testing.make_case("packed_bias", [7, 31, 2], [900, 40, 1300], 8, 2, head_dim, dtype,
                             seed=extent, rel_table=rel_table, rel_extent=extent,
                             rel_width=extent + 3, rel_dtype=rel_dtype, scale=0.1)
    _check(case, cuda)


@pytest.mark.gpu
@pytest.mark.parametrize("causal,window,bottom_right", [(False, -1, True), (True, -1, False),
                                                        (False, 50, False), (True, 0, True),
                                                        (True, 63, True), (True, 200, True)])
def test_packed_masks(cuda, causal, window, bottom_right):
    # sequence 1 has more queries than keys: rows without a visible key bottom-right
    case = testing.make_case("packed_mask", [5, 60, 17], [640, 40, 2100], 8, 2, 128,
                             torch.bfloat16, seed=31, causal=causal, window_left=window,
                             scale=0.15)
    _check(case, cuda, bottom_right)


@pytest.mark.gpu
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("keys", [1300, 9000])
def test_merge_of_many_chunks(cuda, head_dim, keys):
    # few rows over tens of chunks: eight groups of chunks per row
    case = testing.make_case("many_chunks", [3, 20], [keys, keys // 3], 4, 4, head_dim,
                             torch.bfloat16, seed=keys, scale=0.1)
    _check(case, cuda)
