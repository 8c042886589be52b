"""Decode of short caches: one workgroup per (sequence, kv head), one launch.

The rule takes caches (or windows) of up to 20 steps of 32 keys, 32 steps from 128
segments on, 10 and 16 for groups above 8; sizes sit at step, wave and rule edges:
fewer steps than waves, a partial last step, one key, empty caches, sequences without
or with two queries.  Against the fp32 oracle (16-bit rounding of P and of the output:
2e-2; LSE 1e-3) on every cache format; a longer cache in max_seqlen_k sends the same
sequences through the two-pass kernels, which must agree (LSE 1e-4).
"""
import ctypes

import pytest
import torch

from inkling_fa4 import (_abi, inkling_fa4_rel_attention_decode, inkling_fa4_rel_attention_decode_paged,
                         testing)
from oracle import ref_rel_attn_with_lse


def _check(case, dev, bottom_right, kind="bf16", block=16):
    print(f"{case.name} {kind}: keys {case.cu_k.diff().tolist()[:6]}, Hq {case.q.shape[1]}, "
          f"Hkv {case.k.shape[1]}, d {case.q.shape[2]}, window {case.window_left}", flush=True)
    kw, ref, src = {}, case, case
    if "fp8" in kind:
        k8, v8, ks, vs, ref = testing.fp8_kv(case)
        kw = {"k_scale": ks, "v_scale": vs}
        src = testing.replace(case, k=k8, v=v8)
    want_out, want_lse = ref_rel_attn_with_lse(
        case.q, ref.k, ref.v, case.rel, case.cu_q, case.cu_k, case.scale, case.rel_extent,
        causal=case.causal, window_left=case.window_or_none, bottom_right=bottom_right)
    c = src.to(dev)
    common = dict(causal=case.causal, window_size=case.window_size, softmax_scale=case.scale,
                  return_lse=True, bottom_right=bottom_right, **kw)
    pk = None
    if "paged" in kind:
        pk = testing.paginate(src, block_size=block, extra_columns=200,
                              fill=0.0 if "fp8" in kind else float("nan")).to(dev)
    got = []
    for max_k in (c.max_k, max(c.max_k, 3000)):  # 3000: 94 steps, two passes (unless windowed)
        if pk is not None:
            got.append(inkling_fa4_rel_attention_decode_paged(
                c.q, pk.k_cache, pk.v_cache, c.rel, c.cu_q, pk.seqused_k, pk.block_table, 1,
                max_k, c.rel_extent, **common))
        else:
            got.append(inkling_fa4_rel_attention_decode(
                c.q, c.k, c.v, c.rel, c.cu_q, c.cu_k, 1, max_k, c.rel_extent, **common))
    rows = ~torch.isnan(want_out).any(-1)
    for out, lse in got:
        out, lse = out.cpu(), lse.cpu()
        torch.testing.assert_close(out.float()[rows], want_out.float()[rows], atol=2e-2, rtol=2e-2)
        torch.testing.assert_close(lse.T[rows], want_lse.T[rows], atol=1e-3, rtol=0)
        assert bool((out[~rows] == 0).all()) and bool((lse.T[~rows] == float("-inf")).all())
    torch.testing.assert_close(got[0][1], got[1][1], atol=1e-4, rtol=0)


LENS = [640, 1, 0, 31, 32, 33, 255, 256, 257, 513, 289, 2]


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["bf16", "fp8", "paged", "paged fp8"])
@pytest.mark.parametrize("hq,hkv,head_dim", [(8, 2, 128), (4, 4, 128), (8, 1, 64), (6, 2, 128),
                                             (12, 1, 128), (16, 1, 64)])
def test_short_caches(cuda, kind, hq, hkv, head_dim):
    lens = LENS if hq // hkv <= 8 else [min(n, 320) for n in LENS]
    case = testing.make_case("short", [1] * len(lens), lens, hq, hkv, head_dim, torch.bfloat16,
                             seed=hq + head_dim, causal=True, rel_table=False, rel_extent=100,
                             rel_dtype=torch.bfloat16, scale=0.1)
    _check(case, cuda, True, kind)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["bf16", "paged", "fp8"])
@pytest.mark.parametrize("causal,window,bottom_right", [(False, -1, False), (True, -1, False),
                                                        (True, 511, True), (True, 0, True),
                                                        (False, 300, True), (True, 600, True)])
def test_short_masks_and_windows(cuda, kind, causal, window, bottom_right):
    lens = [100, 640, 7] if window < 0 else [700, 2500, 33, 512, 1031]
    case = testing.make_case("short_win", [1] * len(lens), lens, 8, 2, 128, torch.float16,
                             seed=window + 9, causal=causal, window_left=window, rel_extent=512,
                             rel_dtype=torch.float32, scale=0.1)
    _check(case, cuda, bottom_right, kind, block=32)


@pytest.mark.gpu
@pytest.mark.parametrize("keys", [640, 1024])
def test_many_short_segments(cuda, keys):
    lens = [(keys * (i + 1)) // 70 for i in range(69)] + [keys]
    case = testing.make_case("short_many", [1] * 70, lens, 8, 2, 128, torch.bfloat16, seed=keys,
                             causal=False, scale=0.1)
    _check(case, cuda, False)


@pytest.mark.gpu
def test_short_rows_without_exactly_one_query(cuda):
    # cu_seqlens_q [0, 0, 2, 3]: no query, two queries, one: only the last is decoded
    case = testing.make_case("short_rows", [1, 1, 1], [50, 60, 70], 8, 2, 128, torch.bfloat16,
                             seed=3, causal=False, scale=0.1)
    c = case.to(cuda)
    cu_q = torch.tensor([0, 0, 2, 3], dtype=torch.int32, device=cuda)
    print("short decode with cu_seqlens_q = [0, 0, 2, 3]", flush=True)
    out, lse = inkling_fa4_rel_attention_decode(
        c.q, c.k, c.v, c.rel, cu_q, c.cu_k, 1, 70, c.rel_extent, causal=False,
        softmax_scale=c.scale, return_lse=True)
    ref = inkling_fa4_rel_attention_decode(
        c.q, c.k, c.v, c.rel, c.cu_q, c.cu_k, 1, 70, c.rel_extent, causal=False,
        softmax_scale=c.scale, return_lse=True)
    assert bool((out[:2] == 0).all()) and bool((lse[:, :2] == float("-inf")).all())
    assert torch.equal(out[2], ref[0][2]) and torch.equal(lse[:, 2], ref[1][:, 2])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_short_windows_keep_the_rounding_of_one_step(cuda, dtype):
    # The error against fp64 is that of rounding each 32-key step's weights, relative to the
    # step's largest, and the output to 16 bits: emulated here on the same numbers, so the two
    # differ by fp32 rounding only (1%: with one base for a wave's steps it was 3% above).
    lens = [520 + 83 * i for i in range(24)]
    case = testing.make_case("short_round", [1] * 24, lens, 8, 2, 128, dtype, seed=11,
                             window_left=511, rel_table=False, rel_extent=512, rel_dtype=dtype,
                             scale=1 / 128)
    print(f"rounding of windowed short decode, {dtype}", flush=True)
    c = case.to(cuda)
    out = inkling_fa4_rel_attention_decode(*c.args(), causal=True, window_size=(511, 0),
                                           softmax_scale=c.scale, bottom_right=True).cpu().double()
    want, rounded, ks = torch.zeros_like(out), torch.zeros_like(out), 0
    for b, n in enumerate(lens):
        lo = n - 512
        k, v = (x[ks + lo:ks + n].double() for x in (case.k, case.v))
        ks += n
        for h in range(8):
            x = k[:, h // 4] @ case.q[b, h].double() / 128 + case.rel[b, h].double().flip(0)
            p = torch.exp(x - x.max())
            want[b, h] = p @ v[:, h // 4] / p.sum()
            step = torch.arange(lo, n) // 32 - lo // 32  # steps start at multiples of 32 keys
            top = torch.full((int(step[-1]) + 1,), -torch.inf, dtype=torch.float64)
            top = top.scatter_reduce(0, step, p, "amax")[step]
            p16 = (p / top).to(dtype).double() * top
            rounded[b, h] = (p16 @ v[:, h // 4] / p.sum()).to(dtype).double()
    err, bound = (float((y - want).norm() / want.norm()) for y in (out, rounded))
    assert err < 1.01 * bound, (err, bound)


# (waves per workgroup, keys per wave) that the tile query reports: the one-launch form on
# both sides of its rule, and the persistent waves
@pytest.mark.parametrize("batch,keys,hq,hkv,window,waves,chunk", [
    (1, 512, 8, 2, -1, 8, 64), (1, 640, 8, 2, -1, 8, 96), (1, 641, 8, 2, -1, 1, 64),
    (64, 1024, 8, 2, -1, 8, 128), (64, 1025, 8, 2, -1, 1, 160), (63, 1024, 8, 2, -1, 1, 160),
    (1, 320, 16, 1, -1, 4, 96), (1, 321, 16, 1, -1, 1, 64), (24, 16384, 8, 2, 511, 8, 96),
    (24, 16384, 8, 2, 1023, 1, 896), (4, 0, 8, 2, -1, 8, 0)])
def test_decode_tile_reports_what_runs(batch, keys, hq, hkv, window, waves, chunk):
    a = _abi.make_args(q=1 << 20, k=1 << 20, v=1 << 20, out=1 << 20, cu_seqlens_q=1 << 20,
                       cu_seqlens_k=1 << 20, q_stride_t=hq * 128, q_stride_h=128,
                       k_stride_t=hkv * 128, k_stride_h=128, v_stride_t=hkv * 128,
                       v_stride_h=128, out_stride_t=hq * 128, out_stride_h=128, total_q=batch,
                       total_k=batch * keys, batch=batch, n_heads=hq, kv_heads=hkv, head_dim=128,
                       max_seqlen_q=1, max_seqlen_k=keys, causal=1, window_left=window,
                       flags=_abi.IFA4_FLAG_BOTTOM_RIGHT, qkv_dtype=_abi.IFA4_BF16,
                       rel_dtype=_abi.IFA4_BF16)
    tile = _abi.Ifa4Tile()
    assert _abi.lib().ifa4_decode_tile(a, ctypes.byref(tile)) == _abi.IFA4_OK
    assert (tile.block_k, tile.waves, tile.kv_chunk) == (32, waves, chunk)
