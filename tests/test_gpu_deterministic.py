"""Under torch.use_deterministic_algorithms, rows that no sequence covers come back as
torch fills uninitialised memory (NaN), in every prefill operator's outputs."""
import pytest
import torch

from inkling_fa4 import inkling_fa4_rel_attention, inkling_fa4_rel_attention_rproj, testing


@pytest.mark.gpu
@pytest.mark.parametrize("rproj", [False, True])
def test_uncovered_rows_are_filled(cuda, rproj):
    c = testing.make_case("fill", [33, 7], [33, 7], 4, 2, 64, torch.bfloat16, seed=1).to(cuda)
    cu = torch.tensor([0, 30, 35], dtype=torch.int32, device=cuda)  # of 40 rows
    r, w = torch.randn(40, 4, 16, device=cuda), torch.randn(16, 128, device=cuda)
    print(f"deterministic fill, projection {rproj}", flush=True)
    torch.use_deterministic_algorithms(True)
    try:
        if rproj:
            out, lse = inkling_fa4_rel_attention_rproj(c.q, c.k, c.v, r, w, cu, cu, 30, 30, 128,
                                                       return_lse=True)
        else:
            out, lse = inkling_fa4_rel_attention(c.q, c.k, c.v, c.rel, cu, cu, 30, 30, 128,
                                                 return_lse=True)
    finally:
        torch.use_deterministic_algorithms(False)
    assert bool(out[35:].isnan().all()) and bool(lse[:, 35:].isnan().all())
    assert not bool(out[:35].isnan().any()) and not bool(lse[:, :35].isnan().any())
