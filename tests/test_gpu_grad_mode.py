"""The operators have no backward: outputs never require a gradient, whatever the
inputs and the grad mode."""
import pytest
import torch

from inkling_fa4 import (inkling_fa4_rel_attention, inkling_fa4_rel_attention_decode,
                         inkling_fa4_rel_attention_rproj, testing)


@pytest.mark.gpu
@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("which", range(5))
def test_outputs_never_require_grad(cuda, grad, which):
    c = testing.make_case("grad", [33, 5], [33, 5], 4, 2, 64, torch.bfloat16, seed=1).to(cuda)
    d = testing.make_case("grad_dec", [1, 1], [33, 5], 4, 2, 64, torch.bfloat16, seed=1).to(cuda)
    r, w = torch.randn(38, 4, 16, device=cuda), torch.randn(16, 128, device=cuda)
    print(f"grad mode {grad}, input {which} requires grad", flush=True)
    with torch.set_grad_enabled(grad):
        if which < 4:
            for case in (c, d):
                t = [case.q, case.k, case.v, case.rel]
                t[which] = t[which].detach().clone().requires_grad_()
                op = inkling_fa4_rel_attention if case is c else inkling_fa4_rel_attention_decode
                out, lse = op(*t, *case.args()[4:], return_lse=True)
                assert not out.requires_grad and not lse.requires_grad
                assert torch.equal(out, op(*case.args()))
        out = inkling_fa4_rel_attention_rproj(c.q, c.k, c.v, r, w.requires_grad_(which == 4),
                                              *c.args()[4:])
        assert not out.requires_grad


@pytest.mark.parametrize("grad", [True, False])
def test_other_objects_are_refused_by_the_operator(grad):
    c = testing.make_case("none", [3], [3], 4, 2, 64, torch.bfloat16, seed=1)
    with torch.set_grad_enabled(grad), pytest.raises(RuntimeError):
        inkling_fa4_rel_attention(c.q, c.k, c.v, None, *c.args()[4:])
