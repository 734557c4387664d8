"""Which way a call takes on the host side: the plain C functions and the kernels behind them are for ordinary tensors in
an ordinary context; whoever traces, batches, differentiates or watches a call gets tensor operations or the registered
operator."""
import pytest
import torch

from fstattention_amd import attention as attention_module
from fstattention_amd import (create_fst_attention_kernel_inputs, fst_attention, quantize_kv_fp8, shift_for_prefix, trees)


class _NoOperators:
    """Stands in for ``torch.ops.fsta``: a call that reaches it has missed the C function."""

    def __getattr__(self, name):
        raise AssertionError(f"operator {name} called")


def _call_inputs():
    parent = trees.medusa_parents(n=64, seed=5)
    lineage, level = trees.lineage_from_parents(parent)
    max_anc = trees.required_max_ancestors(parent, 64)
    a_idx, packed, l_idx = create_fst_attention_kernel_inputs(lineage.cuda(), level.cuda(), 64, max_anc, want_bool_mask=False)
    g = torch.Generator(device="cuda").manual_seed(3)
    q, k, v = (torch.randn((1, 2, 64, 64), generator=g, device="cuda").to(torch.bfloat16) for _ in range(3))
    return (q, k, v, a_idx, packed, l_idx, 0.125), {"BLOCK_M": 64, "MAX_ANCESTORS": max_anc}


@pytest.mark.gpu
def test_inference_mode_takes_the_c_function(monkeypatch):
    args, options = _call_inputs()
    want = fst_attention(*args, **options)
    monkeypatch.setattr(attention_module, "_OPS", _NoOperators())
    with torch.inference_mode():
        got = fst_attention(*args, **options)
        assert got.is_inference()
    assert torch.equal(got, want)


@pytest.mark.gpu
def test_a_profiler_sees_the_call():
    args, options = _call_inputs()
    want = fst_attention(*args, **options)
    for shapes in (False, True):
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU], record_shapes=shapes) as prof:
            got = fst_attention(*args, **options)
        assert torch.equal(got, want)
        seen = [e for e in prof.events() if e.name == "fsta::attention_fwd"]
        assert len(seen) == 1
        assert not shapes or [list(s) for s in seen[0].input_shapes[:3]] == [[1, 2, 64, 64]] * 3
