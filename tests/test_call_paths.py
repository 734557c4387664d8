"""Which way a call takes on the host side: the plain C functions and the kernels behind them are for ordinary tensors in
an ordinary context; whoever traces, batches, differentiates or watches a call gets tensor operations or the registered
operator."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

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


def _same_bytes(got, want):
    for a, b in zip(got, want):
        assert a.dtype == b.dtype and a.shape == b.shape
        assert torch.equal(a.view(torch.uint8) if a.dtype is torch.float8_e4m3fn else a,
                           b.view(torch.uint8) if b.dtype is torch.float8_e4m3fn else b)


def test_quantize_of_fake_tensors():
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        k = torch.empty((1, 3, 64, 128), dtype=torch.bfloat16, device="cuda")
        k8, v8, k_scale, v_scale = quantize_kv_fp8(k, k)
    assert k8.shape == v8.shape == k.shape and k8.dtype is torch.float8_e4m3fn
    assert k_scale.shape == v_scale.shape == (3,) and k_scale.device.type == "cuda"


@pytest.mark.gpu
def test_quantize_under_transforms_matches_the_kernel():
    g = torch.Generator(device="cuda").manual_seed(4)
    k, v = (torch.randn((3, 1, 2, 48, 64), generator=g, device="cuda").to(torch.bfloat16) for _ in range(2))
    want = [quantize_kv_fp8(k[i], v[i]) for i in range(3)]
    batched = torch.vmap(quantize_kv_fp8)(k, v)
    for i in range(3):
        _same_bytes([t[i] for t in batched], want[i])
    _same_bytes(torch.compile(quantize_kv_fp8, backend="eager", fullgraph=True)(k[0], v[0]), want[0])
    _same_bytes(torch.jit.trace(quantize_kv_fp8, (k[1], v[1]), check_trace=False)(k[0], v[0]), want[0])
    import torch.autograd.forward_ad as forward_ad
    with forward_ad.dual_level():
        x = k[0].float()
        dual = quantize_kv_fp8(forward_ad.make_dual(x, x), v[0].float())
        scale, tangent = forward_ad.unpack_dual(dual[2])
        torch.testing.assert_close(tangent, scale)      # (the scale is linear in the largest magnitude)
    x = k[0].float().requires_grad_()
    assert quantize_kv_fp8(x, v[0].float())[2].requires_grad
    with torch.inference_mode():      # the usual way to serve: the kernel
        _same_bytes(quantize_kv_fp8(k[0], v[0]), want[0])
        assert attention_module._CALLS.quantizes(k[0], v[0])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_quantize_as_tensor_operations_gives_the_same_bytes(dtype):
    g = torch.Generator(device="cuda").manual_seed(5)
    k, v = (torch.randn((2, 5, 96, 64), generator=g, device="cuda").to(dtype) for _ in range(2))
    seen = []

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))
    with Watch():
        steps = quantize_kv_fp8(k, v)
    assert torch.ops.fsta.quantize_kv.default not in seen
    _same_bytes(quantize_kv_fp8(k, v), steps)
    with torch.device("cuda"):      # (a mode that watches calls from Python: the kernel)
        assert attention_module._CALLS.quantizes(k, v)
        _same_bytes(quantize_kv_fp8(k, v), steps)


@pytest.mark.gpu
def test_quantize_of_more_slices_than_a_grid_holds():
    g = torch.Generator(device="cuda").manual_seed(6)
    k = torch.randn((1 << 21, 1, 1, 16), generator=g, device="cuda").to(torch.bfloat16)
    part = [k[:1 << 20].contiguous(), k[1 << 20:].contiguous()]
    assert not attention_module._calls().quantizes(k, k) and attention_module._calls().quantizes(*part)
    k8, v8, k_scale, v_scale = quantize_kv_fp8(k, k)      # tensor operations
    a8, b8, a_scale, b_scale = quantize_kv_fp8(*part)     # the kernel
    _same_bytes((k8, k_scale), (torch.cat([a8.view(torch.uint8), b8.view(torch.uint8)]).view(k8.dtype), torch.cat([a_scale, b_scale])))
    _same_bytes((v8, v_scale), (k8, k_scale))


def test_shift_is_traceable_and_needs_no_library_on_the_host(monkeypatch):
    a_idx = torch.arange(12).view(2, 6) - 3
    l_idx = torch.arange(8).view(2, 4) - 1
    want = [torch.where(t >= 0, t + 100, t) for t in (a_idx, l_idx)]
    got = torch.compile(lambda a, l: shift_for_prefix(a, l, 100), backend="eager", fullgraph=True)(a_idx, l_idx)
    assert all(torch.equal(g, w) for g, w in zip(got, want))
    monkeypatch.setattr(attention_module, "_CALLS", None)

    def missing():
        raise ImportError("library asked for")
    monkeypatch.setattr(attention_module, "_calls", missing)
    assert all(torch.equal(g, w) for g, w in zip(shift_for_prefix(a_idx, l_idx, 100), want))
