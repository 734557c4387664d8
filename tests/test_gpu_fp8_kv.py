"""8-bit K/V storage (float8_e4m3fn rows + one scale per (batch, head) slice) against the dense oracle.

The oracle is the dense-masked attention on the DEQUANTISED keys and values (``k8 * k_scale``,
``v8 * v_scale``, formed in float64 on the host): the kernel widens the stored bytes exactly, so the
tolerance is the one of the 16-bit kernels (2e-3, asserted on the float32 output).
"""
import math

import numpy as np
import pytest
import torch

from fstattention_amd import fst_attention, quantize_kv_fp8, shift_for_prefix, trees
from helpers import assert_close, dense_oracle, oracle_inputs, rand_qkv

pytestmark = pytest.mark.gpu


def run_fp8(parent, block_m, z, h, d, dtype, seed, prefix=0, scales=True, spread=1.0):
    n = len(parent)
    a_idx, a_mask, l_idx, max_anc = oracle_inputs(parent, block_m)
    nq = a_idx.shape[0] * block_m
    q, k, v = rand_qkv(z, h, nq, nq + prefix, d, dtype, seed)
    if spread != 1.0:      # slices of very different magnitude: the per-slice scales must be honoured
        factor = torch.logspace(0, math.log10(spread), z * h).view(z, h, 1, 1)
        k, v = (k.float() * factor).to(dtype), (v.float() / factor).to(dtype)
    k8, v8, k_scale, v_scale = quantize_kv_fp8(k, v)
    if not scales:         # N(0,1) values rounded to the 8-bit format and used as they are
        k_scale = v_scale = None
        k8, v8 = k.to(torch.float8_e4m3fn), v.to(torch.float8_e4m3fn)
        k_deq, v_deq = k8.double(), v8.double()
    else:
        k_deq = k8.double() * k_scale.double().view(z, h, 1, 1)
        v_deq = v8.double() * v_scale.double().view(z, h, 1, 1)
    scale = 1.0 / math.sqrt(d)
    want, want_lse = dense_oracle(q.double(), k_deq, v_deq, parent, scale, prefix=prefix, nq_pad=nq - n)
    if prefix:
        a_idx, l_idx = shift_for_prefix(a_idx, l_idx, prefix)
    dev = lambda t: None if t is None else t.cuda()
    o, lse = fst_attention(q.cuda(), k8.cuda(), v8.cuda(), a_idx.cuda(), a_mask.cuda(), l_idx.cuda(), scale,
                           BLOCK_M=block_m, MAX_ANCESTORS=max_anc, out_dtype=torch.float32, return_lse=True,
                           k_scale=dev(k_scale), v_scale=dev(v_scale))
    assert_close(o, want, dtype, f"fp8 K/V n={n} m={block_m} d={d} {dtype} prefix={prefix}")
    torch.testing.assert_close(lse.cpu().double().view(z, h, nq), want_lse, atol=2e-3, rtol=2e-3)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("block_m", [32, 64, 128])
def test_shapes(block_m, d, dtype):
    parent = trees.random_recursive_parents(300, 40 + block_m + d, window=48)      # ragged last block
    run_fp8(parent, block_m, 2, 3, d, dtype, 7)


@pytest.mark.parametrize("index", [2, 3, 4])
def test_benchmark_trees_full_size(index):
    cfg = trees.config(index)
    run_fp8(cfg.parent, cfg.block_m, cfg.batch, cfg.heads, cfg.head_dim, torch.bfloat16, cfg.tensor_seed)


def test_config5_head_subset():
    cfg = trees.config(5)
    run_fp8(cfg.parent, cfg.block_m, 2, 4, cfg.head_dim, torch.bfloat16, cfg.tensor_seed)


@pytest.mark.parametrize("prefix", [100, 64, 7])
def test_shared_prefix(prefix):
    parent = trees.random_recursive_parents(200, 3, window=32)
    run_fp8(parent, 64, 1, 4, 128, torch.bfloat16, 9, prefix=prefix)


@pytest.mark.parametrize("nodes,block_m,d,z,h,prefix", [(1, 32, 128, 1, 1, 1), (40, 64, 64, 1, 2, 287), (70, 32, 128, 1, 3, 2050),
                                                        (129, 64, 128, 2, 60, 600), (30, 64, 64, 1, 8, 5000)])
def test_prefix_remainders_and_runs(nodes, block_m, d, z, h, prefix):
    """Remainders of tiles and waves, several runs of keys, more workgroups than CUs."""
    parent = trees.random_recursive_parents(nodes, prefix, window=24)
    run_fp8(parent, block_m, z, h, d, torch.bfloat16 if nodes % 2 else torch.float16, 15, prefix=prefix)


@pytest.mark.parametrize("nodes,block_m,d,h,prefix,kernel", [
    (512, 64, 128, 2, 300, "cache"), (513, 64, 128, 2, 300, "cache"), (700, 32, 64, 30, 33, "cache"), (1500, 128, 64, 3, 2050, "cache"),
    (1025, 64, 64, 17, 99, "mfma16"), (1025, 64, 64, 17, 100, "cache"), (650, 128, 128, 26, 699, "mfma16"), (650, 128, 128, 26, 700, "cache"),
    (600, 128, 128, 25, 100, "cache")])
def test_long_trees_behind_a_prefix(nodes, block_m, d, h, prefix, kernel):
    """More than 512 rows: both kernels, on both sides of the rule that chooses."""
    from fstattention_amd import _lib
    parent = trees.random_recursive_parents(nodes, prefix, window=64)
    run_fp8(parent, block_m, 1, h, d, torch.bfloat16 if nodes % 2 else torch.float16, 16, prefix=prefix)
    assert f"attn_{kernel}_kernel" in _lib.load().fsta_last_attention_kernel().decode()


def test_per_slice_scales_and_no_scales():
    parent = trees.medusa_parents(n=256, seed=77)
    run_fp8(parent, 64, 2, 4, 128, torch.bfloat16, 11, spread=64.0)
    run_fp8(parent, 64, 2, 4, 64, torch.float16, 12, scales=False)


def test_short_and_single_tile_lists():
    bushy = np.maximum((np.arange(90) - 1) // 3, -1).astype(np.int64)
    bushy[0] = -1
    run_fp8(bushy, 32, 1, 2, 128, torch.bfloat16, 13)
    run_fp8(np.full(40, -1, dtype=np.int64), 32, 1, 2, 64, torch.bfloat16, 14)       # roots only: no ancestor tile


@pytest.mark.parametrize("keys,d,dtype", [(1, 64, torch.bfloat16), (128, 128, torch.bfloat16), (129, 128, torch.float16),
                                          (512, 128, torch.bfloat16), (513, 128, torch.bfloat16), (1023, 64, torch.float16),
                                          (512, 128, torch.float32), (515, 128, torch.float32), (2100, 64, torch.float32),
                                          (64, 16, torch.float32), (4000, 128, torch.bfloat16)])
def test_quantize_matches_the_formula(keys, d, dtype):
    """Slices on both sides of the one-launch limit (65536 elements), whole and partial pieces: bytes and scales of the
    kernel are those of the formula, evaluated on the host, for ordinary values, zeros, tiny and huge magnitudes, infinities
    and NaN."""
    g = torch.Generator().manual_seed(keys + d)
    k = torch.randn((2, 4, keys, d), generator=g).to(dtype)
    v = torch.randn((2, 4, keys, d), generator=g) * torch.logspace(-3, 3, keys * d)[torch.randperm(keys * d, generator=g)].view(keys, d)
    v = v.to(dtype)
    k[0, 1] = 0.0
    k[0, 2] *= 1e-4 if dtype is torch.float16 else 1e-36        # a scale near the end of the type's range
    k[0, 3, 0, 3] = float("inf")
    k[1, 0, -1, -1] = float("nan")
    k[1, 1] = -k[1, 1].abs()
    k[1, 1, 0, :4] = -0.0
    if dtype is not torch.float32 and keys * d >= 65536:        # every bit pattern that is a finite number
        bits = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dtype)
        v[1, 3].view(-1)[:65536] = torch.where(bits.isfinite(), bits, torch.zeros_like(bits))
    got = quantize_kv_fp8(k.cuda(), v.cuda())
    for t, t8, scale in ((k, got[0], got[2]), (v, got[1], got[3])):
        amax = t.float().abs().amax(dim=(2, 3))
        want = torch.where(amax > 0, amax * torch.tensor(1.0 / 448.0, dtype=torch.float32), torch.ones_like(amax))
        assert torch.equal(scale.cpu().nan_to_num(nan=-1.0), want.view(-1).nan_to_num(nan=-1.0))
        want8 = (t.float() / want[:, :, None, None]).to(torch.float8_e4m3fn)
        a, b = t8.cpu().view(torch.uint8), want8.view(torch.uint8)
        same = (a == b) | ((a & 0x7f == 0x7f) & (b & 0x7f == 0x7f))     # (the sign of a NaN is nobody's)
        assert bool(same.all()), f"{int((~same).sum())} bytes differ"


@pytest.mark.parametrize("keys", [64, 2100])      # one launch, two
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_quantize_at_the_ends_of_the_range(keys, dtype):
    """Slices whose scale is huge, tiny, denormal or rounds to zero, with zeros, infinities and NaN among them: the bytes and
    scales of the formula, evaluated on the host."""
    info = torch.finfo(dtype)
    g = torch.Generator().manual_seed(keys)
    x = torch.randn((1, 12, keys, 64), generator=g, dtype=torch.float64)
    x = x / x.abs().amax(dim=(2, 3), keepdim=True)
    x[0, :, :, 0] *= 2.0 ** -7                                # quotients down to the smallest bytes
    x[0, :, :, 1] *= 2.0 ** -16
    x[0, :, 0, 2:6] = torch.tensor([0.0, -0.0, 1.0, -1.0])
    tops = [info.max, info.max / 3, 2.0 ** 69, 2.0 ** 68.9, 2.0 ** -51, 2.0 ** -52, info.tiny, info.tiny * 448, info.tiny / 50,
            info.tiny * info.eps * 300, info.tiny * info.eps * 3, info.max]
    k = (x * torch.tensor([min(t, info.max) for t in tops], dtype=torch.float64).view(1, -1, 1, 1)).to(dtype)
    v = k.flip(1).clone()
    v[0, 0, 1, 1], v[0, 1, 1, 2], v[0, 4, 2, 3], v[0, 11, 0, 0] = float("inf"), -float("inf"), float("nan"), -float("nan")
    got = quantize_kv_fp8(k.cuda(), v.cuda())
    for t, t8, scale in ((k, got[0], got[2]), (v, got[1], got[3])):
        amax = t.float().abs().amax(dim=(2, 3))
        want = torch.where(amax > 0, amax * torch.tensor(1.0 / 448.0, dtype=torch.float32), torch.ones_like(amax))
        assert torch.equal(scale.cpu().nan_to_num(nan=-1.0), want.view(-1).nan_to_num(nan=-1.0))
        want8 = (t.float() / want[:, :, None, None]).to(torch.float8_e4m3fn)      # (scale 1 where a NaN is the largest)
        a, b = t8.cpu().view(torch.uint8), want8.view(torch.uint8)
        same = (a == b) | ((a & 0x7f == 0x7f) & (b & 0x7f == 0x7f))
        assert bool(same.all()), f"{int((~same).sum())} bytes differ, slices {(~same).any(-1).any(-1).nonzero().tolist()}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_quantize_one_tensor_after_the_other(dtype):
    """Tensors too large for a grid of both go one after the other and share the workspace: a pair of ordinary size, the
    grid's end set below it, against the launch of both."""
    import ctypes
    from fstattention_amd import _lib
    lib = ctypes.CDLL(_lib.LIB_PATH)
    fn = lib.fsta_internal_quantize_fp8
    fn.restype = ctypes.c_int
    fn.argtypes = [ctypes.c_void_p] * 6 + [ctypes.c_int64, ctypes.c_int64, ctypes.c_int32, ctypes.c_void_p, ctypes.c_size_t,
                                           ctypes.c_double, ctypes.c_void_p]
    code = _lib.BF16 if dtype is torch.bfloat16 else _lib.F32
    slices, elements = 6, 1111 * 64
    k, v, _ = (t.cuda() for t in rand_qkv(2, 3, 1111, 1111, 64, dtype, 77))
    v = v * 3.0
    need = _lib.load().fsta_quantize_workspace_bytes(slices, elements, code)
    assert need > 0
    per_tensor = slices * -(-elements // 8192) * 512       # threads
    results = []
    for grid_threads in (2.0 ** 32, 2.0 * per_tensor, 2.0 * per_tensor + 1, 0.0):
        k8, v8 = (torch.full(t.shape, 0x55, dtype=torch.uint8, device="cuda") for t in (k, v))
        ks, vs = torch.zeros(slices, device="cuda"), torch.zeros(slices, device="cuda")
        work = torch.full((need,), 0xff, dtype=torch.uint8, device="cuda")
        rc = fn(k.data_ptr(), v.data_ptr(), k8.data_ptr(), v8.data_ptr(), ks.data_ptr(), vs.data_ptr(), slices, elements, code,
                work.data_ptr(), need, grid_threads, torch.cuda.current_stream().cuda_stream)
        assert rc == _lib.OK
        # (the shared workspace's second half is written by the launch of both only)
        assert bool((work[need // 2:] == 0xff).all()) == (grid_threads <= 2.0 * per_tensor)
        results.append([t.cpu() for t in (k8, v8, ks, vs)])
    want = quantize_kv_fp8(k, v)
    for r in results:
        for got, ref in zip(r, want):
            assert torch.equal(got.view(torch.uint8), ref.cpu().view(torch.uint8).view(got.view(torch.uint8).shape))


def test_argument_errors():
    parent = trees.random_recursive_parents(64, 5)
    a_idx, a_mask, l_idx, max_anc = oracle_inputs(parent, 32)
    q, k, v = rand_qkv(1, 2, 64, 64, 64, torch.bfloat16, 1)
    k8, v8, ks, vs = quantize_kv_fp8(k, v)
    dev = [t.cuda() for t in (q, k8, v8, a_idx, a_mask, l_idx)]
    with pytest.raises(ValueError):      # scales without 8-bit storage
        fst_attention(q.cuda(), k.cuda(), v.cuda(), *dev[3:], 0.1, BLOCK_M=32, MAX_ANCESTORS=max_anc, k_scale=ks.cuda())
    with pytest.raises(ValueError):      # mixed storage
        fst_attention(dev[0], dev[1], v.cuda(), *dev[3:], 0.1, BLOCK_M=32, MAX_ANCESTORS=max_anc)
    with pytest.raises(ValueError):      # float32 queries
        fst_attention(q.float().cuda(), dev[1], dev[2], *dev[3:], 0.1, BLOCK_M=32, MAX_ANCESTORS=max_anc)
    with pytest.raises(ValueError):      # wrong number of scales
        fst_attention(*dev, 0.1, BLOCK_M=32, MAX_ANCESTORS=max_anc, k_scale=ks[:1].cuda())
    with pytest.raises(ValueError):      # no kernel choice
        fst_attention(*dev, 0.1, BLOCK_M=32, MAX_ANCESTORS=max_anc, generic=True)
