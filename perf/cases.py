"""Performance cases of the package: what its users have it do, over the range of sizes they do it at.

A case is a dict of plain values.  ``listed()`` are the fixed ones, ``draw(rng)`` gives further ones of the same
ranges; ``prepare`` makes on the GPU what a program holds before the call, ``run`` is one pass through the public
entry points, ``work`` the bytes and operations that pass cannot do without, ``tolerance`` how far another correct
implementation at the same precision may be off.

``path`` says which use a case is of:

* ``attention``  one layer's attention of a decoding step: the tree's kernel inputs are in hand (they are built once
  per step and used by every layer), q, k and v are the layer's.  ``prefix`` > 0: k and v hold the KV cache of the
  sequence in front of the tree's own rows.  ``kv8``: K and V are stored as 8-bit floats with a scale per head.
* ``encode``     K and V of a prompt are brought to the 8-bit storage.
* ``step``       a whole decoding step: draft-head probabilities -> tree -> kernel inputs -> every layer's attention.
* ``rebuild``    a tree that arrives as a parent array is brought to depth-first order and to kernel inputs.
"""
import functools
import math

import torch

from fstattention_amd import (create_fst_attention_kernel_inputs, dfs_order_gpu, fst_attention,
                              kernel_inputs_from_parents_gpu, medusa_parents_gpu, quantize_kv_fp8, renumber_parents_gpu,
                              shift_for_prefix, trees)

DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
BYTES = {"float32": 4, "float16": 2, "bfloat16": 2}


def attention(name, tree, nodes, block_m, batch, heads, head_dim, dtype, prefix=0, kv8=False, lse=False):
    case = {"path": "attention", "tree": tree, "nodes": nodes, "block_m": block_m, "batch": batch, "heads": heads,
            "head_dim": head_dim, "dtype": dtype, "prefix": prefix, "kv8": kv8, "lse": lse}
    return dict(case, name=name) if name else case


def listed():
    return [
        # the smallest call: one small tree in float32, where the launch and the latency of a single block are all there is
        attention("plumbing_fp32_64", "random", 64, 16, 1, 8, 64, "float32"),
        # the ordinary decoding call: a static draft tree of 256 candidates, one sequence, one layer
        attention("medusa_256", "medusa", 256, 64, 1, 32, 128, "bfloat16"),
        # long chains with side branches: many ancestors per block
        attention("deep_1024", "deep", 1024, 64, 1, 32, 128, "bfloat16"),
        # wide and shallow, many nodes and few ancestors, a ragged last block, the log-sum-exp wanted (to be joined with
        # the part of another attention call)
        attention("wide_4001_lse", "wide", 4001, 64, 1, 32, 128, "float16", lse=True),
        # a batch of sequences that share one dynamic tree of 2048 nodes
        attention("batched_2048", "random64", 2048, 128, 8, 64, 128, "bfloat16"),
        # the largest of the left-weighted top-k trees the package's own benchmark runs
        attention("topk_65536", "topk", 65536, 128, 4, 48, 64, "float16"),
        # the same draft tree behind a long KV cache: what a decoding step of one long sequence spends its time on
        attention("cache_16384", "medusa", 256, 64, 1, 32, 128, "bfloat16", prefix=16384),
        # several sequences with a shorter cache and a small tree, odd sizes throughout
        attention("cache_3001_batch", "medusa", 61, 64, 4, 32, 128, "float16", prefix=3001, lse=True),
        # the KV cache kept in 8 bits
        attention("cache_8192_fp8", "medusa", 128, 64, 1, 32, 128, "bfloat16", prefix=8192, kv8=True),
        # a prompt's K and V written to that storage
        {"name": "encode_8192_fp8", "path": "encode", "batch": 1, "heads": 32, "keys": 8192, "head_dim": 128, "dtype": "bfloat16"},
        # a whole step of a 32-layer model whose tree changes with every step
        {"name": "step_32_layers", "path": "step", "nodes": 256, "depths": 4, "topk": 10, "block_m": 64, "max_ancestors": 96,
         "layers": 32, "heads": 32, "head_dim": 128, "prefix": 1000, "dtype": "bfloat16"},
        # a dynamic tree of 2048 nodes, renumbered depth-first before its kernel inputs are built
        {"name": "rebuild_2048", "path": "rebuild", "nodes": 2048, "window": 64, "block_m": 128, "max_ancestors": 224, "width": 112},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _draw_tree_attention(rng):
    """Trees without a cache in front: 16 to 65536 nodes, single sequences and batches."""
    dtype = rng.choice(["bfloat16", "bfloat16", "float16", "float16", "float32"])
    head_dim = rng.choice([64, 128])
    if dtype == "float32":
        tree = rng.choice(["random", "random64", "medusa"])
        nodes = _log_int(rng, 16, 512)
        return attention(None, tree, nodes, rng.choice([16, 32, 64]), 1, rng.randint(4, 16), head_dim, dtype, lse=rng.random() < 0.3)
    tree = rng.choice(["random", "random64", "medusa", "deep", "wide", "topk"])
    if tree == "topk":
        nodes = 2 ** rng.randint(10, 16)
        return attention(None, tree, nodes, 128, rng.randint(1, 4), rng.choice([8, 16, 32, 48]), 64, dtype)
    nodes = {"random": _log_int(rng, 24, 4096), "random64": _log_int(rng, 24, 4096), "medusa": _log_int(rng, 24, 1024),
             "deep": _log_int(rng, 160, 2048), "wide": _log_int(rng, 100, 8192)}[tree]
    block_m = rng.choice([32, 64, 128]) if nodes >= 128 else rng.choice([32, 64])
    heads = rng.choice([8, 16, 28, 32, 40, 64])
    batch = max(1, min(rng.randint(1, 8), (1 << 19) // (nodes * heads)))
    return attention(None, tree, nodes, block_m, batch, heads, head_dim, dtype, lse=rng.random() < 0.3)


def _draw_cache_attention(rng, kv8):
    """Draft trees of 8 to 256 nodes behind a cache of 64 to 32768 keys (8-bit cache: 16384)."""
    prefix = _log_int(rng, 64, 16384 if kv8 else 32768)
    nodes = _log_int(rng, 8, 256)
    heads = rng.choice([8, 16, 28, 32, 40, 64])
    head_dim = rng.choice([64, 128, 128])
    batch = max(1, min(rng.randint(1, 8), (1 << 20) // ((prefix + nodes) * heads)))
    return attention(None, rng.choice(["medusa", "random"]), nodes, rng.choice([32, 64]), batch, heads, head_dim,
                     rng.choice(["bfloat16", "float16"]), prefix=prefix, kv8=kv8, lse=not kv8 and rng.random() < 0.3)


def draw(rng):
    kind = rng.choices(["tree", "cache", "cache8", "encode", "step", "rebuild"], weights=[9, 6, 2, 2, 2, 2])[0]
    if kind == "tree":
        return _draw_tree_attention(rng)
    if kind in ("cache", "cache8"):
        return _draw_cache_attention(rng, kind == "cache8")
    if kind == "encode":
        heads, keys = rng.choice([8, 16, 28, 32, 40, 64]), _log_int(rng, 16, 16384)
        return {"path": "encode", "batch": max(1, min(rng.randint(1, 8), (1 << 18) // (heads * keys))), "heads": heads,
                "keys": keys, "head_dim": rng.choice([64, 128]), "dtype": rng.choice(["bfloat16", "float16"])}
    if kind == "step":
        heads, prefix = rng.choice([8, 16, 32]), _log_int(rng, 64, 4096)
        depths = rng.choice([3, 4])
        return {"path": "step", "nodes": _log_int(rng, 16, 256), "depths": depths, "topk": 10, "block_m": rng.choice([32, 64]),
                "max_ancestors": 96, "layers": rng.randint(4, 24), "heads": heads, "head_dim": rng.choice([64, 128]),
                "prefix": prefix, "dtype": rng.choice(["bfloat16", "float16"])}
    nodes = _log_int(rng, 64, 8192)
    window = max(16, -(-nodes // rng.randint(4, 32)))
    block_m = rng.choice([32, 64, 128])
    budget = -(-(block_m + 3 * nodes // window) // 32) * 32
    return {"path": "rebuild", "nodes": nodes, "window": window, "block_m": block_m, "max_ancestors": budget,
            "width": 3 * nodes // window + 16}


def _tree(tree, nodes, seed):
    """(lineage, level_lookup, parent or None) of one tree on the host."""
    if tree == "topk":      # the tree has 4 nodes fewer than its tensors have rows, and always 64 ancestor slots
        lineage, level = trees.create_tree(trees.DEPTH_MAPPING[nodes])
        return lineage, level, None
    if tree == "random":
        parent = trees.random_recursive_parents(nodes, seed)
    elif tree == "random64":
        parent = trees.random_recursive_parents(nodes, seed, window=64)
    elif tree == "medusa":
        parent = trees.medusa_parents(nodes, seed=seed)
    elif tree == "deep":
        parent = trees.deep_narrow_parents(nodes, seed=seed)
    else:
        parent = trees.wide_shallow_parents(nodes, 8)
    return trees.lineage_from_parents(parent) + (parent,)


def _normal(shape, dtype, generator):
    return torch.randn(shape, generator=generator, dtype=dtype, device="cuda")


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return {"attention": _prepare_attention, "encode": _prepare_encode, "step": _prepare_step,
            "rebuild": _prepare_rebuild}[case["path"]](case, seed, g)


def _prepare_attention(case, seed, g):
    dtype, n, d, m, prefix = DTYPES[case["dtype"]], case["nodes"], case["head_dim"], case["block_m"], case["prefix"]
    lineage, level, parent = _tree(case["tree"], n, seed)
    max_anc = trees.MAX_ANCESTOR_MAPPING[n] if parent is None else trees.required_max_ancestors(parent, m)
    a_idx, a_mask, l_idx = create_fst_attention_kernel_inputs(lineage.cuda(), level.cuda(), m, max_anc,
                                                              want_bool_mask=prefix == 0)
    if prefix:
        a_idx, l_idx, a_mask = shift_for_prefix(a_idx, l_idx, prefix, a_mask)
    shape, kv_shape = (case["batch"], case["heads"], n, d), (case["batch"], case["heads"], n + prefix, d)
    q, k, v = _normal(shape, dtype, g), _normal(kv_shape, dtype, g), _normal(kv_shape, dtype, g)
    options = {"BLOCK_M": m, "MAX_ANCESTORS": max_anc}
    if case["lse"]:
        options["return_lse"] = True
    if case["kv8"]:
        k, v, options["k_scale"], options["v_scale"] = quantize_kv_fp8(k, v)
    return {"path": "attention", "args": (q, k, v, a_idx, a_mask, l_idx, 1.0 / math.sqrt(d)), "options": options}


def _prepare_encode(case, seed, g):
    shape = (case["batch"], case["heads"], case["keys"], case["head_dim"])
    return {"path": "encode", "k": _normal(shape, DTYPES[case["dtype"]], g), "v": _normal(shape, DTYPES[case["dtype"]], g)}


def _prepare_step(case, seed, g):
    dtype, n, d = DTYPES[case["dtype"]], case["nodes"], case["head_dim"]
    probs = torch.from_numpy(trees.medusa_probs(case["depths"], case["topk"], seed=seed)).to("cuda", torch.float32)
    shape, kv_shape = (1, case["heads"], n, d), (1, case["heads"], n + case["prefix"], d)
    layers = [(_normal(shape, dtype, g), _normal(kv_shape, dtype, g), _normal(kv_shape, dtype, g)) for _ in range(case["layers"])]
    return {"path": "step", "case": dict(case), "probs": probs, "layers": layers,
            "status": torch.zeros((1,), dtype=torch.int32, device="cuda")}


def _prepare_rebuild(case, seed, g):
    parent = trees.random_recursive_parents(case["nodes"], seed, window=case["window"])
    return {"path": "rebuild", "case": dict(case), "parent": torch.from_numpy(parent).cuda()}


def run(state):
    if state["path"] == "attention":
        return fst_attention(*state["args"], **state["options"])
    if state["path"] == "encode":
        return quantize_kv_fp8(state["k"], state["v"])
    return _run_step(state) if state["path"] == "step" else _run_rebuild(state)


def _run_step(state):
    """Nothing of the step waits for the host; the status word of its stages is one the caller looks at later."""
    case, status = state["case"], state["status"]
    status.zero_()
    parent = medusa_parents_gpu(state["probs"], case["nodes"], status=status)
    a_idx, packed, l_idx, _ = kernel_inputs_from_parents_gpu(parent, case["block_m"], case["max_ancestors"], case["depths"] + 1,
                                                             check=False, status=status)
    a_idx, l_idx, packed = shift_for_prefix(a_idx, l_idx, case["prefix"], packed)
    scale = 1.0 / math.sqrt(case["head_dim"])
    return [fst_attention(q, k, v, a_idx, packed, l_idx, scale, BLOCK_M=case["block_m"], MAX_ANCESTORS=case["max_ancestors"])
            for q, k, v in state["layers"]]


def _run_rebuild(state):
    """A caller that wants to know about a malformed tree or too small a budget before it goes on."""
    case = state["case"]
    perm, rank = dfs_order_gpu(state["parent"], "light_first", check=False)
    parent = renumber_parents_gpu(state["parent"], perm, rank)
    a_idx, packed, l_idx = kernel_inputs_from_parents_gpu(parent, case["block_m"], case["max_ancestors"], case["width"])
    return perm, rank, parent, a_idx, packed.mask_bits, packed.anc_count, l_idx


@functools.lru_cache(maxsize=None)
def _tree_pairs(tree, nodes):
    """(query, key) pairs of one tree: every node with itself and its ancestors."""
    _, level, _ = _tree(tree, nodes, 1)
    return int(level.sum()) + nodes


def work(case):
    if case["path"] == "encode":
        elements = 2 * case["batch"] * case["heads"] * case["keys"] * case["head_dim"]
        return {"bytes": elements * (BYTES[case["dtype"]] + 1), "flops": 3 * elements}
    if case["path"] == "rebuild":
        n, blocks = case["nodes"], -(-case["nodes"] // case["block_m"])
        a, m = case["max_ancestors"], case["block_m"]
        return {"bytes": 8 * 4 * n + blocks * (8 * a + 8 * m + 4 * m * (-(-a // 32)) + 4), "flops": 0}
    n, d, esz = case["nodes"], case["head_dim"], BYTES[case["dtype"]]
    if case["path"] == "step":
        slices = case["heads"] * case["layers"]
        pairs = _tree_pairs("medusa", n) + n * case["prefix"]
        return {"bytes": slices * d * esz * (4 * n + 2 * case["prefix"]), "flops": 4 * d * slices * pairs}
    slices = case["batch"] * case["heads"]
    kv_esz = 1 if case["kv8"] else esz
    pairs = _tree_pairs(case["tree"], n) + n * case["prefix"]
    return {"bytes": slices * (d * (2 * n * esz + 2 * (n + case["prefix"]) * kv_esz) + (4 * n if case["lse"] else 0)),
            "flops": 4 * d * slices * pairs}


def tolerance(case):
    # integers and stored bytes are defined to the bit; attention is summed in float32 and rounded once to the output type
    if case["path"] in ("rebuild", "encode"):
        return "exact"
    return {"float32": {"rel": 1e-5, "max": 1e-4}, "float16": {"rel": 1e-3, "max": 1e-2},
            "bfloat16": {"rel": 5e-3, "max": 3e-2}}[case["dtype"]]
