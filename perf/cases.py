"""The work this library is timed on: calls of its public entry points at the
sizes its users make them with.

Five families, each with the options its users set:

* ``blocks``: gather / scatter of a block-id list between a paged KV pool (one
  storage per layer and K or V) and a device staging buffer, with or without
  an fp8 cache's scale tables;
* ``pack``: offset-table pack / unpack of a parameter set;
* ``split``: column split of row-major weights over tensor-parallel ranks;
* ``tile``: tile / detile of weights kept in an XLA-style tiled layout;
* ``offload``: the whole path to the pinned host tier and back over PCIe.

Every output is a copy of input bytes, so every comparison is exact.
"""
import random

import numpy
import torch

from __graft_entry__ import load_package

kvx = load_package()

MIB = 1 << 20
GIB = 1 << 30

# Shapes of a Llama-3-8B layer's matrices.
LAYER_8B = ((4096, 4096), (1024, 4096), (1024, 4096), (4096, 4096),
            (14336, 4096), (14336, 4096), (4096, 14336))


def listed():
    return [
        # Decode: one new block of a sequence leaves the cache of a Llama-3-8B
        # (32 layers, K and V apart, 16 tokens x 8 heads x 128 in bf16).
        # Launch latency.
        dict(name="gather_one_block", family="blocks", gather=True, storages=64,
             block_bytes=32768, scale_bytes=0, pool=2048, n=1, run=1, block_major=False),
        # Prefill: a batch of 512 blocks of the same cache, ids as a worked-in
        # allocator hands them out, out of the pool and back into it.
        dict(name="gather_batch", family="blocks", gather=True, storages=64,
             block_bytes=32768, scale_bytes=0, pool=2048, n=512, run=1, block_major=False),
        dict(name="scatter_batch", family="blocks", gather=False, storages=64,
             block_bytes=32768, scale_bytes=0, pool=2048, n=512, run=1, block_major=False),
        # One rank of Llama-3-70B over 8 GPUs (80 layers, one KV head a rank):
        # 4 KiB blocks in bf16.
        dict(name="gather_one_head", family="blocks", gather=True, storages=160,
             block_bytes=4096, scale_bytes=0, pool=4096, n=768, run=1, block_major=False),
        # The same rank with an fp8 cache: 2 KiB blocks and one fp32 scale per
        # (layer, block), in one call.
        dict(name="scatter_one_head_fp8", family="blocks", gather=False, storages=160,
             block_bytes=2048, scale_bytes=4, pool=4096, n=768, run=1, block_major=False),
        # Weight sync of quantised weights: 8-bit matrices, each with one fp32
        # scale, and the bf16 norms, packed by the offset table.
        dict(name="pack_8bit_scaled", family="pack", pack=True, layers=4, itemsize=1,
             scalars=True),
        # Resharding bf16 weights over 8 ranks, and over 3, where a chunk's
        # rows no longer start on vector boundaries.
        dict(name="split_8", family="split", rows=14336, cols=4096, itemsize=2, parts=8,
             matrices=4),
        dict(name="split_3", family="split", rows=14336, cols=4096, itemsize=2, parts=3,
             matrices=4),
        # A weight kept in the bf16 T(8,128)(2,1) layout, to its row-major image.
        dict(name="detile_rows", family="tile", tile=False, itemsize=2, packed=True,
             batch=1, height=14336, width=4096, column_major=False),
        # An output projection with an odd vocabulary, into the same layout.
        dict(name="tile_odd_width", family="tile", tile=True, itemsize=2, packed=True,
             batch=1, height=4096, width=32003, column_major=False),
        # A weight that the producer keeps column-major under the same tiles.
        dict(name="detile_columns", family="tile", tile=False, itemsize=2, packed=True,
             batch=1, height=4096, width=14336, column_major=True),
        # Offload of one batch and reload of another at once over PCIe.
        dict(name="offload_reload", family="offload", storages=64, block_bytes=32768,
             pool=1024, n=256, slots=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _draw_blocks(rng):
    heads = rng.choice([1, 1, 2, 4, 8])
    itemsize = rng.choice([1, 2])
    tokens = rng.choice([8, 16, 16, 32, 64])
    block = tokens * heads * rng.choice([64, 80, 96, 128, 128, 256]) * itemsize
    storages = 2 * _log_int(rng, 4, 80)
    most = max(1, min(1024, GIB // (storages * block)))
    n = _log_int(rng, 1, most)
    scales = itemsize == 1 and rng.random() < 0.7
    return dict(family="blocks", gather=rng.random() < 0.5, storages=storages,
                block_bytes=block, scale_bytes=4 * heads if scales else 0, pool=2 * n + 61,
                n=n, run=rng.choice([1, 1, 4, 16]),
                block_major=not scales and rng.random() < 0.25)


def _draw_pack(rng):
    itemsize = rng.choice([1, 2])
    return dict(family="pack", pack=rng.random() < 0.5, layers=rng.randint(1, 4 // itemsize),
                itemsize=itemsize, scalars=rng.random() < 0.7)


def _draw_split(rng):
    itemsize = rng.choice([1, 2, 2, 4])
    rows, cols = _log_int(rng, 256, 16384), _log_int(rng, 512, 14336)
    if rng.random() < 0.6:
        cols = (cols + 127) // 128 * 128
    matrices = max(1, min(4, GIB // 2 // (rows * cols * itemsize)))
    return dict(family="split", rows=rows, cols=cols, itemsize=itemsize,
                parts=rng.choice([2, 3, 4, 5, 6, 7, 8]), matrices=matrices)


def _draw_tile(rng):
    itemsize = rng.choice([1, 2, 2, 4])
    height, width = _log_int(rng, 128, 16384), _log_int(rng, 128, 16384)
    if rng.random() < 0.5:
        width = (width + 127) // 128 * 128
    batch = rng.choice([1, 1, 2, 8])
    while batch > 1 and batch * height * width * itemsize > GIB // 4:
        batch //= 2
    return dict(family="tile", tile=rng.random() < 0.5, itemsize=itemsize,
                packed=itemsize < 4 and rng.random() < 0.8, batch=batch, height=height,
                width=width, column_major=rng.random() < 0.35)


def _draw_offload(rng):
    storages = 2 * _log_int(rng, 8, 32)
    block = rng.choice([4096, 16384, 32768, 32768])
    n = _log_int(rng, 8, 256)
    return dict(family="offload", storages=storages, block_bytes=block, pool=4 * n, n=n,
                slots=rng.random() < 0.5)


def draw(rng):
    family = rng.choice(["blocks"] * 5 + ["pack"] * 2 + ["split"] * 3 + ["tile"] * 4
                        + ["offload"])
    return {"blocks": _draw_blocks, "pack": _draw_pack, "split": _draw_split,
            "tile": _draw_tile, "offload": _draw_offload}[family](rng)


def _bytes(gen, n):
    """n random bytes on the GPU (a uint8 tensor)."""
    words = torch.empty((n + 7) // 8, dtype=torch.int64, device="cuda")
    return words.random_(generator=gen).view(torch.uint8)[:n]


def _whole(t):
    """t's bytes as one flat integer tensor, of the widest type that divides them."""
    t = t.reshape(-1).view(torch.uint8)
    for dtype, size in ((torch.int64, 8), (torch.int32, 4), (torch.int16, 2)):
        if t.numel() % size == 0 and t.data_ptr() % size == 0:
            return t.view(dtype)
    return t


def _ids(rng, pool, n, run):
    """n distinct block ids of [0, pool): runs of `run` consecutive ids in random order."""
    starts = list(range(0, pool, run))
    rng.shuffle(starts)
    ids = [i for s in starts for i in range(s, min(s + run, pool))]
    return ids[:n]


def _prepare_blocks(case, gen, rng):
    S, P, B, n = case["storages"], case["pool"], case["block_bytes"], case["n"]
    pool = _bytes(gen, S * P * B)
    caches = [pool[w * P * B:(w + 1) * P * B].view(P, B) for w in range(S)]
    total, scales, tables = S * n * B, None, []
    if case["scale_bytes"]:
        L, K = S // 2, case["scale_bytes"]
        scales = _bytes(gen, L * P * K)
        tables = [scales[w * P * K:(w + 1) * P * K].view(P, K) for w in range(L)]
        total += L * n * K
    mgr = kvx.KVCacheManager(caches, host_blocks_to_allocate=1, scale_tables=tables)
    ids = _ids(rng, P, n, case["run"])
    staging = _bytes(gen, total)
    return dict(case=case, mgr=mgr, ids=ids, staging=staging, pool=pool, scales=scales)


def _run_blocks(s):
    fn = s["mgr"].gather if s["case"]["gather"] else s["mgr"].scatter
    fn(s["ids"], s["staging"], block_major=s["case"]["block_major"])
    if s["case"]["gather"]:
        return _whole(s["staging"])
    return [_whole(t) for t in (s["pool"], s["scales"]) if t is not None]


def _pack_shapes(case):
    """(shape, itemsize) of every parameter of the set."""
    out = []
    for _ in range(case["layers"]):
        out.append(((4096,), 2))
        for shape in LAYER_8B:
            out.append((shape, case["itemsize"]))
            if case["scalars"]:
                out.append(((1,), 4))
        out.append(((4096,), 2))
    return out


def _numel(shape):
    n = 1
    for d in shape:
        n *= d
    return n


def _prepare_pack(case, gen, rng):
    del rng
    dtype = {1: torch.uint8, 2: torch.int16, 4: torch.int32}
    params = [_bytes(gen, _numel(shape) * size).view(dtype[size]).view(shape)
              for shape, size in _pack_shapes(case)]
    sync = kvx.WeightSynchronizer([[p] for p in params])
    staging = _bytes(gen, sync.total_bytes)
    return dict(case=case, sync=sync, params=params, staging=staging)


def _run_pack(s):
    if s["case"]["pack"]:
        s["sync"].pack(s["staging"])
        return _whole(s["staging"])
    s["sync"].unpack(s["staging"])
    return [_whole(p) for p in s["params"]]


def _prepare_split(case, gen, rng):
    del rng
    dtype = {1: torch.uint8, 2: torch.int16, 4: torch.int32}[case["itemsize"]]
    R, C, k = case["rows"], case["cols"], case["parts"]
    weights, chunks, entries = [], [], []
    bounds = [box[1] for box in kvx.compute_nd_shard_slices((R, C), (1, k))]
    for _ in range(case["matrices"]):
        w = _bytes(gen, R * C * case["itemsize"]).view(dtype).view(R, C)
        outs = [torch.zeros(R, c1 - c0, dtype=dtype, device="cuda") for c0, c1 in bounds]
        entries += kvx.column_split_entries(w, outs)
        weights.append(w)
        chunks += outs
    return dict(case=case, plan=kvx.StridedPlan(entries), weights=weights, chunks=chunks)


def _run_split(s):
    kvx.copy_strided(s["plan"])
    return s["chunks"]


def _layout(case):
    tiles = [(8, 128)]
    if case["packed"]:
        tiles.append((4 // case["itemsize"], 1))
    dims = (case["height"], case["width"])
    if case["batch"] > 1:
        dims = (case["batch"],) + dims
    order = list(range(len(dims) - 1, -1, -1))
    if case["column_major"]:
        order[0], order[1] = order[1], order[0]
    return kvx.tiling.TiledLayout(case["itemsize"], dims, tiles, order)


def _prepare_tile(case, gen, rng):
    del rng
    lay = _layout(case)
    return dict(case=case, layout=lay, linear=_bytes(gen, lay.logical_bytes),
                tiled=_bytes(gen, lay.tiled_bytes))


def _run_tile(s):
    if s["case"]["tile"]:
        kvx.tiling.tile_buffer(s["layout"], s["linear"], s["tiled"])
        return _whole(s["tiled"])
    kvx.tiling.detile_buffer(s["layout"], s["tiled"], s["linear"])
    return _whole(s["linear"])


class _HostMirror:
    """One storage's host mirror as an array that keeps its manager alive."""

    def __init__(self, mgr, storage):
        self.mgr = mgr
        self.__array_interface__ = mgr.host_view(storage).__array_interface__


def _prepare_offload(case, gen, rng):
    S, P, B, n = case["storages"], case["pool"], case["block_bytes"], case["n"]
    pool = _bytes(gen, S * P * B)
    caches = [pool[w * P * B:(w + 1) * P * B].view(P, B) for w in range(S)]
    mgr = kvx.KVCacheManager(caches, host_blocks_to_allocate=2 * n)
    ids = _ids(rng, P, 2 * n, 1)
    # Offloaded blocks go to host blocks [0, n), reloaded ones come from
    # [n, 2n): a slot's consecutive blocks, or blocks of a worked-in tier.
    out_host, in_host = list(range(n)), list(range(n, 2 * n))
    if not case["slots"]:
        rng.shuffle(out_host)
        rng.shuffle(in_host)
    # The host tier holds what was offloaded before.
    mgr.d2h(ids[:n], in_host).Await()
    hosts = [torch.from_numpy(numpy.asarray(_HostMirror(mgr, w))) for w in range(S)]
    return dict(case=case, mgr=mgr, pool=pool, out_ids=ids[:n], in_ids=ids[n:],
                out_host=out_host, in_host=in_host, hosts=hosts)


def _run_offload(s):
    mgr = s["mgr"]
    save = mgr.d2h(s["out_ids"], s["out_host"])
    load = mgr.h2d(s["in_host"], s["in_ids"])
    save.Await()
    load.Await()
    n = s["case"]["n"] * s["case"]["block_bytes"]
    return [_whole(s["pool"])] + [_whole(h[:n]) for h in s["hosts"][:60]]


_FAMILIES = {"blocks": (_prepare_blocks, _run_blocks), "pack": (_prepare_pack, _run_pack),
             "split": (_prepare_split, _run_split), "tile": (_prepare_tile, _run_tile),
             "offload": (_prepare_offload, _run_offload)}


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    state = _FAMILIES[case["family"]][0](case, gen, random.Random(seed))
    state["run"] = _FAMILIES[case["family"]][1]
    return state


def run(state):
    return state["run"](state)


def _moved(case):
    """Bytes of the input that reach the output."""
    if case["family"] == "blocks":
        S, n = case["storages"], case["n"]
        return n * (S * case["block_bytes"] + S // 2 * case["scale_bytes"])
    if case["family"] == "pack":
        return sum(_numel(shape) * size for shape, size in _pack_shapes(case))
    if case["family"] == "split":
        return case["matrices"] * case["rows"] * case["cols"] * case["itemsize"]
    if case["family"] == "tile":
        return case["batch"] * case["height"] * case["width"] * case["itemsize"]
    return 2 * case["n"] * case["storages"] * case["block_bytes"]


def work(case):
    moved = _moved(case)
    written = moved
    if case["family"] == "tile" and case["tile"]:
        # The tiled buffer's padding is output too.
        h, w = case["height"], case["width"]
        if case["column_major"]:
            h, w = w, h
        written = (case["batch"] * ((h + 7) // 8 * 8) * ((w + 127) // 128 * 128)
                   * case["itemsize"])
    return {"bytes": moved + written, "flops": 0}


def tolerance(case):
    del case
    return "exact"
