"""The calls whose speed this framework is judged by, over the range that its users meet.

A decode step of a sparse-KV server resolves the Top-K tokens of every request to device slots, replaces the
missing ones in the hot buffers, promotes their rows from pinned host memory and reads the selected rows. Each case
below is one of those calls, or all of them in one, made through the package's public functions on buffers that a
serving loop keeps. Everything is integer or byte work, so outputs are compared bit for bit.

listed() names the cases, draw() gives others of the same ranges; prepare() builds what the caller holds before the
call, run() makes one pass, work() states the bytes that a pass cannot do without.
"""

import sys
from pathlib import Path

import torch

_PACKAGE = Path(__file__).resolve().parents[1] / "elastic-kv-vmm_amd"
if str(_PACKAGE) not in sys.path:
    sys.path.insert(0, str(_PACKAGE))

from adaptive_sparse.decode_step import decode_step, decode_step_workspace  # noqa: E402
from adaptive_sparse.hisparse_swap import load_blocks_to_device_buffer_mha  # noqa: E402
from adaptive_sparse.host_arena import HostArena  # noqa: E402
from adaptive_sparse.kv_pool import BlockMajorLayout, KVPlanes, PlanePoolLayout  # noqa: E402
from adaptive_sparse.migration_engine import MigrationEngine, PagedKVPool  # noqa: E402
from adaptive_sparse.resident_lookup import build_residency_bits, resolve_resident  # noqa: E402
from adaptive_sparse.sparse_read import gather_kv  # noqa: E402
from adaptive_sparse.swap_in import HotBuffers, swap_in  # noqa: E402
from elastic_kv.backing import Backing  # noqa: E402
from experimental.resident_arena import VmmResidentArena  # noqa: E402
from experimental.sparse_read import gather_rows  # noqa: E402
from experimental.virtual_layout import VirtualKVLayout  # noqa: E402

DEVICE = "cuda"
STREAM = 6          # Top-K sets of a decode stream that the stateful cases walk through, over and over
MISSING = 0.4       # share of a stream's selected tokens that an LRU hot buffer of twice their number lacks, roughly


def listed():
    return [
        # The smallest call: the reference's lookup microbenchmark, a two-level lookup of 16 blocks of 128 tokens for
        # four requests. Latency and the launch are all of it.
        {"name": "lookup_micro", "kind": "mapped", "layers": 1, "batch": 4, "context": 8192, "blocks": 16,
         "block_size": 128},
        # One layer's lookup of a decode step, as a server that interleaves it with attention issues it.
        {"name": "lookup_layer", "kind": "lookup", "layers": 1, "batch": 32, "context": 49152, "blocks": 2048,
         "block_size": 1, "hot": 4096, "table": "int16", "shift": 6},
        # All 60 layers' lookups of the largest batch in one call: 15.7 M lanes with their miss lists.
        {"name": "lookup_step", "kind": "lookup", "layers": 60, "batch": 128, "context": 65536, "blocks": 2048,
         "block_size": 1, "hot": 4096, "table": "int16", "shift": 6},
        # Top-K of token blocks (block-sparse attention) over every layer.
        {"name": "lookup_blocks", "kind": "lookup", "layers": 28, "batch": 48, "context": 40000, "blocks": 32,
         "block_size": 64, "hot": 4096, "table": "int16", "shift": 6},
        # The Top-K K/V read of a large decode batch from the VMM pool, six layers in one call (the layers are alike).
        {"name": "gather_step", "kind": "gather", "layers": 6, "batch": 128, "lanes": 2048, "hot": 4096,
         "row_bytes": 512},
        # The reference's row gather behind a software table: 8192 rows of 512 B.
        {"name": "gather_rows", "kind": "rows", "batch": 4, "context": 65536, "selected": 2048, "width": 256,
         "indirect": True},
        # Device side of page migration: whole 2.25 MiB pages packed into staging and unpacked into other pages.
        {"name": "migrate_pages", "kind": "pages", "pages": 120, "layers": 36, "row_bytes": 32768},
        # Lookup and LRU replacement of a layer group at the composite step's shape: 43 % of the lanes miss.
        {"name": "swap_in", "kind": "swap", "layers": 20, "batch": 128, "context": 32699, "lanes": 2048, "hot": 4096,
         "table": "int16", "shift": 0},
        # The whole decode step of a small server: five launches of a few microseconds each.
        {"name": "step_small", "kind": "step", "layers": 1, "batch": 8, "context": 4096, "lanes": 64, "hot": 256,
         "row_bytes": 512, "host_rows": 8192, "table": "int16", "shift": 6},
        # The whole decode step of one layer of an ordinary batch, rows promoted over PCIe.
        {"name": "step_layer", "kind": "step", "layers": 1, "batch": 48, "context": 20011, "lanes": 1024, "hot": 2048,
         "row_bytes": 512, "host_rows": 65536, "table": "int16", "shift": 6},
        # The same swap-in with SGLang's calling convention, one layer of an ordinary batch.
        {"name": "hisparse_swap", "kind": "hisparse", "batch": 24, "context": 32768, "blocks": 16, "block_size": 128,
         "hot": 4096, "row_bytes": 512, "host_rows": 131072},
        # The residency summary made exact again after the table was edited outside the swap-in (a remap, an install).
        {"name": "summary_refresh", "kind": "summary", "layers": 16, "batch": 96, "context": 32699, "table": "int16",
         "shift": 6},
    ]


def _log(rng, low, high):
    """A whole number spread over the logarithm of [low, high]."""
    return min(high, max(low, round(low * (high / low) ** rng.random())))


def draw(rng):
    kind = rng.choice(["mapped", "lookup", "lookup", "lookup", "gather", "gather", "rows", "pages", "swap", "swap", "step",
                       "step", "hisparse", "hisparse", "summary"])
    if kind == "mapped":
        block = rng.choice([1, 16, 32, 64, 128])
        blocks = max(1, _log(rng, 256, 2048) // block)
        return {"kind": kind, "layers": rng.choice([1, 1, 4]), "batch": _log(rng, 1, 64),
                "context": _log(rng, max(2048, blocks * block), 32768), "blocks": blocks, "block_size": block}
    if kind == "lookup":
        block = rng.choice([1, 1, 1, 16, 64])
        blocks = max(1, _log(rng, 256, 2048) // block)
        table = rng.choice(["int16", "int16", "int32"])
        return {"kind": kind, "layers": _log(rng, 1, 60), "batch": _log(rng, 1, 128), "context": _log(rng, 8192, 65536),
                "blocks": blocks, "block_size": block, "hot": rng.choice([2048, 4096]), "table": table,
                "shift": rng.choice([0, 6, 6])}
    if kind == "gather":
        row_bytes = rng.choice([256, 512, 512, 1024, 1152])
        lanes = _log(rng, 64, 2048)
        hot = 2 * lanes
        layers, batch = rng.randint(1, 6), _log(rng, 1, 128)
        while layers * batch * lanes * row_bytes > 6 * 128 * 2048 * 512:
            batch = batch * 3 // 4
        return {"kind": kind, "layers": layers, "batch": batch, "lanes": lanes, "hot": hot, "row_bytes": row_bytes}
    if kind == "rows":
        return {"kind": kind, "batch": _log(rng, 1, 16), "context": _log(rng, 4096, 65536),
                "selected": _log(rng, 256, 4096), "width": rng.choice([64, 100, 128, 256, 576]),
                "indirect": rng.random() < 0.5}
    if kind == "pages":
        return {"kind": kind, "pages": _log(rng, 4, 120), "layers": rng.choice([8, 28, 36]),
                "row_bytes": rng.choice([8192, 16384, 32768])}
    if kind == "swap":
        lanes = _log(rng, 128, 2048)
        return {"kind": kind, "layers": _log(rng, 1, 20), "batch": _log(rng, 1, 128),
                "context": _log(rng, max(8192, 5 * lanes), 32768), "lanes": lanes, "hot": 2 * lanes,
                "table": rng.choice(["int16", "int32"]), "shift": rng.choice([0, 6])}
    if kind == "step":
        lanes = _log(rng, 48, 1024)
        return {"kind": kind, "layers": rng.choice([1, 1, 2]), "batch": _log(rng, 1, 24),
                "context": _log(rng, max(2048, 5 * lanes), 32768), "lanes": lanes, "hot": 2 * lanes,
                "row_bytes": rng.choice([256, 512, 1024]), "host_rows": 16384,
                "table": rng.choice(["int16", "int16", "int32"]), "shift": rng.choice([0, 6])}
    if kind == "hisparse":
        block = rng.choice([16, 64, 128])
        blocks = max(2, _log(rng, 256, 2048) // block)
        hot = rng.choice([blocks * block, 2 * blocks * block])
        return {"kind": kind, "batch": _log(rng, 1, 24), "context": _log(rng, 4 * blocks * block, 65536),
                "blocks": blocks, "block_size": block, "hot": min(4096, hot), "row_bytes": rng.choice([256, 512, 1024]),
                "host_rows": 65536}
    return {"kind": "summary", "layers": _log(rng, 1, 16), "batch": _log(rng, 4, 96),
            "context": _log(rng, 4096, 32768), "table": rng.choice(["int16", "int32"]), "shift": rng.choice([0, 6])}


# ---------------------------------------------------------------- inputs


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _i32(t):
    return t.to(torch.int32)


def _dtype(case):
    return torch.int16 if case["table"] == "int16" else torch.int32


def _lengths(case, gen, batch):
    """Ragged context lengths, from half of the widest to the widest."""
    span = case["context"] // 2
    lengths = case["context"] - torch.randint(0, span, (batch,), generator=gen, device=DEVICE)
    lengths[0] = case["context"]
    return lengths


def _choose(gen, layers, batch, units, count, window):
    """[layers, batch, count] distinct unit ids per row, in random order: four fifths from the row's last `window`
    units, the rest from the older ones (a row as short as the window takes all from it). units: [batch]."""
    window = max(window, count)
    older = (units - window).clamp_min(0).view(1, batch, 1)
    want = count - (count * 4) // 5
    recent = torch.rand((layers, batch, window), generator=gen, device=DEVICE).argsort(-1)[..., :count]
    recent = recent.minimum(units.view(1, batch, 1) - 1) if bool((units < window).any()) else recent
    recent = recent + older
    # One pick from each of `want` equal parts of the older units.
    part = torch.arange(want, device=DEVICE).view(1, 1, want)
    jitter = torch.rand((layers, batch, want), generator=gen, device=DEVICE, dtype=torch.float64)
    old = ((part + jitter) * older / max(want, 1)).long()
    lane = torch.arange(count, device=DEVICE)
    use_old = (lane >= count - want).view(1, 1, count) & (older >= want)
    ids = torch.where(use_old, torch.nn.functional.pad(old, (count - want, 0)), recent)
    order = torch.rand((layers, batch, count), generator=gen, device=DEVICE).argsort(-1)
    return _i32(torch.gather(ids, -1, order)).contiguous()


def _buffers(case, gen, lengths):
    """Hot buffers holding each request's most recent tokens in random slots."""
    layers, batch, hot = case["layers"], case["batch"], case["hot"]
    buffers = HotBuffers(layers, batch, case["context"], hot, DEVICE, table_dtype=_dtype(case),
                         bits_shift=case["shift"])
    tokens = (lengths.view(1, batch, 1) - hot + torch.arange(hot, device=DEVICE)).expand(layers, batch, hot)
    slots = torch.rand((layers, batch, hot), generator=gen, device=DEVICE).argsort(-1)
    buffers.install(tokens, slots)
    return buffers


def _plane_tensor(layers, rows, row_bytes):
    """K and V planes of `rows` rows in device memory, and their description."""
    pool = torch.zeros((layers, 2, rows, row_bytes), dtype=torch.uint8, device=DEVICE)
    plane = rows * row_bytes
    return pool, KVPlanes(base=pool.data_ptr(), device=pool.device.index, layers=layers, kv=2, layer_stride=2 * plane,
                          kv_stride=plane, row_stride=row_bytes, row_bytes=row_bytes, rows=rows, owner=pool)


def _bytes(gen, shape):
    return torch.randint(0, 256, shape, generator=gen, device=DEVICE, dtype=torch.uint8)


def prepare(case, seed):
    gen = _generator(seed)
    return {"kind": case["kind"], **globals()["_prepare_" + case["kind"]](case, gen)}


def _prepare_mapped(case, gen):
    layers, batch, context, block = case["layers"], case["batch"], case["context"], case["block_size"]
    total = batch * context
    # Each request's tokens sit at logical ids of its own; half of the ids are resident.
    table = (torch.randperm(total, generator=gen, device=DEVICE) + 1).reshape(batch, context)
    mapping = torch.randperm(total + 1, generator=gen, device=DEVICE)
    mapping = torch.where(torch.rand(total + 1, generator=gen, device=DEVICE) < 0.5, mapping, 0)
    lengths = _lengths(case, gen, batch)
    units = (lengths + block - 1) // block
    topk = _choose(gen, layers, batch, units, case["blocks"], 2 * case["blocks"])
    shape = (layers, batch, case["blocks"] * block)
    return {"topk": topk, "table": table, "mapping": mapping, "rows": torch.arange(batch, device=DEVICE).flip(0),
            "lengths": _i32(lengths), "selected": torch.arange(batch, device=DEVICE), "block": block,
            "slots": torch.full(shape, -1, dtype=torch.int32, device=DEVICE)}


def _prepare_lookup(case, gen):
    layers, batch, block = case["layers"], case["batch"], case["block_size"]
    hot, context = case["hot"], case["context"]
    lengths = _lengths(case, gen, batch)
    units = (lengths + block - 1) // block
    topk = _choose(gen, layers, batch, units, case["blocks"], hot // block)
    base = torch.arange(batch, device=DEVICE) * hot + 1
    padded = -(-context // 128) * 128
    table = torch.zeros((layers, batch, padded), dtype=_dtype(case), device=DEVICE)[..., :context]
    tokens = (lengths.view(1, batch, 1) - hot + torch.arange(hot, device=DEVICE)).expand(layers, batch, hot)
    slot = torch.rand((layers, batch, hot), generator=gen, device=DEVICE).argsort(-1)
    local = case["table"] == "int16"
    table.scatter_(2, tokens, (slot + (1 if local else base.view(1, batch, 1))).to(table.dtype))
    shape = (layers, batch, case["blocks"] * block)
    return {"topk": topk, "table": table, "rows": torch.arange(batch, device=DEVICE), "lengths": _i32(lengths),
            "selected": torch.arange(batch, device=DEVICE), "block": block, "shift": case["shift"],
            "bits": build_residency_bits(table, shift=case["shift"]), "base": base if local else None,
            "slots": torch.full(shape, -1, dtype=torch.int32, device=DEVICE),
            "misses": torch.full(shape, -1, dtype=torch.int32, device=DEVICE),
            "counts": torch.zeros(shape[:2], dtype=torch.int32, device=DEVICE)}


def _prepare_gather(case, gen):
    layers, batch, lanes, hot = case["layers"], case["batch"], case["lanes"], case["hot"]
    layout = PlanePoolLayout(layers=layers, kv=2, rows=1 + batch * hot, row_bytes=case["row_bytes"])
    backing = Backing(layout.capacity_bytes, layout.chunk_bytes)
    backing.ensure(range(backing.chunk_count))
    raw = backing.raw
    raw.view(torch.bfloat16).normal_(generator=gen)
    # Four fifths of the lanes are resident, in any of the request's hot slots; the rest read as zero rows.
    slots = torch.rand((layers, batch, hot), generator=gen, device=DEVICE).argsort(-1)[..., :lanes]
    slots = slots + torch.arange(batch, device=DEVICE).view(1, batch, 1) * hot + 1
    miss = torch.rand((layers, batch, lanes), generator=gen, device=DEVICE) >= 0.8
    return {"planes": layout.kv_planes(backing.base, backing.device, owner=backing), "raw": raw,
            "slots": _i32(slots.masked_fill(miss, 0)),
            "out": torch.empty((batch, layers, 2, lanes, case["row_bytes"] // 2), dtype=torch.bfloat16, device=DEVICE)}


def _prepare_rows(case, gen):
    batch, context, width = case["batch"], case["context"], case["width"]
    layout = VirtualKVLayout(batch, context, width)
    arena = VmmResidentArena(layout)
    for req in range(batch):
        arena.reserve(req, context)
        arena.row_view(req, context, torch.bfloat16).normal_(generator=gen)
    # A few positions lie past the request's length and read as zero rows.
    lengths = _lengths(case, gen, batch)
    positions = torch.randint(0, context, (batch, case["selected"]), generator=gen, device=DEVICE)
    positions = torch.where(torch.rand(positions.shape, generator=gen, device=DEVICE) < 0.9,
                            positions % lengths.view(batch, 1), positions)
    total = batch * context
    table = (torch.randperm(total, generator=gen, device=DEVICE) + 1).reshape(batch, context)
    offsets = torch.zeros(total + 1, dtype=torch.int64, device=DEVICE)
    item = layout.itemsize
    req = torch.arange(batch, device=DEVICE).view(batch, 1)
    offsets[table] = (layout.chunk_bytes // item + req * (layout.request_bytes // item)
                      + torch.arange(context, device=DEVICE) * width)
    return {"raw": arena.backing.raw.view(torch.bfloat16), "arena": arena, "layout": layout, "positions": positions,
            "ids": torch.arange(batch, device=DEVICE).flip(0), "lengths": lengths, "table": table, "offsets": offsets,
            "indirect": case["indirect"],
            "out": torch.empty((batch, case["selected"], width), dtype=torch.bfloat16, device=DEVICE)}


def _prepare_pages(case, gen):
    pages = case["pages"]
    layout = BlockMajorLayout(blocks=2 * pages + 1, layers=case["layers"], kv=2, row_bytes=case["row_bytes"])
    pool = PagedKVPool(layout, device=torch.cuda.current_device())
    pool.take(2 * pages)
    held = pool.backing.raw.narrow(0, layout.block_bytes, 2 * pages * layout.block_bytes)
    held.view(torch.bfloat16).normal_(generator=gen)
    order = torch.randperm(2 * pages, generator=gen, device=DEVICE) + 1
    return {"pool": pool, "held": held, "engine": MigrationEngine(pool, pages), "sources": order[:pages].contiguous(),
            "targets": order[pages:].contiguous()}


def _stream(case, gen, lengths):
    batch = case["batch"]
    return [_choose(gen, case["layers"], batch, lengths, case["lanes"], case["hot"]) for _ in range(STREAM)]


def _prepare_swap(case, gen):
    batch = case["batch"]
    lengths = _lengths(case, gen, batch)
    buffers = _buffers(case, gen, lengths)
    shape = (case["layers"], batch, case["lanes"])
    table = torch.randint(0, 1 << 20, (batch, case["context"]), generator=gen, device=DEVICE, dtype=torch.int32)
    state = {name: torch.full(shape, -1, dtype=torch.int32, device=DEVICE) for name in ("slots", "misses", "src", "dst")}
    return {"buffers": buffers, "stream": _stream(case, gen, lengths), "at": 0, "lengths": _i32(lengths),
            "rows": torch.arange(batch, device=DEVICE), "host_table": table,
            "counts": torch.zeros(shape[:2], dtype=torch.int32, device=DEVICE), **state}


def _prepare_step(case, gen):
    layers, batch, lanes, row_bytes = case["layers"], case["batch"], case["lanes"], case["row_bytes"]
    lengths = _lengths(case, gen, batch)
    buffers = _buffers(case, gen, lengths)
    host_rows = case["host_rows"]
    plane = host_rows * row_bytes
    arena = HostArena(2 * layers * plane)
    arena.host.copy_(_bytes(gen, (arena.nbytes,)))
    pool, planes = _plane_tensor(layers, 1 + batch * case["hot"], row_bytes)
    pool.copy_(_bytes(gen, pool.shape))
    host = KVPlanes(base=arena.device_ptr, device=pool.device.index, layers=layers, kv=2, layer_stride=2 * plane,
                    kv_stride=plane, row_stride=row_bytes, row_bytes=row_bytes, rows=host_rows, owner=arena)
    table = torch.randint(0, host_rows, (batch, case["context"]), generator=gen, device=DEVICE, dtype=torch.int32)
    size = decode_step_workspace(layers, batch, lanes)
    return {"buffers": buffers, "stream": _stream(case, gen, lengths), "at": 0, "lengths": _i32(lengths),
            "rows": torch.arange(batch, device=DEVICE), "host_table": table, "host": host, "pool": pool,
            "planes": planes, "slots": torch.full((layers, batch, lanes), -1, dtype=torch.int32, device=DEVICE),
            "out": torch.zeros((batch, layers, 2, lanes, row_bytes), dtype=torch.uint8, device=DEVICE),
            "workspace": torch.empty(size, dtype=torch.uint8, device=DEVICE)}


def _prepare_hisparse(case, gen):
    batch, context, hot, block = case["batch"], case["context"], case["hot"], case["block_size"]
    host_rows, row_bytes = case["host_rows"], case["row_bytes"]
    host = torch.empty((2, host_rows, row_bytes), dtype=torch.uint8, pin_memory=True)
    host.copy_(_bytes(gen, host.shape))
    lengths = _lengths(case, gen, batch) - STREAM
    stream, seq = [], []
    for step in range(STREAM):
        length = lengths + step + 1
        last = (length - 1) // block
        blocks = _choose(gen, 1, batch, last, case["blocks"], hot // block)[0]
        blocks[:, 0] = last          # the newest token's block is always selected
        stream.append(blocks)
        seq.append(_i32(length))
    device = torch.zeros((2, batch * (hot + 1) + 1, row_bytes), dtype=torch.uint8, device=DEVICE)
    return {"stream": stream, "seq": seq, "at": 0, "host": host, "device": device,
            "tokens": torch.full((batch, hot + 1), -1, dtype=torch.int32, device=DEVICE),
            "lru": torch.arange(hot, dtype=torch.int16, device=DEVICE).repeat(batch, 1),
            "host_locs": torch.randint(0, host_rows, (batch, context), generator=gen, device=DEVICE),
            "dev_locs": _i32(torch.arange(batch * (hot + 1), device=DEVICE).reshape(batch, hot + 1) + 1),
            "req": torch.arange(batch, device=DEVICE), "hot": hot, "block": block, "row_bytes": row_bytes,
            "out": torch.full((batch, case["blocks"] * block), -1, dtype=torch.int32, device=DEVICE)}


def _prepare_summary(case, gen):
    layers, batch, context = case["layers"], case["batch"], case["context"]
    hot = min(4096, context // 4)
    buffers = HotBuffers(layers, batch, context, hot, DEVICE, table_dtype=_dtype(case), bits_shift=case["shift"])
    lengths = _lengths(case, gen, batch)
    # A churned hot buffer: half recent tokens, half left over from anywhere in the context.
    recent = (lengths.view(1, batch, 1) - 1 - torch.arange(hot // 2, device=DEVICE)).expand(layers, batch, hot // 2)
    old = torch.randint(0, context, (layers, batch, hot - hot // 2), generator=gen, device=DEVICE)
    tokens = torch.cat([recent, old], -1)
    buffers.table.scatter_(2, tokens, 1 + torch.arange(hot, device=DEVICE).to(buffers.table.dtype).expand_as(tokens))
    # Tokens named twice keep whichever entry landed: only residency counts here, and it is the same.
    buffers.table.copy_((buffers.table != 0).to(buffers.table.dtype))
    return {"buffers": buffers}


# ---------------------------------------------------------------- one pass


def run(state):
    return globals()["_run_" + state["kind"]](state)


def _next(state):
    at = state["at"]
    state["at"] = (at + 1) % STREAM
    return at


def _run_mapped(s):
    resolve_resident(s["topk"], s["table"], s["mapping"], s["rows"], s["lengths"], s["selected"], s["slots"], s["block"])
    return s["slots"]


def _run_lookup(s):
    resolve_resident(s["topk"], s["table"], None, s["rows"], s["lengths"], s["selected"], s["slots"], s["block"],
                     misses=s["misses"], miss_count=s["counts"], resident_bits=s["bits"], bits_shift=s["shift"],
                     slot_base=s["base"])
    return s["slots"], s["misses"], s["counts"]


def _run_gather(s):
    gather_kv(s["planes"], s["slots"], s["out"])
    return s["out"]


def _run_rows(s):
    gather_rows(s["raw"], s["positions"], s["ids"], s["lengths"], s["table"], s["offsets"], s["out"], s["layout"],
                indirect=s["indirect"])
    return s["out"]


def _run_pages(s):
    engine = s["engine"]
    engine.pack(s["sources"], engine.out_staging)
    engine.unpack(s["targets"], engine.out_staging)
    return engine.out_staging, s["held"]


def _hot_state(buffers):
    kept = [buffers.table, buffers.bits, buffers.slot_token, buffers.stamps, buffers.status]
    return kept + ([buffers.resident_counts] if buffers.resident_counts is not None else [])


def _run_swap(s):
    buffers, topk = s["buffers"], s["stream"][_next(s)]
    resolve_resident(topk, buffers.table, None, s["rows"], s["lengths"], s["rows"], s["slots"], 1, misses=s["misses"],
                     miss_count=s["counts"], resident_bits=buffers.bits, bits_shift=buffers.bits_shift,
                     slot_base=buffers.slot_base if buffers.table.dtype == torch.int16 else None)
    swap_in(topk, 1, s["rows"], s["rows"], s["slots"], s["misses"], s["counts"], buffers, s["host_table"], s["src"],
            s["dst"])
    return [s["slots"], s["misses"], s["counts"], s["src"], s["dst"]] + _hot_state(buffers)


def _run_step(s):
    decode_step(s["stream"][_next(s)], s["rows"], s["lengths"], s["buffers"], s["host_table"], s["host"], s["planes"],
                s["slots"], s["out"], selected=s["rows"], workspace=s["workspace"])
    return [s["slots"], s["out"], s["pool"]] + _hot_state(s["buffers"])


def _run_hisparse(s):
    at = _next(s)
    load_blocks_to_device_buffer_mha(
        top_k_blocks=s["stream"][at], device_buffer_tokens=s["tokens"], host_cache_locs=s["host_locs"],
        device_buffer_locs=s["dev_locs"], host_cache_k=s["host"][0], host_cache_v=s["host"][1],
        device_buffer_k=s["device"][0], device_buffer_v=s["device"][1], top_k_device_locs=s["out"],
        req_pool_indices=s["req"], seq_lens=s["seq"][at], lru_slots=s["lru"], item_size_bytes=s["row_bytes"],
        hot_buffer_size=s["hot"], sparse_block_size=s["block"])
    return s["out"], s["tokens"], s["lru"], s["device"]


def _run_summary(s):
    buffers = s["buffers"]
    buffers.refresh_bits()
    return [buffers.bits] + ([buffers.resident_counts] if buffers.resident_counts is not None else [])


# ---------------------------------------------------------------- what a pass cannot do without


def work(case):
    """Bytes of one pass: each input element that the call must see read once, each output written once."""
    kind = case["kind"]
    entry = 2 if case.get("table") == "int16" else 4
    if kind in ("mapped", "lookup"):
        ids = case["layers"] * case["batch"] * case["blocks"]
        lanes = ids * case["block_size"]
        if kind == "mapped":        # id, logical id, slot (int64 tables), result
            return {"bytes": 4 * ids + lanes * (8 + 8 + 4), "flops": 0}
        # id, table entry, result; a fifth of the lanes are misses
        return {"bytes": 4 * ids + lanes * (entry + 4) + lanes // 5 * 4, "flops": 0}
    if kind == "gather":
        lanes = case["layers"] * case["batch"] * case["lanes"]
        return {"bytes": lanes * 4 + lanes * 2 * case["row_bytes"] * 9 // 5, "flops": 0}
    if kind == "rows":
        lanes = case["batch"] * case["selected"]
        return {"bytes": lanes * (4 * case["width"] + 8 + (16 if case["indirect"] else 0)), "flops": 0}
    if kind == "pages":
        return {"bytes": case["pages"] * case["layers"] * 2 * case["row_bytes"] * 4, "flops": 0}
    if kind in ("swap", "step"):
        rows = case["layers"] * case["batch"]
        lanes = rows * case["lanes"]
        missed = int(lanes * MISSING)
        # lookup: id, entry, slot, miss entry; swap-in: stamps read and written, slots, and per miss its list entry,
        # id, host row, victim's token, slot, new token, two table entries, two summary words, two promotions
        total = lanes * (4 + entry + 4) + missed * 4 + rows * 8 * case["hot"] + lanes * 4 + missed * (40 + 2 * entry)
        if kind == "step":          # promoted rows read and written, gathered rows read and written, K and V
            total += missed * 4 * case["row_bytes"] + lanes * (4 * case["row_bytes"] + 4)
        return {"bytes": total, "flops": 0}
    if kind == "hisparse":
        lanes = case["batch"] * case["blocks"] * case["block_size"]
        missed = int(lanes * MISSING)
        # hot tokens, LRU order (read, written), locations; per miss its host row index and both rows; results
        return {"bytes": case["batch"] * case["hot"] * (4 + 2 + 2) + lanes * 8 + missed * (12 + 4 * case["row_bytes"]),
                "flops": 0}
    entries = case["layers"] * case["batch"] * case["context"]
    groups = entries // (1 << case["shift"])
    return {"bytes": entries * entry + groups // 8 + (4 * groups if case["shift"] else 0), "flops": 0}


def tolerance(case):
    """Slots, counts, states and copied rows are whole numbers and bytes: the same from every implementation."""
    return "exact"
