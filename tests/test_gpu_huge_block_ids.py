"""Top-K block ids far past the table, whose product with the block size does not fit 64 bits.

Padding with INT64_MAX, and garbage ids whose product wraps to a small or a negative position, name no token: every
lookup returns -1 there, counts no miss and reads nothing for them, as for any other position past the row.
"""

import numpy as np
import pytest
import torch

from adaptive_sparse.decode_step import decode_step
from adaptive_sparse.hisparse_swap import load_blocks_to_device_buffer_mha
from adaptive_sparse.host_arena import HostArena
from adaptive_sparse.kv_pool import KVPlanes
from adaptive_sparse.resident_lookup import build_residency_bits, resolve_resident
from adaptive_sparse.swap_in import HotBuffers, swap_in

pytestmark = pytest.mark.gpu

BIG = np.iinfo(np.int64).max
HUGE = np.array([BIG, BIG - 1, 1 << 62, (1 << 62) + 1, 1 << 61, (1 << 61) + (1 << 28), (1 << 61) + 3, 1 << 60, 1 << 56,
                 BIG // 3 + 1, 1 << 32, (1 << 32) + 5, 1 << 31, -BIG - 1, -BIG])


def with_huge_ids(rng, shape, blocks):
    """Block ids of the table, every third one replaced by an id that is far outside it; also with -1 there."""
    ids = rng.integers(0, blocks, shape)
    far = rng.random(shape) < 1 / 3
    far[..., 0] = True
    huge = np.where(far, rng.choice(HUGE, shape), ids)
    return huge, np.where(far, -1, ids)


@pytest.mark.parametrize("bs", [1, 3, 4, 8, 64])
@pytest.mark.parametrize("form", ["int16", "int32", "int64", "strided", "mapped"])
def test_lookups_return_no_slot_for_huge_ids(gpu, coracle, bs, form):
    rng = np.random.default_rng(bs)
    layers, batch, k, table_rows, cols = 2, 5, 2048 // bs, 4, 4096
    table = rng.integers(1, 1 << 14, (layers, table_rows, cols)) * (rng.random((layers, table_rows, cols)) < 0.6)
    base = np.arange(table_rows) * 7 + 1
    stored = np.where(table > 0, base.reshape(1, -1, 1) + table - 1, 0) if form == "int16" else table
    mapping = np.concatenate([[0], rng.integers(1, 1 << 20, 1 << 14)]) if form == "mapped" else None
    topk, clean = with_huge_ids(rng, (layers, batch, k), cols // bs)
    rows, selected = rng.integers(0, table_rows, batch), np.arange(batch)
    lengths = np.array([cols, cols - 5, 9, -4, 1 << 30])
    blank = np.full((layers, batch, k * bs), -77, np.int32)
    want, want_misses, want_counts = coracle.resolve_resident(clean, stored, mapping, rows, lengths, selected, bs,
                                                              blank, with_misses=True)
    dtype = {"int16": torch.int16, "int64": torch.int64}.get(form, torch.int32)
    table_d = torch.tensor(table, dtype=dtype, device=gpu)
    step = 2 if form == "strided" else 1
    out = torch.full((*blank.shape, step), -77, dtype=torch.int32, device=gpu)[..., 0]
    misses = torch.full(blank.shape, -5, dtype=torch.int32, device=gpu)
    counts = torch.zeros((layers, batch), dtype=torch.int32, device=gpu)
    mapping_d = None if mapping is None else torch.tensor(mapping, device=gpu)
    for bits in ([None] if form in ("mapped", "int64") else [None, build_residency_bits(table_d)]):
        resolve_resident(torch.tensor(topk, device=gpu), table_d, mapping_d, torch.tensor(rows, device=gpu),
                         torch.tensor(lengths, device=gpu), torch.tensor(selected, device=gpu), out, bs,
                         misses=misses, miss_count=counts, resident_bits=bits,
                         slot_base=torch.tensor(base, device=gpu) if form == "int16" else None)
        assert np.array_equal(out.cpu().numpy(), want)
        assert np.array_equal(counts.cpu().numpy(), want_counts)
        for layer in range(layers):
            for row in range(batch):
                c = want_counts[layer, row]
                assert np.array_equal(misses[layer, row, :c].cpu().numpy(), want_misses[layer, row, :c])


@pytest.mark.parametrize("bs", [1, 4, 8])
@pytest.mark.parametrize("table_dtype,shift", [(torch.int16, 6), (torch.int32, 0)])
def test_decode_step_and_swap_in_ignore_huge_ids(gpu, bs, table_dtype, shift):
    # The step with the huge ids against the step with -1 in their place: one launch (dense) and the separate kernels
    # (a strided slot tensor); then a swap-in whose miss list names the huge ids' lanes.
    rng = np.random.default_rng(40 + bs)
    L, R, T, C, W, ROW = 2, 4, 1024, 256, 128, 64
    arena = HostArena(2 * L * T * ROW)
    try:
        arena.host.copy_(torch.randint(0, 256, (arena.nbytes,), dtype=torch.uint8))
        host = KVPlanes(base=arena.device_ptr, device=0, layers=L, kv=2, layer_stride=2 * T * ROW, kv_stride=T * ROW,
                        row_stride=ROW, row_bytes=ROW, rows=T, owner=arena)
        host_table = torch.arange(T, dtype=torch.int32, device=gpu).expand(R, T).contiguous()
        rows = torch.arange(R, device=gpu)
        lengths = torch.tensor([T, T - 9, 70, T], dtype=torch.int32, device=gpu)
        huge, clean = with_huge_ids(rng, (L, R, W // bs), T // bs)
        results = []
        for ids, step in ((huge, 1), (clean, 1), (huge, 2), (clean, 2)):
            buffers = HotBuffers(L, R, T, C, gpu, table_dtype=table_dtype, bits_shift=shift)
            pool = torch.zeros((L, 2, 1 + R * C, ROW), dtype=torch.uint8, device=gpu)
            plane = (1 + R * C) * ROW
            planes = KVPlanes(base=pool.data_ptr(), device=0, layers=L, kv=2, layer_stride=2 * plane, kv_stride=plane,
                              row_stride=ROW, row_bytes=ROW, rows=1 + R * C, owner=pool)
            slots = torch.full((L, R, W, step), -9, dtype=torch.int32, device=gpu)[..., 0]
            out = torch.zeros((R, L, 2, W, ROW), dtype=torch.uint8, device=gpu)
            topk = torch.tensor(ids, device=gpu)
            decode_step(topk, rows, lengths, buffers, host_table, host, planes, slots, out, block_size=bs)
            state = [slots, out, pool, buffers.table, buffers.bits, buffers.slot_token, buffers.stamps, buffers.status]
            # Every lane listed as a miss: those whose ids name no token change nothing.
            listed = torch.arange(W, dtype=torch.int32, device=gpu).expand(L, R, W).contiguous()
            counts = torch.full((L, R), W, dtype=torch.int32, device=gpu)
            src, dst = torch.full_like(listed, -3), torch.full_like(listed, -3)
            blank = torch.zeros_like(listed)
            swap_in(topk, bs, rows, rows, blank, listed, counts, buffers, host_table, src, dst)
            state += [blank, src, dst]
            results.append([t.cpu() for t in state])
        for other in results[1:]:
            for a, b in zip(results[0], other):
                assert torch.equal(a, b)
    finally:
        torch.cuda.synchronize()
        arena.close()


@pytest.mark.parametrize("bs", [1, 4, 16])
def test_sglang_convention_ignores_huge_ids(gpu, bs):
    rng = np.random.default_rng(90 + bs)
    batch, T, hot, W, row = 3, 600, 128, 64, 64
    host = [torch.randint(0, 256, (T, row), dtype=torch.uint8).pin_memory() for _ in range(2)]
    huge, clean = with_huge_ids(rng, (batch, W // bs), T // bs)
    results = []
    for ids in (huge, clean):
        device = [torch.zeros((batch * (hot + 1), row), dtype=torch.uint8, device=gpu) for _ in range(2)]
        tokens = torch.full((batch, hot + 1), -1, dtype=torch.int32, device=gpu)
        lru = torch.arange(hot, dtype=torch.int16, device=gpu).repeat(batch, 1)
        out = torch.full((batch, W), -7, dtype=torch.int32, device=gpu)
        load_blocks_to_device_buffer_mha(
            top_k_blocks=torch.tensor(ids, device=gpu), device_buffer_tokens=tokens,
            host_cache_locs=torch.arange(T, device=gpu).repeat(batch, 1),
            device_buffer_locs=torch.arange(batch * (hot + 1), dtype=torch.int32, device=gpu).view(batch, hot + 1),
            host_cache_k=host[0], host_cache_v=host[1], device_buffer_k=device[0], device_buffer_v=device[1],
            top_k_device_locs=out, req_pool_indices=torch.arange(batch, device=gpu),
            seq_lens=torch.tensor([T, T - 7, 1 << 30], device=gpu), lru_slots=lru, item_size_bytes=row,
            hot_buffer_size=hot, sparse_block_size=bs)
        results.append([t.cpu() for t in (out, tokens, lru, *device)])
    for a, b in zip(*results):
        assert torch.equal(a, b)
