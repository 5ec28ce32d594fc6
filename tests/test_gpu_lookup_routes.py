"""Each lookup kernel at the sizes that its rule gives it, with the route asserted.

The direct kernel takes the small jobs, so the prefetching and the strided kernels are reached by large ones only:
rows enough to pass the rule's limits, over exact and superset summaries, permuted selections with stray entries, short,
negative and over-long rows, requests without a table row, with and without miss lists. The C oracle checks every lane.
"""

import numpy as np
import pytest
import torch

from adaptive_sparse.resident_lookup import build_residency_bits, lookup_route, resolve_resident

pytestmark = pytest.mark.gpu


def check(coracle, gpu, route, layers, batch, k, cols, dtype, *, bs=1, shift=0, bits=None, superset=False, compact=True,
          mapped=None, topk_dtype=torch.int32, stray=True, seed=0):
    rng = np.random.default_rng(seed)
    table_rows = 9
    width = k * bs
    topk = rng.integers(-1, cols // bs + 2, (layers, batch, k))
    lengths = rng.integers(cols // 2, cols + 9, batch)
    lengths[:3] = (cols, -4, cols // 3)
    rows = rng.integers(0, table_rows, batch)
    rows[rng.random(batch) < 0.05] = table_rows                          # names no table row
    rows[4] = -1
    selected = rng.permutation(batch)
    if stray:
        selected = np.insert(selected[:-2], [0, 5, 5, batch - 2], [batch, -1, batch + 7, -9])
    base = rng.integers(1, 1 << 20, table_rows)
    entries = rng.integers(1, 1 << 15, (table_rows, cols)) * (rng.random((table_rows, cols)) < 0.4)
    entries = np.where(rng.random(entries.shape) < 0.02, -entries, entries)
    mapping = None
    if mapped is not None:
        entries = rng.integers(-2, 5002, entries.shape)
        mapping = rng.integers(1, 1 << 20, 5000) * (rng.random(5000) < 0.6)
    stored = np.where(entries > 0, base.reshape(-1, 1) + entries - 1, 0) if dtype == torch.int16 else entries
    blank = np.full((layers, batch, width), -77, np.int32)
    want, want_misses, want_counts = coracle.resolve_resident(topk, stored, mapping, rows, lengths, selected, bs, blank,
                                                              with_misses=True)
    table = torch.tensor(entries, dtype=dtype, device=gpu)
    summary = None
    if bits:
        summary = build_residency_bits(table, shift=shift)
        if superset:
            extra = (rng.random(summary.shape) < 0.3) * rng.integers(0, 1 << 31, summary.shape)
            summary |= torch.tensor(extra, dtype=torch.int32, device=gpu)
    slots = torch.tensor(blank, device=gpu)
    misses = torch.full(blank.shape, -5, dtype=torch.int32, device=gpu) if compact else None
    counts = torch.full(blank.shape[:2], -5, dtype=torch.int32, device=gpu) if compact else None
    args = (torch.tensor(topk, dtype=topk_dtype, device=gpu), table,
            None if mapping is None else torch.tensor(mapping, dtype=mapped, device=gpu),
            torch.tensor(rows, device=gpu), torch.tensor(lengths, dtype=torch.int32, device=gpu),
            torch.tensor(selected, device=gpu), slots, bs)
    extra = dict(misses=misses, miss_count=counts, resident_bits=summary, bits_shift=shift,
                 slot_base=torch.tensor(base, device=gpu) if dtype == torch.int16 else None)
    assert lookup_route(*args, **extra) == route
    resolve_resident(*args, **extra)
    assert np.array_equal(slots.cpu().numpy(), want)
    if compact:
        chosen = np.zeros(batch, bool)
        chosen[selected[(selected >= 0) & (selected < batch)]] = True
        got_counts, got = counts.cpu().numpy(), misses.cpu().numpy()
        assert np.array_equal(got_counts[:, chosen], want_counts[:, chosen])
        assert (got_counts[:, ~chosen] == -5).all()
        listed = np.arange(width)[None, None, :] < np.where(chosen, want_counts, 0)[:, :, None]
        assert np.array_equal(got[listed], want_misses[listed])
        assert (got[~listed] == -5).all()


# (layers, batch) past the rule's limit of table bytes for the width and entry size.
PREFETCHED = [(8, 100, 2048, torch.int16), (8, 90, 2040, torch.int16), (4, 100, 2040, torch.int32),
              (10, 150, 1032, torch.int16), (20, 150, 520, torch.int16), (10, 150, 520, torch.int32),
              (100, 210, 264, torch.int16)]


@pytest.mark.parametrize("layers,batch,k,dtype", PREFETCHED)
@pytest.mark.parametrize("superset,compact", [(False, True), (True, True), (True, False)])
def test_two_stage_prefetch(gpu, coracle, layers, batch, k, dtype, superset, compact):
    # Summary rows of at most 1024 words; widths whose threads past the row store its last piece again.
    for cols, shift in ((4001, 0), (32_768, 0), (9001, 6)):
        check(coracle, gpu, "two-stage prefetch", layers, batch, k, cols, dtype, shift=shift, bits=True,
              superset=superset, compact=compact, seed=k + shift)


@pytest.mark.parametrize("layers,batch,k,dtype", PREFETCHED[:5])
@pytest.mark.parametrize("superset,compact", [(False, True), (True, True), (True, False)])
def test_one_stage_prefetch(gpu, coracle, layers, batch, k, dtype, superset, compact):
    # Summary rows of 1025 to 2048 words.
    for cols in (32_769, 65_536):
        check(coracle, gpu, "one-stage prefetch", layers, batch, k, cols, dtype, bits=True, superset=superset,
              compact=compact, seed=k + cols)


@pytest.mark.parametrize("dtype,layers,batch,k,cols", [
    (torch.int16, 110, 310, 264, 3000), (torch.int16, 110, 310, 264, 40_000), (torch.int32, 110, 310, 264, 3000)])
def test_prefetch_with_a_raised_grid(gpu, coracle, dtype, layers, batch, k, cols):
    # 34,320 items: more than 16 for each of the (about 2048) resident workgroups, so the host raises the grid.
    route = "one-stage prefetch" if cols > 32_768 else "two-stage prefetch"
    check(coracle, gpu, route, layers, batch, k, cols, dtype, bits=True, superset=True, seed=cols)


@pytest.mark.parametrize("dtype,layers,batch,k,bits,route", [
    (torch.int16, 8, 160, 1201, True, "local"), (torch.int16, 8, 160, 1201, False, "strided"),
    (torch.int32, 8, 100, 1201, True, "strided"), (torch.int32, 8, 100, 2047, False, "strided"),
    (torch.int16, 20, 210, 700, False, "strided"), (torch.int16, 20, 210, 701, True, "local"),
    (torch.int32, 10, 210, 701, True, "strided")])
@pytest.mark.parametrize("compact", [True, False])
def test_large_ragged_rows(gpu, coracle, dtype, layers, batch, k, bits, route, compact):
    check(coracle, gpu, route, layers, batch, k, 4001, dtype, bits=bits, superset=bits, compact=compact, seed=k)


@pytest.mark.parametrize("dtype,layers,batch,k,route", [
    (torch.int16, 8, 86, 2048, "direct"),              # with two stray ones 704 rows, 2.75 MiB: the last direct ones
    (torch.int16, 8, 87, 2048, "two-stage prefetch"),
    (torch.int32, 100, 210, 256, "direct"), (torch.int32, 100, 210, 264, "two-stage prefetch"),
    (torch.int16, 20, 150, 512, "direct"), (torch.int16, 40, 260, 512, "two-stage prefetch")])
def test_the_lines_between_direct_and_prefetched(gpu, coracle, dtype, layers, batch, k, route):
    check(coracle, gpu, route, layers, batch, k, 4001, dtype, bits=True, shift=6, seed=batch)


@pytest.mark.parametrize("mapped", [torch.int32, torch.int64])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("batch,bs,k", [(256, 1, 600), (257, 1, 600), (256, 128, 16), (257, 128, 16)])
@pytest.mark.parametrize("compact", [True, False])
def test_two_level_lookups_at_the_direct_limit(gpu, coracle, mapped, dtype, batch, bs, k, compact):
    # Two layers: 512 rows are the last direct ones. The stray entries of a selection count as rows.
    for stray in (False, True):
        rows = batch if not stray else batch + 2
        route = "two-level direct" if 2 * rows <= 512 else "two-level"
        check(coracle, gpu, route, 2, batch, k, 4001, dtype, bs=bs, mapped=mapped, compact=compact, stray=stray,
              seed=batch + bs)
