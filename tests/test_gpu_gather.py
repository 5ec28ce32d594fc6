"""GPU parity of the HIP gather family against the oracle (bit-exact bytes)."""

import numpy as np
import pytest
import torch

from adaptive_sparse.kv_pool import KVPlanes
from adaptive_sparse.sparse_read import gather_kv, scatter_kv

pytestmark = pytest.mark.gpu


def make_pool(gpu, seed, layers, kv, rows, row_bytes, row_stride=None, pad=0):
    row_stride = row_stride or row_bytes
    plane = rows * row_stride + pad
    gen = torch.Generator(device="cpu").manual_seed(seed)
    host = torch.randint(0, 256, (layers * kv * plane,), dtype=torch.uint8, generator=gen)
    pool = host.to(gpu)
    planes = KVPlanes(base=pool.data_ptr(), device=gpu.index or 0, layers=layers, kv=kv,
                      layer_stride=kv * plane, kv_stride=plane, row_stride=row_stride,
                      row_bytes=row_bytes, rows=rows, owner=pool)
    return pool, host.numpy(), planes


GATHER_CASES = [
    # layers, kv, rows, row_bytes, batch, k, zero_below, row_stride
    (2, 2, 300, 512, 3, 70, 1, None),       # config-3 rows (2 heads x 128 bf16)
    (3, 2, 90, 2048, 2, 33, 1, None),       # config-1 rows (8 heads x 128 bf16)
    (2, 1, 50, 6, 4, 300, 1, None),         # 2-byte lanes
    (1, 2, 40, 24, 3, 17, 0, 40),           # 8-byte lanes, padded rows, block mode (0 valid)
    (1, 2, 12, 32768, 2, 5, 0, None),       # one 32 KiB row per tile (config-2 blocks)
    (1, 1, 6, 40960, 1, 4, 1, None),        # large rows split into 2 segments
]


@pytest.mark.parametrize("case", range(len(GATHER_CASES)))
def test_gather_kv_matches_oracle(gpu, coracle, case):
    layers, kv, rows, row_bytes, batch, k, zero_below, row_stride = GATHER_CASES[case]
    pool, host, planes = make_pool(gpu, 10 + case, layers, kv, rows, row_bytes, row_stride, pad=64)
    rng = np.random.default_rng(case)
    slots = rng.integers(-1, rows + 2, size=(layers, batch, k))
    out = torch.full((batch, layers, kv, k, row_bytes), 0xAB, dtype=torch.uint8, device=gpu)
    gather_kv(planes, torch.tensor(slots, dtype=torch.int32, device=gpu), out, zero_below=zero_below)
    want = coracle.gather_kv(host, planes.layer_stride, planes.kv_stride, planes.row_stride, row_bytes, rows,
                             slots, kv, zero_below=zero_below)
    assert np.array_equal(out.cpu().numpy(), want)


def test_gather_kv_shared_layer_slots_and_strided_output(gpu, coracle):
    layers, kv, rows, row_bytes, batch, k = 4, 2, 128, 256, 3, 50
    pool, host, planes = make_pool(gpu, 3, layers, kv, rows, row_bytes)
    rng = np.random.default_rng(5)
    slots = rng.integers(0, rows, size=(batch, k))
    shared = torch.tensor(slots, dtype=torch.int64, device=gpu).unsqueeze(0).expand(layers, batch, k)
    big = torch.zeros((batch, layers, kv, k + 3, row_bytes // 2), dtype=torch.bfloat16, device=gpu)
    out = big[:, :, :, 2:k + 2]
    gather_kv(planes, shared, out)
    want = coracle.gather_kv(host, planes.layer_stride, planes.kv_stride, planes.row_stride, row_bytes, rows,
                             slots, kv, shared_layers=layers)
    got = out.contiguous().view(torch.uint8).reshape(batch, layers, kv, k, row_bytes).cpu().numpy()
    assert np.array_equal(got, want)
    assert (big[:, :, :, :2] == 0).all() and (big[:, :, :, k + 2:] == 0).all()


@pytest.mark.parametrize("row_bytes", [512, 24, 40960])
def test_scatter_kv_matches_oracle_and_inverts_gather(gpu, coracle, row_bytes):
    layers, kv, rows, batch, k = 2, 2, 64, 2, 9
    pool, host, planes = make_pool(gpu, 21, layers, kv, rows, row_bytes)
    rng = np.random.default_rng(row_bytes)
    slots = np.stack([rng.permutation(np.arange(1, rows))[: batch * k].reshape(batch, k) for _ in range(layers)])
    slots[0, 0, 0] = -1  # padding lane writes nothing
    src = torch.randint(0, 256, (batch, layers, kv, k, row_bytes), dtype=torch.uint8, device=gpu)
    scatter_kv(planes, torch.tensor(slots, dtype=torch.int32, device=gpu), src)
    want = coracle.scatter_kv(host, planes.layer_stride, planes.kv_stride, planes.row_stride, row_bytes, rows,
                              slots, kv, src.cpu().numpy())
    assert np.array_equal(pool.cpu().numpy(), want)
    back = torch.zeros_like(src)
    gather_kv(planes, torch.tensor(slots, dtype=torch.int32, device=gpu), back)
    expect = src.clone()
    expect[0, 0, :, 0] = 0  # the padding lane gathers zeros
    assert torch.equal(back, expect)


def test_gather_kv_rejects_bad_shapes(gpu):
    pool, _, planes = make_pool(gpu, 1, 1, 2, 8, 16)
    slots = torch.zeros((1, 2, 3), dtype=torch.int32, device=gpu)
    with pytest.raises(ValueError):
        gather_kv(planes, slots, torch.zeros((2, 1, 2, 4, 16), dtype=torch.uint8, device=gpu))
    with pytest.raises(ValueError):
        gather_kv(planes, slots, torch.zeros((2, 1, 2, 3, 15), dtype=torch.uint8, device=gpu))
    with pytest.raises(ValueError):
        gather_kv(planes, torch.zeros((2, 2, 3), dtype=torch.int32, device=gpu),
                  torch.zeros((2, 2, 2, 3, 16), dtype=torch.uint8, device=gpu))


@pytest.mark.parametrize("row_bytes,kv,layers,batch,k", [
    (512, 2, 2, 24, 160),      # several strides of the grid per batch of rows
    (512, 2, 2, 700, 6),       # more (layer, batch) rows than one batch of rows holds
    (1040, 1, 1, 3, 340),      # a row that is no power of two of vectors
    (200, 2, 1, 5, 333), (36, 1, 2, 3, 3000), (6, 2, 1, 20, 2500), (3, 2, 1, 20, 5000),    # narrower vectors
    (512, 2, 1, 8, 64), (512, 2, 1, 8, 65),
    (16, 2, 1, 1, 1),
    (512, 2, 1, 6, 1023), (512, 2, 1, 6, 1024),  # the largest list of the tile kernel, the smallest past it
    (1040, 1, 1, 3, 2100),
    (256, 2, 1, 24, 513), (240, 2, 1, 24, 600),  # the shortest row past the tile kernel, a shorter one
    (520, 2, 1, 12, 520)])                       # 8-byte vectors: the tile kernel
def test_move_from_host_memory_matches_oracle(gpu, row_bytes, kv, layers, batch, k):
    from adaptive_sparse.host_arena import HostArena
    from adaptive_sparse.kv_pool import KVPlanes
    from adaptive_sparse.swap_in import move_kv
    from oracle import oracle as ref

    rng = np.random.default_rng(row_bytes + batch)
    src_n, dst_n = 300, layers * batch * k + 1
    arena = HostArena(layers * kv * src_n * row_bytes)
    try:
        source = rng.integers(0, 256, arena.nbytes, dtype=np.uint8)
        arena.host.copy_(torch.from_numpy(source))
        pool = torch.zeros(layers * kv * dst_n * row_bytes, dtype=torch.uint8, device=gpu)

        def planes(base, rows):
            return KVPlanes(base=base, device=0, layers=layers, kv=kv, layer_stride=kv * rows * row_bytes,
                            kv_stride=rows * row_bytes, row_stride=row_bytes, row_bytes=row_bytes, rows=rows, owner=None)

        src_planes, dst_planes = planes(arena.device_ptr, src_n), planes(pool.data_ptr(), dst_n)
        src_rows = rng.integers(-2, src_n + 2, (layers, batch, k))
        dst_rows = np.stack([rng.permutation(batch * k).reshape(batch, k) for _ in range(layers)])   # 0: skipped
        counts = rng.integers(-1, k + 2, (layers, batch)) * (rng.random((layers, batch)) < 0.7)
        t = lambda a: torch.tensor(a, dtype=torch.int32, device=gpu)  # noqa: E731
        layout = lambda p: (p.layer_stride, p.kv_stride, p.row_stride, row_bytes, p.rows)  # noqa: E731
        for current in (counts, np.full_like(counts, k), np.zeros_like(counts)):
            pool.zero_()
            move_kv(src_planes, t(src_rows), dst_planes, t(dst_rows), t(current))
            want = ref.move_kv(source, layout(src_planes), np.zeros(pool.numel(), np.uint8), layout(dst_planes),
                               src_rows, dst_rows, current, kv, zero_below=1)
            assert np.array_equal(pool.cpu().numpy(), want)
    finally:
        arena.close()


def test_host_moves_replay_from_a_graph(gpu):
    # A list past the tile kernel's limit: the call asks where its source lies while a stream is captured, and replays
    # follow rows, counts and host bytes rewritten in place.
    from adaptive_sparse.host_arena import HostArena
    from adaptive_sparse.kv_pool import KVPlanes
    from adaptive_sparse.swap_in import move_kv

    rng = np.random.default_rng(7)
    batch, k, n, row_bytes = 8, 800, 900, 512
    arena = HostArena(2 * n * row_bytes)
    try:
        pool = torch.zeros((2, batch * k + 1, row_bytes), dtype=torch.uint8, device=gpu)

        def planes(base, rows):
            return KVPlanes(base=base, device=0, layers=1, kv=2, layer_stride=0, kv_stride=rows * row_bytes,
                            row_stride=row_bytes, row_bytes=row_bytes, rows=rows, owner=None)

        src, dst = planes(arena.device_ptr, n), planes(pool.data_ptr(), batch * k + 1)
        src_rows = torch.zeros((1, batch, k), dtype=torch.int32, device=gpu)
        dst_rows = torch.arange(1, batch * k + 1, dtype=torch.int32, device=gpu).view(1, batch, k)
        counts = torch.zeros((1, batch), dtype=torch.int32, device=gpu)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            move_kv(src, src_rows, dst, dst_rows, counts)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            move_kv(src, src_rows, dst, dst_rows, counts)
        for _ in range(4):
            host = rng.integers(0, 256, (2, n, row_bytes), dtype=np.uint8)
            torch.cuda.synchronize()
            arena.host.copy_(torch.from_numpy(host.reshape(-1)))
            rows, count = rng.integers(0, n, (batch, k)), rng.integers(0, k + 1, batch)
            src_rows.copy_(torch.tensor(rows).view(1, batch, k))
            counts.copy_(torch.tensor(count).view(1, batch))
            pool.zero_()
            graph.replay()
            want = np.zeros((2, batch, k, row_bytes), np.uint8)
            for b in range(batch):
                want[:, b, :count[b]] = host[:, rows[b, :count[b]]]
            assert np.array_equal(pool[:, 1:].cpu().numpy().reshape(want.shape), want)
        torch.cuda.synchronize()
    finally:
        arena.close()
