"""Slots and tile tables of packed prompts written on the device, against the host's."""
from __future__ import annotations

import random

import pytest
import torch

from conftest import announce
from specdec_amd import SdvError
from specdec_amd.engine.paged_cache import PagedKVCache
from specdec_amd.kernels import ops

pytestmark = pytest.mark.gpu


def _host(cache, lengths):
    slots = [cache.blocks[b][p // 16] * 16 + p % 16 for b, n in enumerate(lengths) for p in range(n)]
    return torch.tensor(slots, dtype=torch.int32), torch.tensor(ops.varlen_tile_starts(lengths), dtype=torch.int32)


@pytest.mark.parametrize("lengths", [[1], [16], [17, 0, 0, 31, 1], [0, 0, 5], [0], [300, 4000, 1, 16, 15],
                                     [random.Random(7).choice([0, 1, 15, 16, 17, 40]) for _ in range(700)]])
def test_varlen_slots_match_the_host(cuda_device, lengths):
    """One-row and one-block prompts, empty ones between and at the ends, several launches (256
    sequences each)."""
    announce(f"varlen slots of {len(lengths)} sequences")
    cache = PagedKVCache(1, 64, batch=len(lengths), num_blocks=sum(-(-n // 16) for n in lengths) + 3, device=cuda_device, seed=3)
    for b, n in enumerate(lengths):
        cache.reserve(b, n + 5 * (b % 2 == 0))
    slots, tiles = ops.varlen_slots(cache.block_table(), lengths)
    want_slots, want_tiles = _host(cache, lengths)
    torch.cuda.synchronize()
    assert torch.equal(slots.cpu(), want_slots) and torch.equal(tiles.cpu(), want_tiles)
    assert torch.equal(cache.varlen_slots(lengths).cpu(), want_slots)


def test_prefill_tables_follow_lengths_and_streams(cuda_device):
    """One pool, several lengths and streams in turn: prefill builds its table again when the lengths or
    the stream change, takes the same one when neither does, and writes the pages of every call
    where they belong."""
    announce("prefill tables per lengths and stream")
    g = torch.Generator(device="cuda")
    g.manual_seed(4)
    side = torch.cuda.Stream()
    cache, ref = (PagedKVCache(2, 64, batch=2, num_blocks=6, device=cuda_device, seed=5) for _ in range(2))
    for b in range(2):
        cache.reserve(b, 40)
        ref.reserve(b, 40)
    last = None
    for lengths, stream in (([20, 30], None), ([30, 20], None), ([30, 20], None), ([30, 20], side), ([30, 20], side),
                            ([20, 30], side), ([20, 30], None), ([17, 33], None), ([17, 33], side)):
        k = torch.randn((50, 2, 64), generator=g, device="cuda").to(torch.bfloat16)
        torch.cuda.synchronize()
        with torch.cuda.stream(stream or torch.cuda.current_stream()):
            slots = cache.prefill(0, k, k, lengths)
            table = cache._tiles[2]
            cache.prefill(0, k, k, lengths, slots)
            assert cache._tiles[2] is table, "same lengths, same stream, slots passed: same table"
        torch.cuda.synchronize()
        key = (tuple(lengths), (stream or torch.cuda.current_stream()).cuda_stream)
        assert cache._tiles[:2] == key
        assert torch.equal(cache._tiles[2].cpu(), _host(cache, lengths)[1])
        if last is not None and last[0] != key:
            assert cache._tiles[2] is not last[1], "other lengths or another stream: another table"
        last = key, cache._tiles[2]
        ops.quant_append(k, _host(ref, lengths)[0].cuda(), *ref.layer(0), k)
        torch.cuda.synchronize()
        for x, y in zip(cache.layer(0), ref.layer(0)):
            assert torch.equal(x, y)


def test_varlen_slots_refuse_unreserved_positions(cuda_device):
    cache = PagedKVCache(2, 64, batch=2, num_blocks=8, device=cuda_device)
    cache.reserve(0, 40)
    with pytest.raises(IndexError):
        cache.varlen_slots([49])
    with pytest.raises(RuntimeError):
        ops.varlen_slots(cache.block_table(), [1, 2, 3])


def _replay_test(cuda_device, warm, record):
    """Record prefill with the slots of a warm-up on stream `warm` (capture stream `record`), then
    replay it with new K and V between eager prefills that replace the pool's tables, with whatever
    those freed overwritten; every replay gives the pages of the same call run eagerly."""
    g = torch.Generator(device="cuda")
    g.manual_seed(11)
    lengths, others = [37, 80, 5], ([80, 5, 37], [37, 80, 5], [1, 1, 1])
    k = torch.zeros((sum(lengths), 2, 64), dtype=torch.bfloat16, device="cuda")
    v = torch.zeros_like(k)
    cache = PagedKVCache(2, 64, batch=3, num_blocks=18, device=cuda_device, seed=12, growable=False)
    for b in range(3):
        cache.reserve(b, 80)
    torch.cuda.synchronize()
    with torch.cuda.stream(warm):
        slots = cache.prefill(0, k, v, lengths)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=record):
        cache.prefill(0, k, v, lengths, slots)
    for i, other in enumerate(others):
        with torch.cuda.stream(torch.cuda.Stream() if i % 2 else record):
            cache.prefill(0, *(2 * [torch.randn((sum(other), 2, 64), generator=g, device="cuda").to(torch.bfloat16)]), other)
        torch.cuda.synchronize()
        junk = [torch.full((n,), 3, dtype=torch.int32, device="cuda") for n in (8, 16, 64, 128, 256) for _ in range(8)]
        k.copy_(torch.randn(k.shape, generator=g, device="cuda"))
        v.copy_(torch.randn(k.shape, generator=g, device="cuda"))
        for x in (cache.k_pages, cache.v_pages, cache.v_scales):
            x.zero_()
        graph.replay()
        torch.cuda.synchronize()
        ref = PagedKVCache(2, 64, batch=3, num_blocks=18, device=cuda_device, seed=12, growable=False)
        for x in (ref.k_pages, ref.v_pages, ref.v_scales):
            x.zero_()
        ops.quant_append(v, slots, *ref.layer(0), k)
        torch.cuda.synchronize()
        for x, y in zip(cache.layer(0), ref.layer(0)):
            assert torch.equal(x, y), f"replay {i}"
        del junk


def test_recorded_prefill_keeps_its_table(cuda_device):
    """A table that a graph reads outlives the prefills that replace it."""
    announce("recorded prefill, table kept")
    side = torch.cuda.Stream()
    _replay_test(cuda_device, side, side)


def test_prefill_records_on_another_stream(cuda_device):
    """The warm-up's table serves a recording on the capture stream, as torch.cuda.graph makes one;
    lengths not called before, and a recording without slots, are refused before anything is copied,
    and the recording goes on."""
    announce("recorded prefill, capture stream")
    _replay_test(cuda_device, torch.cuda.Stream(), torch.cuda.Stream())
    _replay_test(cuda_device, torch.cuda.current_stream(), torch.cuda.Stream())
    k = torch.randn((40, 2, 64), device="cuda").to(torch.bfloat16)
    cache = PagedKVCache(2, 64, batch=1, num_blocks=4, device=cuda_device)
    slots = cache.prefill(0, k, k, [40])
    torch.cuda.synchronize()
    want = [x.clone() for x in cache.layer(0)]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        with pytest.raises(SdvError, match="recorded"):
            cache.prefill(0, k, k, [40])
        with pytest.raises(SdvError, match="recorded"):
            cache.prefill(0, k[:39], k[:39], [39], slots[:39])
        with pytest.raises(SdvError, match="recorded"):
            cache.varlen_slots([40])
        cache.prefill(0, k, k, [40], slots)
    for _ in range(3):
        for x in cache.layer(0):
            x.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for x, y in zip(cache.layer(0), want):
            assert torch.equal(x[cache.blocks[0][:2]], y[cache.blocks[0][:2]])   # whole blocks


def test_prefill_takes_slots_of_a_busy_stream(cuda_device):
    """Slots made on one stream and passed to a later layer's prefill on another: the second stream
    waits for the kernel that writes them, also where its own table need not be built again."""
    announce("prefill, slots of a busy stream")
    lengths = [300, 41]
    k = torch.randn((sum(lengths), 2, 64), device="cuda").to(torch.bfloat16)
    cache, ref = (PagedKVCache(2, 64, num_layers=3, batch=2, num_blocks=24, device=cuda_device, seed=6) for _ in range(2))
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    x = torch.randn((4096, 4096), device="cuda").to(torch.bfloat16)
    for c in (cache, ref):
        for i, n in enumerate(lengths):
            c.reserve(i, n)
        c.block_table()
    torch.cuda.synchronize()

    def busy():
        for _ in range(200):
            x @ x

    with torch.cuda.stream(a):
        busy()
        slots = cache.prefill(0, k, k, lengths)
    with torch.cuda.stream(b):
        cache.prefill(1, k, k, lengths, slots)
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        busy()
        again = cache.varlen_slots(lengths)
    with torch.cuda.stream(b):
        cache.prefill(2, k, k, lengths, again)
    torch.cuda.synchronize()
    for layer in range(3):
        ops.quant_append(k, _host(ref, lengths)[0].cuda(), *ref.layer(layer), k)
    torch.cuda.synchronize()
    assert torch.equal(cache.k_pages, ref.k_pages) and torch.equal(cache.v_pages, ref.v_pages)
