"""Slots and tile tables of packed prompts written on the device, against the host's."""
from __future__ import annotations

import random

import pytest
import torch

from conftest import announce
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
    """prefill reuses a table only for the same lengths on the same stream."""
    announce("prefill tables per lengths and stream")
    g = torch.Generator(device="cuda")
    g.manual_seed(4)
    k = torch.randn((50, 2, 64), generator=g, device="cuda").to(torch.bfloat16)
    side = torch.cuda.Stream()
    for lengths in ([20, 30], [30, 20], [30, 20]):
        for stream in (torch.cuda.current_stream(), side):
            cache = PagedKVCache(2, 64, batch=2, num_blocks=6, device=cuda_device, seed=5)
            ref = PagedKVCache(2, 64, batch=2, num_blocks=6, device=cuda_device, seed=5)
            with torch.cuda.stream(stream):
                stream.wait_stream(torch.cuda.default_stream())
                for _ in range(2):
                    cache.prefill(0, k, k, lengths)
            torch.cuda.synchronize()
            for b in range(2):
                ref.reserve(b, lengths[b])
            ops.quant_append(k, _host(ref, lengths)[0].cuda(), *ref.layer(0), k)
            torch.cuda.synchronize()
            assert torch.equal(cache.k_pages, ref.k_pages) and torch.equal(cache.v_pages, ref.v_pages)
    assert cache._tiles[:2] == ((30, 20), side.cuda_stream)


def test_varlen_slots_refuse_unreserved_positions(cuda_device):
    cache = PagedKVCache(2, 64, batch=2, num_blocks=8, device=cuda_device)
    cache.reserve(0, 40)
    with pytest.raises(IndexError):
        cache.varlen_slots([49])
    with pytest.raises(RuntimeError):
        ops.varlen_slots(cache.block_table(), [1, 2, 3])
