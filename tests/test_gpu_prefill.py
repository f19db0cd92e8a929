"""Paged prefill / chunked-prefill attention (many query rows) against the eager oracle.

Reference: the prefill chunk of model_self.py:637-648 (2048-token chunks) attends over the
cache plus the chunk with the offset-causal keep-mask of model_self.py:471-479 (row i sees keys
j <= T - S + i); its fused path (cuDNN SDPA, :491-504) exists to avoid the O(S*T) score tensor
of the eager path (docs/data_ledger.md:1145-1152: 74.1 MiB transient at 12q/2048q/8192kv).
Here the two prefill passes keep 64 bytes per query row in the workspace (a (max, sum) for
each of eight key parts); the numbers must still be the eager BF16 path's (max-abs 2e-2,
rel-L2 1e-3 per row block).  The oracle runs on the
CPU in row chunks (row i of a chunk of rows [i0, i1) sees keys j <= T - S + i0 + i, the same
mask), so its memory stays bounded.
"""
from __future__ import annotations

import pytest
import torch

from conftest import announce
from helpers import assert_close
from oracle import attention as oatt
from oracle import quant as oq
from specdec_amd import _native
from specdec_amd import workloads as wl
from specdec_amd.engine.paged_cache import PagedKVCache
from specdec_amd.kernels import ops

pytestmark = pytest.mark.gpu


def _oracle_rows(q, k, v_hat, i0, i1, t):
    """Eager attention of rows [i0, i1) of an S-row block over T keys (all heads)."""
    s = q.shape[2]
    tk = t - s + i1
    return oatt.eager_attention(q[:, :, i0:i1], k[:, :, :tk], v_hat[:, :, :tk])


def _prefill_case(dev, h, kv, d, s, t, seed, chunk_rows=256, check_rows=None):
    g = wl.gen(seed, dev)
    cache = PagedKVCache(kv, d, num_blocks=t // 16 + 11, device=dev, seed=seed, growable=False)
    k = torch.randn((t, kv, d), generator=g, device=dev).to(torch.bfloat16)
    v = torch.randn((t, kv, d), generator=g, device=dev).to(torch.bfloat16)
    cache.prefill(0, k, v, [t])
    q = torch.randn((1, h, s, d), generator=g, device=dev).to(torch.bfloat16)
    kp, vp, vs = cache.layer(0)
    nbytes = ops.attention_workspace_bytes(1, 1, h, kv, s, d, t)
    ws = ops.new_workspace(dev, nbytes)
    out = ops.paged_attention(q, kp, vp, vs, cache.block_table(), cache.seq_lens_tensor(), t, workspace_tensor=ws)
    torch.cuda.synchronize()
    kc, vc, sc = cache.gather(0, 0)
    v_hat = oq.dequantize_kv_fp8(vc.cpu()[None], sc.cpu()[None], torch.bfloat16)
    qc, kcc = q.cpu(), kc.cpu()[None]
    rows = check_rows or [(i, min(s, i + chunk_rows)) for i in range(0, s, chunk_rows)]
    worst = (0.0, 0.0)
    for i0, i1 in rows:
        want = _oracle_rows(qc, kcc, v_hat, i0, i1, t)
        st = assert_close(out[:, :, i0:i1].cpu(), want, f"{h}/{kv}/{d} S={s} T={t} rows {i0}:{i1}")
        worst = (max(worst[0], st["max_abs"]), max(worst[1], st["rel_l2"]))
    return nbytes, worst


def test_prefill_chunk_target_2048x8192(cuda_device):
    """The reference's target prefill chunk: 12 query heads, 2048 query rows over 8192 keys."""
    announce("prefill 12/2/128 S=2048 T=8192")
    nbytes, worst = _prefill_case(cuda_device, 12, 2, 128, 2048, 8192, seed=700)
    print(f"workspace {nbytes / 2**20:.2f} MiB, worst max-abs {worst[0]:.3e} rel-L2 {worst[1]:.3e}")
    assert nbytes <= 100 * 2**20


def test_prefill_chunk_draft_2048x8192(cuda_device):
    """The draft's prefill chunk: 14 query heads, head_dim 64."""
    announce("prefill 14/2/64 S=2048 T=8192")
    nbytes, worst = _prefill_case(cuda_device, 14, 2, 64, 2048, 8192, seed=701)
    print(f"workspace {nbytes / 2**20:.2f} MiB, worst max-abs {worst[0]:.3e} rel-L2 {worst[1]:.3e}")
    assert nbytes <= 100 * 2**20


@pytest.mark.parametrize("h,d,s,t", [(12, 128, 2048, 2048), (12, 128, 300, 1000), (14, 64, 33, 77),
                                     (12, 128, 11, 40000), (12, 128, 1000, 1000), (14, 64, 11, 270000)])
def test_prefill_shapes(cuda_device, h, d, s, t):
    """A first chunk from an empty cache (T = S, triangular mask), odd sizes, short blocks over
    long contexts and S not a multiple of 16; at T = 270,000 (4,219 stages of 64 keys for each of
    two row groups) pass 1's statistics hold 64 segments per row."""
    announce(f"prefill {h}/2/{d} S={s} T={t}")
    _prefill_case(cuda_device, h, 2, d, s, t, seed=710 + s + t, chunk_rows=512)


@pytest.mark.parametrize("s,h,d", [(96, 12, 128), (256, 12, 128), (256, 14, 64)])
def test_prefill_ragged_batch_token_major(cuda_device, s, h, d):
    """Two sequences of different lengths in one call, q in the projection layout (B, S, H, D).
    The launches are sized for the longest sequence and the ranges of stages cut from the
    actual lengths; S = 256 takes the workspace of S a multiple of 128."""
    announce(f"prefill ragged batch, token-major q, S={s} {h}/2/{d}")
    g = wl.gen(720 + s + d, cuda_device)
    lens, kv = [3000, 700], 2
    cache = PagedKVCache(kv, d, batch=2, num_blocks=sum(-(-x // 16) for x in lens) + 5, device=cuda_device,
                         seed=721, growable=False)
    k = torch.randn((sum(lens), kv, d), generator=g, device=cuda_device).to(torch.bfloat16)
    v = torch.randn((sum(lens), kv, d), generator=g, device=cuda_device).to(torch.bfloat16)
    cache.prefill(0, k, v, lens)
    q = torch.randn((2, s, h, d), generator=g, device=cuda_device).to(torch.bfloat16)
    kp, vp, vs = cache.layer(0)
    assert ops.single_launch_workgroups(1, 2, h, kv, s, d, max(lens)) == 0
    out = ops.paged_attention(q, kp, vp, vs, cache.block_table(), cache.seq_lens_tensor(), max(lens),
                              q_token_major=True)
    torch.cuda.synchronize()
    for b, t in enumerate(lens):
        kc, vc, sc = cache.gather(0, b)
        v_hat = oq.dequantize_kv_fp8(vc.cpu()[None], sc.cpu()[None], torch.bfloat16)
        want = oatt.eager_attention(q[b:b + 1].transpose(1, 2).cpu(), kc.cpu()[None], v_hat)
        assert_close(out[b:b + 1].transpose(1, 2).cpu(), want, f"ragged b={b} T={t}")


def test_prefill_multi_layer_call(cuda_device):
    """Two layers x two ragged sequences of 128 new rows in one call (q in the projection layout
    (L, B, S, H, D)): every (layer, sequence) pair has its own pass-1 statistics, dequantized V
    and pass-2 parts, and each output is within the bar of the eager reference."""
    announce("prefill 2 layers x 2 ragged sequences, S=128, one call")
    g = wl.gen(725, cuda_device)
    L, lens, s, h, kv, d = 2, [2500, 900], 128, 12, 2, 128
    cache = PagedKVCache(kv, d, num_layers=L, batch=2, num_blocks=sum(-(-x // 16) for x in lens) + 5,
                         device=cuda_device, seed=726, growable=False)
    slots = None
    for layer in range(L):
        k = torch.randn((sum(lens), kv, d), generator=g, device=cuda_device).to(torch.bfloat16)
        v = torch.randn((sum(lens), kv, d), generator=g, device=cuda_device).to(torch.bfloat16)
        slots = cache.prefill(layer, k, v, lens, slots)
    q = torch.randn((L, 2, s, h, d), generator=g, device=cuda_device).to(torch.bfloat16)
    out = ops.paged_attention(q, cache.k_pages, cache.v_pages, cache.v_scales, cache.block_table(),
                              cache.seq_lens_tensor(), max(lens), q_token_major=True)
    torch.cuda.synchronize()
    for layer in range(L):
        for b, t in enumerate(lens):
            kc, vc, sc = cache.gather(layer, b)
            v_hat = oq.dequantize_kv_fp8(vc.cpu()[None], sc.cpu()[None], torch.bfloat16)
            want = oatt.eager_attention(q[layer, b:b + 1].transpose(1, 2).cpu(), kc.cpu()[None], v_hat)
            assert_close(out[layer, b:b + 1].transpose(1, 2).cpu(), want, f"layer {layer} b={b} T={t}")


def test_prefill_deterministic(cuda_device):
    """Repeated calls are bitwise identical (fixed-order reductions, no atomics)."""
    announce("prefill determinism")
    g = wl.gen(730, cuda_device)
    cache = PagedKVCache(2, 128, num_blocks=140, device=cuda_device, seed=731, growable=False)
    t = 2000
    cache.prefill(0, torch.randn((t, 2, 128), generator=g, device=cuda_device).to(torch.bfloat16),
                  torch.randn((t, 2, 128), generator=g, device=cuda_device).to(torch.bfloat16), [t])
    q = torch.randn((1, 12, 500, 128), generator=g, device=cuda_device).to(torch.bfloat16)
    kp, vp, vs = cache.layer(0)
    outs = [ops.paged_attention(q, kp, vp, vs, cache.block_table(), cache.seq_lens_tensor(), t) for _ in range(3)]
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[1], outs[2])


@pytest.mark.parametrize("h,d,s", [(14, 64, 300), (12, 128, 300), (12, 128, 256)])
def test_prefill_key_parts_repeat_and_replay(cuda_device, h, d, s):
    """Row groups that several workgroups' ranges cut leave their parts in slots, which a third
    launch sums: repeated eager calls and the replays of a recorded call -- which reuse one tag -- with eager calls between them are bitwise equal, on
    a batch of two sequences; S = 256 takes the workspace of S a multiple of 128."""
    announce(f"prefill {h}/2/{d} S={s} key parts: repeats and graph replays")
    g = wl.gen(740 + d + s, cuda_device)
    lens, kv = [3000, 1200], 2
    cache = PagedKVCache(kv, d, batch=2, num_blocks=sum(-(-x // 16) for x in lens) + 5, device=cuda_device,
                         seed=741, growable=False)
    cache.prefill(0, torch.randn((sum(lens), kv, d), generator=g, device=cuda_device).to(torch.bfloat16),
                  torch.randn((sum(lens), kv, d), generator=g, device=cuda_device).to(torch.bfloat16), lens)
    q = torch.randn((2, s, h, d), generator=g, device=cuda_device).to(torch.bfloat16)
    kp, vp, vs = cache.layer(0)
    bt, sl = cache.block_table(), cache.seq_lens_tensor()
    ws = ops.new_workspace(cuda_device, ops.attention_workspace_bytes(1, 2, h, kv, s, d, max(lens)))

    def call(out=None):
        return ops.paged_attention(q, kp, vp, vs, bt, sl, max(lens), q_token_major=True, out=out, workspace_tensor=ws)

    eager = [call() for _ in range(3)]
    torch.cuda.synchronize()
    assert torch.equal(eager[0], eager[1]) and torch.equal(eager[1], eager[2])
    out = torch.empty_like(q)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(out)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        call(out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager[0]), "a replay differs from the eager call"
        again = call()
        torch.cuda.synchronize()
        assert torch.equal(again, eager[0]), "an eager call after a replay differs"
    for b, t in enumerate(lens):  # and the numbers are the eager path's
        kc, vc, sc = cache.gather(0, b)
        v_hat = oq.dequantize_kv_fp8(vc.cpu()[None], sc.cpu()[None], torch.bfloat16)
        want = oatt.eager_attention(q[b:b + 1].transpose(1, 2).cpu(), kc.cpu()[None], v_hat)
        assert_close(eager[0][b:b + 1].transpose(1, 2).cpu(), want, f"key parts b={b} T={t}")


def test_prefill_many_row_groups_and_windows(cuda_device):
    """260 row groups of one layer without part slots (130 sequences of 11 new rows): a workgroup
    takes whole row groups, and at T = 33,000 (2,063 blocks) both passes stage the page ids in two
    windows of 2,048.  The sequences share one sequence's pages; the first and the last are
    checked."""
    announce("prefill 130 sequences S=11 T=33000 (whole row groups, two page-id windows)")
    b, h, kv, d, s, t = 130, 12, 2, 128, 11, 33000
    g = wl.gen(750, cuda_device)
    cache = PagedKVCache(kv, d, num_blocks=t // 16 + 3, device=cuda_device, seed=751, growable=False)
    cache.prefill(0, torch.randn((t, kv, d), generator=g, device=cuda_device).to(torch.bfloat16),
                  torch.randn((t, kv, d), generator=g, device=cuda_device).to(torch.bfloat16), [t])
    q = torch.randn((b, s, h, d), generator=g, device=cuda_device).to(torch.bfloat16)
    kp, vp, vs = cache.layer(0)
    out = ops.paged_attention(q, kp, vp, vs, cache.block_table().expand(b, -1).contiguous(), None, t, q_token_major=True)
    torch.cuda.synchronize()
    kc, vc, sc = cache.gather(0, 0)
    v_hat = oq.dequantize_kv_fp8(vc.cpu()[None], sc.cpu()[None], torch.bfloat16)
    for i in (0, b - 1):
        want = oatt.eager_attention(q[i:i + 1].transpose(1, 2).cpu(), kc.cpu()[None], v_hat)
        assert_close(out[i:i + 1].transpose(1, 2).cpu(), want, f"sequence {i}")


@pytest.mark.parametrize("h,d,s,t", [(12, 128, 2048, 131072), (14, 64, 1500, 150001)])
def test_prefill_ranges_over_page_id_windows(cuda_device, h, d, s, t):
    """Ranges of more than 512 stages stage their page ids in several windows of 2,048 that begin where
    the range does (769 stages a workgroup for 2048 rows over 128K keys, 768 and more for 1500 over
    150,001); the first, two middle and the last rows are checked."""
    announce(f"prefill {h}/2/{d} S={s} T={t} page-id windows inside ranges")
    rows = 256
    stages = sum(6 + (t - s + min(s - 1, (rows * (i + 1) - 1) // (h // 2)) + 64) // 64 for i in range(-(-s * (h // 2) // rows)))
    assert 2 * stages > 256 * 512, "a workgroup's range is longer than a window"
    _prefill_case(cuda_device, h, 2, d, s, t, seed=755 + d,
                  check_rows=[(0, 4), (s // 3, s // 3 + 4), (s // 2, s // 2 + 4), (s - 4, s)])


@pytest.mark.parametrize("h,d,s,t", [(12, 128, 300, 1500), (14, 64, 96, 900)])
def test_prefill_late_maximum(cuda_device, h, d, s, t):
    """Pass 1 takes its exponentials against an earlier maximum and goes through the online update
    where a sum would leave its bound: scores that jump by far more than 88 in a later stage of the
    same segment, so that the exponentials themselves overflow."""
    announce(f"prefill late maximum {h}/2/{d} S={s} T={t}")
    g = wl.gen(760 + d, cuda_device)
    cache = PagedKVCache(2, d, num_blocks=t // 16 + 3, device=cuda_device, seed=761, growable=False)
    k = torch.randn((t, 2, d), generator=g, device=cuda_device)
    for at in (200, 500, 777):   # past the first stage of a segment that begins at key 0, 256 or 512
        k[at] = 4.0
    v = torch.randn((t, 2, d), generator=g, device=cuda_device).to(torch.bfloat16)
    q = (torch.randn((1, h, s, d), generator=g, device=cuda_device) * 0.25 + 4.0).to(torch.bfloat16)
    cache.prefill(0, k.to(torch.bfloat16), v, [t])
    kp, vp, vs = cache.layer(0)
    out = ops.paged_attention(q, kp, vp, vs, cache.block_table(), cache.seq_lens_tensor(), t)
    torch.cuda.synchronize()
    kc, vc, sc = cache.gather(0, 0)
    v_hat = oq.dequantize_kv_fp8(vc.cpu()[None], sc.cpu()[None], torch.bfloat16)
    assert_close(out.cpu(), oatt.eager_attention(q.cpu(), kc.cpu()[None], v_hat), "late maximum")


def test_prefill_skips_invalid_blocks(cuda_device):
    """Block ids outside the pool are never read and their tokens are masked, in the pages every
    row sees and on the diagonal: the output of the same call over a cache without those tokens."""
    announce("prefill with invalid block ids")
    h, kv, d, s, t = 12, 2, 128, 128, 1600
    g = wl.gen(770, cuda_device)
    k = torch.randn((t, kv, d), generator=g, device=cuda_device).to(torch.bfloat16)
    v = torch.randn((t, kv, d), generator=g, device=cuda_device).to(torch.bfloat16)
    cache = PagedKVCache(kv, d, num_blocks=t // 16 + 3, device=cuda_device, seed=771, growable=False)
    cache.prefill(0, k, v, [t])
    q = torch.randn((1, h, s, d), generator=g, device=cuda_device).to(torch.bfloat16)
    kp, vp, vs = cache.layer(0)
    holes = [3, 4, 40, 71, 99]   # 99: the last block, on the diagonal
    table = cache.block_table().clone()
    table[0, holes] = torch.tensor([-1, 1 << 20, -5, cache.alloc.num_blocks, -1], dtype=torch.int32, device=cuda_device)
    out = ops.paged_attention(q, kp, vp, vs, table, cache.seq_lens_tensor(), t)
    torch.cuda.synchronize()
    kc, vc, sc = cache.gather(0, 0)
    v_hat = oq.dequantize_kv_fp8(vc.cpu()[None], sc.cpu()[None], torch.bfloat16)
    keep = torch.ones(t, dtype=torch.bool)
    for j in holes:
        keep[16 * j:16 * j + 16] = False
    pos = torch.nonzero(keep).flatten()
    for i in (0, 50, 127):       # row i sees the kept keys up to t - s + i
        n = int((pos <= t - s + i).sum())
        want = oatt.eager_attention(q[:, :, i:i + 1].cpu(), kc.cpu()[None][:, :, pos[:n]], v_hat[:, :, pos[:n]])
        assert_close(out[:, :, i:i + 1].cpu(), want, f"row {i}")


@pytest.mark.parametrize("where", ["halves", "segments", "low"])
@pytest.mark.parametrize("jump", [20.0, 60.0, 82.0, 88.5])
@pytest.mark.parametrize("h,d", [(12, 128), (14, 64)])
def test_prefill_finite_jumps(cuda_device, h, d, jump, where):
    """Pass 1 sums exponentials against an earlier maximum; scores that jump by less than what
    overflows one exponential (88.7) must neither overflow the sums that are merged afterwards --
    of a row's two lanes (keys 3 and 5 of a stage: "halves") or of its segments (one key in every
    other stage: "segments") -- nor, 200 below zero ("low"), lose a segment whose maximum the merge
    finds far below another's.  Every element of q is 1, so the scores are exact."""
    announce(f"prefill finite jumps {h}/2/{d} {where} {jump}")
    g = wl.gen(780 + d, cuda_device)
    s, t, base = 80, 2048, -200.0 if where == "low" else 0.0
    score = torch.full((t,), base, device=cuda_device)
    score[(torch.arange(2, t // 64, 7, device=cuda_device)[:, None] * 64 + torch.tensor([3, 5], device=cuda_device)).flatten()
          if where == "halves" else torch.arange(67, t, 128, device=cuda_device)] = base + jump
    k = (score / d ** 0.5)[:, None, None].expand(t, 2, d).to(torch.bfloat16).contiguous()
    v = torch.randn((t, 2, d), generator=g, device=cuda_device).to(torch.bfloat16)
    q = torch.ones((1, h, s, d), dtype=torch.bfloat16, device=cuda_device)
    cache = PagedKVCache(2, d, num_blocks=t // 16 + 3, device=cuda_device, seed=781, growable=False)
    cache.prefill(0, k, v, [t])
    kp, vp, vs = cache.layer(0)
    out = ops.paged_attention(q, kp, vp, vs, cache.block_table(), cache.seq_lens_tensor(), t)
    torch.cuda.synchronize()
    kc, vc, sc = cache.gather(0, 0)
    v_hat = oq.dequantize_kv_fp8(vc.cpu()[None], sc.cpu()[None], torch.bfloat16)
    assert_close(out.cpu(), oatt.eager_attention(q.cpu(), kc.cpu()[None], v_hat), f"{where} {jump}")


@pytest.mark.parametrize("h,d,s,t", [(12, 128, 300, 1500), (14, 64, 777, 3000)])
def test_prefill_wide_scores(cuda_device, h, d, s, t):
    """Scores of N(0, 45^2): a row's maximum rises by far more than an exponential's range, in
    steps.  Whole numbers in q and K, so that both sides round the same products."""
    announce(f"prefill wide scores {h}/2/{d} S={s} T={t}")
    g = wl.gen(790 + d, cuda_device)
    k = torch.randint(-11, 12, (t, 2, d), generator=g, device=cuda_device).to(torch.bfloat16)
    v = torch.randn((t, 2, d), generator=g, device=cuda_device).to(torch.bfloat16)
    q = torch.randint(-11, 12, (1, h, s, d), generator=g, device=cuda_device).to(torch.bfloat16)
    cache = PagedKVCache(2, d, num_blocks=t // 16 + 3, device=cuda_device, seed=791, growable=False)
    cache.prefill(0, k, v, [t])
    kp, vp, vs = cache.layer(0)
    out = ops.paged_attention(q, kp, vp, vs, cache.block_table(), cache.seq_lens_tensor(), t)
    torch.cuda.synchronize()
    kc, vc, sc = cache.gather(0, 0)
    v_hat = oq.dequantize_kv_fp8(vc.cpu()[None], sc.cpu()[None], torch.bfloat16)
    assert_close(out.cpu(), oatt.eager_attention(q.cpu(), kc.cpu()[None], v_hat), "wide scores")


@pytest.mark.parametrize("h,d,s,lens", [(12, 128, 80, [700, 0, 300]), (14, 64, 96, [0, 500]),
                                        (12, 128, 11, [300] * 64 + [0] * 3 + [300] * 63)])
def test_prefill_empty_sequence(cuda_device, h, d, s, lens):
    """A sequence without tokens in a prefill batch gives zeros whatever the workspace held (NaN bits
    here), in ranges of stages and (130 sequences) in whole row groups; the others are as without
    it.  The sequences share one sequence's pages."""
    announce(f"prefill with empty sequences {h}/2/{d} S={s} batch {len(lens)}")
    g = wl.gen(800 + d + s, cuda_device)
    t, b = max(lens), len(lens)
    cache = PagedKVCache(2, d, num_blocks=t // 16 + 3, device=cuda_device, seed=801, growable=False)
    cache.prefill(0, torch.randn((t, 2, d), generator=g, device=cuda_device).to(torch.bfloat16),
                  torch.randn((t, 2, d), generator=g, device=cuda_device).to(torch.bfloat16), [t])
    q = torch.randn((b, h, s, d), generator=g, device=cuda_device).to(torch.bfloat16)
    kp, vp, vs = cache.layer(0)
    ws = ops.new_workspace(cuda_device, ops.attention_workspace_bytes(1, b, h, 2, s, d, t))
    ws[_native.SYNC_BYTES:] = 0xFF
    out = ops.paged_attention(q, kp, vp, vs, cache.block_table().expand(b, -1).contiguous(),
                              torch.tensor(lens, dtype=torch.int32, device=cuda_device), t, workspace_tensor=ws)
    torch.cuda.synchronize()
    kc, vc, sc = cache.gather(0, 0)
    v_hat = oq.dequantize_kv_fp8(vc.cpu()[None], sc.cpu()[None], torch.bfloat16)
    for i, n in enumerate(lens):
        if n == 0:
            assert not out[i].any(), f"sequence {i} is empty"
        elif i < 3 or i == b - 1:
            want = oatt.eager_attention(q[i:i + 1].cpu(), kc.cpu()[None][:, :, :n], v_hat[:, :, :n])
            assert_close(out[i:i + 1].cpu(), want, f"sequence {i} of {n}")


@pytest.mark.parametrize("h,d,s,t", [(12, 128, 11, 11), (12, 128, 11, 384), (12, 128, 11, 385), (12, 128, 21, 64), (12, 128, 22, 65),
                                     (12, 128, 64, 512), (12, 128, 64, 513), (12, 128, 400, 640), (14, 64, 10, 16), (14, 64, 19, 576),
                                     (14, 64, 37, 577), (14, 64, 73, 704), (14, 64, 73, 705), (14, 64, 350, 768)])
def test_prefill_short_contexts(cuda_device, h, d, s, t):
    """Calls over few stages of keys take row groups of 128 rows, a workgroup of four wavefronts each:
    one row group and the first rows of a second, one stage and one key past it, and both sides of
    the rule's limits (6, 8, 10 and 9, 11, 12 stages by the number of row groups)."""
    announce(f"prefill short {h}/2/{d} S={s} T={t}")
    _prefill_case(cuda_device, h, 2, d, s, t, seed=810 + s + t, chunk_rows=128)


@pytest.mark.parametrize("h,d", [(12, 128), (14, 64)])
def test_prefill_short_ragged_batch_replays(cuda_device, h, d):
    """Two layers of five short sequences (one shorter than the new rows, one empty) with invalid block
    ids in one of them, recorded and replayed between eager calls: equal to the eager call, and
    within the bar of the eager reference over the valid keys."""
    announce(f"prefill short ragged batch {h}/2/{d}")
    g = wl.gen(830 + d, cuda_device)
    L, lens, s, kv = 2, [400, 45, 20, 0, 333], 45, 2
    t, rows = max(lens), [0, 1, 2, 4]
    cache = PagedKVCache(kv, d, num_layers=L, batch=5, num_blocks=sum(-(-x // 16) for x in lens) + 5, device=cuda_device,
                         seed=831, growable=False)
    slots = None
    for layer in range(L):
        k = torch.randn((sum(lens), kv, d), generator=g, device=cuda_device).to(torch.bfloat16)
        v = torch.randn((sum(lens), kv, d), generator=g, device=cuda_device).to(torch.bfloat16)
        slots = cache.prefill(layer, k, v, lens, slots)
    table = cache.block_table().clone()
    holes = [0, 7, 20]
    table[4, holes] = torch.tensor([-1, 1 << 20, cache.alloc.num_blocks], dtype=torch.int32, device=cuda_device)
    sl = cache.seq_lens_tensor()
    q = torch.randn((L, 5, s, h, d), generator=g, device=cuda_device).to(torch.bfloat16)
    ws = ops.new_workspace(cuda_device, ops.attention_workspace_bytes(L, 5, h, kv, s, d, t))

    def call(out=None):
        return ops.paged_attention(q, cache.k_pages, cache.v_pages, cache.v_scales, table, sl, t, q_token_major=True, out=out,
                                   workspace_tensor=ws)

    want = call()
    out = torch.empty_like(q)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), "a replay differs from the eager call"
        assert torch.equal(call(), want)
    torch.cuda.synchronize()
    for layer in range(L):
        assert not want[layer, 3].any()
        for b in rows:
            n = lens[b]
            kc, vc, sc = cache.gather(layer, b)
            v_hat = oq.dequantize_kv_fp8(vc.cpu()[None], sc.cpu()[None], torch.bfloat16)
            keep = torch.ones(n, dtype=torch.bool)
            for j in holes if b == 4 else []:
                keep[16 * j:16 * j + 16] = False
            pos = torch.nonzero(keep).flatten()
            for i in (0, 1, 26, s - 1):
                m = int((pos <= n - s + i).sum())
                got = want[layer, b, i].cpu()[None, :, None]
                if m == 0:
                    assert not got.any(), f"row {i} of sequence {b} sees no key"
                    continue
                ref = oatt.eager_attention(q[layer, b, i].cpu()[None, :, None], kc.cpu()[None][:, :, pos[:m]], v_hat[:, :, pos[:m]])
                assert_close(got, ref, f"layer {layer} sequence {b} row {i}")
