"""The contiguous-cache op: its pages against pack_contiguous's bytes, its output against the paged op."""
from __future__ import annotations

import pytest
import torch

from conftest import announce
from specdec_amd import _native
from specdec_amd.kernels import ops

pytestmark = pytest.mark.gpu


def _cache(b, kv, t, d, seed, shift=0):
    """k, payload (every code, NaNs among them), scale; shift: tensors that start mid-allocation."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def at(x):
        buf = torch.empty(x.numel() + shift, dtype=x.dtype, device="cuda")
        buf[shift:] = x.flatten()
        return buf[shift:].view(x.shape)

    k = at(torch.randn((b, kv, t, d), generator=g, device="cuda").to(torch.bfloat16))
    v = at(torch.randint(0, 256, (b, kv, t, d), generator=g, device="cuda", dtype=torch.uint8))
    return k, v, at(torch.rand((b, kv, t, 1), generator=g, device="cuda") + 0.01)


@pytest.mark.parametrize("b,kv,t,d", [(1, 2, 1, 128), (1, 1, 15, 64), (2, 2, 16, 128), (3, 2, 17, 64), (1, 3, 333, 128),
                                      (2, 2, 4097, 64)])
def test_pages_are_pack_contiguous_bytes(cuda_device, b, kv, t, d):
    """One wavefront per page, pages times KV heads not a multiple of a workgroup's four, tokens
    past the end of the last block."""
    announce(f"pack contiguous {b}x{kv}x{t}x{d}")
    k, v, s = _cache(b, kv, t, d, seed=t + d)
    want = ops.pack_contiguous(k, v.view(torch.float8_e4m3fn), s)
    got = [torch.full_like(x.view(torch.uint8) if x.element_size() == 1 else x, 7) for x in want[:4]]
    st = torch.cuda.current_stream().cuda_stream
    rc = _native.load().sdv_pack_contiguous(k.data_ptr(), v.data_ptr(), s.data_ptr(), b, kv, t, d,
                                            *[x.data_ptr() for x in got], st)
    assert rc == _native.SDV_OK
    torch.cuda.synchronize()
    for x, y in zip(got, want):
        assert torch.equal(x.view(torch.uint8), y.contiguous().view(torch.uint8))


@pytest.mark.parametrize("b,t,s,h,kv,d,shift", [(1, 700, 1, 12, 2, 128, 0), (2, 333, 5, 14, 2, 64, 3), (1, 100, 40, 12, 2, 128, 1)])
def test_op_equals_the_paged_op(cuda_device, b, t, s, h, kv, d, shift):
    """ops.attention over the contiguous tensors (also ones that start off a 16-byte boundary)
    against ops.paged_attention over pack_contiguous's pages."""
    announce(f"contiguous op B={b} T={t} S={s} {h}/{kv}/{d} shift={shift}")
    k, v, sc = _cache(b, kv, t, d, seed=5 + t, shift=shift)
    v[(v & 0x7F) == 0x7F] = 0x30     # no NaN codes here: outputs are compared
    g = torch.Generator(device="cuda")
    g.manual_seed(9)
    q = torch.randn((b, h, s, d), generator=g, device="cuda").to(torch.bfloat16)
    got = ops.attention(q, k, (v.view(torch.float8_e4m3fn), sc))
    kp, vp, vs, bt, sl = ops.pack_contiguous(k, v, sc)
    want = ops.paged_attention(q, kp, vp, vs, bt, None, t)
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_op_refuses_what_it_cannot_take(cuda_device):
    k, v, sc = _cache(1, 2, 64, 128, seed=1)
    q = torch.zeros((1, 12, 1, 128), dtype=torch.bfloat16, device="cuda")
    for bad in ((q[..., :96].contiguous(), k, (v, sc)), (q, k, (v.to(torch.int16), sc)), (q, k, (v, sc.double())),
                (q[:, :11].contiguous(), k, (v, sc)), (q, k[:, :, :0], (v[:, :, :0], sc[:, :, :0])), (q.repeat(2, 1, 1, 1), k, (v, sc))):
        with pytest.raises(RuntimeError):
            ops.attention(*bad)
