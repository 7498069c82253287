"""GPU parity of paged decode at the edges of its partition sizes (64 to 512
tokens, chosen from the call's size) and of the merge's chunks of 16
partitions, against the float64 oracle, and the workspace rule on the CPU."""

import numpy as np
import pytest
import torch

from mlx_primitives import _native
from mlx_primitives.cache import paged_attention
from oracle import paged as op


def make(seed, lens, H_kv, D, dtype, bs, width):
    g = torch.Generator().manual_seed(seed)
    pages = [-(-n // bs) for n in lens]
    perm = torch.randperm(sum(pages) + 2, generator=g).to(torch.int32)
    tables = torch.full((len(lens), width), -1, dtype=torch.int32)
    at = 0
    for b, n in enumerate(pages):
        tables[b, :n] = perm[at:at + n]
        at += n
    shape = (sum(pages) + 2, bs, H_kv, D)
    return (torch.randn(shape, generator=g).to(dtype), torch.randn(shape, generator=g).to(dtype),
            tables, torch.tensor(lens, dtype=torch.int32))


# context lengths around one batch of loads, one partition, a chunk of 16 and 64
# partitions; capacity (pages of the tables) beyond the longest context
LENS = [1, 31, 32, 33, 63, 64, 65, 127, 128, 129, 1023, 1024, 1025, 4095, 4097, 0]


@pytest.mark.gpu
@pytest.mark.parametrize("lens,width", [(LENS, 260), ([4097], 300), ([65], 5), ([700, 1], 44)])
@pytest.mark.parametrize("H,H_kv,D,dtype", [
    (8, 2, 128, torch.bfloat16), (4, 4, 128, torch.float16), (16, 1, 128, torch.float16),
    (4, 4, 64, torch.bfloat16), (6, 2, 64, torch.float16), (2, 2, 64, torch.float32),
    (2, 2, 256, torch.bfloat16), (3, 3, 32, torch.float16), (2, 1, 80, torch.float32)])
def test_decode_partitions(device, lens, width, H, H_kv, D, dtype):
    kp, vp, tables, cl = make(len(lens) + H, lens, H_kv, D, dtype, 16, width)
    q = torch.randn(len(lens), 1, H, D, generator=torch.Generator().manual_seed(9)).to(dtype)
    slopes = torch.rand(H, generator=torch.Generator().manual_seed(8)) * 0.1
    out = paged_attention(*(x.to(device) for x in (q, kp, vp, tables, cl)), block_size=16,
                          alibi_slopes=slopes.to(device), enable_gqa=H != H_kv)
    rep = lambda x: x.double().repeat_interleave(H // H_kv, dim=2).numpy()
    want = op.paged_attention_decode(q.double().numpy(), rep(kp), rep(vp), tables.numpy(),
                                     cl.numpy(), 1 / np.sqrt(D), 16, slopes.double().numpy())
    got = out.double().cpu().numpy()
    live = np.array(lens) > 0
    assert np.isnan(got[~live]).all()
    # the repository's forward bars: float32 1e-4 relative, 16 bits 2e-2 absolute
    tol = dict(rtol=1e-4, atol=1e-5) if dtype == torch.float32 else dict(rtol=0, atol=2e-2)
    np.testing.assert_allclose(got[live], want[live], **tol)


@pytest.mark.gpu
def test_decode_with_the_smallest_workspace(device):
    # A workspace for 512-token partitions is enough for any call (it then takes
    # those), and the results agree with the finer partitions' up to rounding.
    B, H, H_kv, D, bs, width = 2, 8, 2, 128, 16, 130
    kp, vp, tables, cl = (x.to(device) for x in make(3, [2000, 77], H_kv, D, torch.float16, bs,
                                                       width))
    q = torch.randn(B, 1, H, D, generator=torch.Generator().manual_seed(1)).half().to(device)
    want = paged_attention(q, kp, vp, tables, cl, block_size=bs, enable_gqa=True)
    lib = _native.load()
    parts = -(-bs * width // 512)
    ws = torch.empty(B * H * parts * (D + 2) * 4, dtype=torch.uint8, device=device)
    assert ws.numel() < lib.mpx_paged_decode_workspace_bytes(B, H, D, bs, width)
    out = torch.empty_like(q)
    st = _native._strides((H * D, D))
    call = lambda n: lib.mpx_paged_decode_gqa(
        q.data_ptr(), kp.data_ptr(), vp.data_ptr(), tables.data_ptr(), cl.data_ptr(), None,
        out.data_ptr(), st, st, B, H, H_kv, D, kp.shape[0], bs, width, D ** -0.5,
        _native.dtype_code(q.dtype), ws.data_ptr(), n, _native._stream_ptr(device))
    assert call(ws.numel()) == _native.MPX_OK
    # two roundings to float16 of values below 1
    assert float((out - want).abs().max()) <= 2e-3
    assert call(ws.numel() - 1) == _native.MPX_EINVAL


def test_workspace_bytes_cover_every_head_count():
    # The query names neither the K/V heads nor the dtype: its bytes hold the
    # partials of the smallest partitions any of them takes, never above the
    # no-allocation scratch unless 512-token partitions need more.
    ws = _native.load().mpx_paged_decode_workspace_bytes
    scratch = 32 << 20
    for B in (1, 3, 64):
        for H in (1, 8, 64):
            for D in (32, 64, 128, 256):
                for pages in (1, 100, 2048):
                    base = B * H * -(-pages * 16 // 512) * (D + 2) * 4
                    got = ws(B, H, D, 16, pages)
                    assert base <= got <= max(base, scratch), (B, H, D, pages)
    assert ws(1, 32, 128, 16, 130) == 32 * 33 * 130 * 4       # 33 partitions of 64
    assert ws(64, 32, 128, 16, 512) == 64 * 32 * 16 * 130 * 4  # 16 of 512
