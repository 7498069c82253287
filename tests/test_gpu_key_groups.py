"""GPU parity of the forward launches that cut a workgroup's waves into key
groups (q-tiles of 128 or 64 rows, every wave a part of each key tile, results
merged in LDS): sizes around the row groups, the key parts and the tiles, with
rows whose keys all lie in one group, against the float64 oracle. Bars: 2e-2
absolute, the repository's 16-bit forward bar."""

import math

import numpy as np
import pytest
import torch

from mlx_primitives import _native
from mlx_primitives.attention import flash_attention, sliding_window_attention
from mlx_primitives.cache import paged_attention
from mlx_primitives.kernels import fused_rope_attention, precompute_rope_cache, rope
from oracle import attention as oa
from oracle import paged as op

pytestmark = pytest.mark.gpu


def rnd(shape, seed, dtype):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(dtype)


def dense(q, k, v, left, right):
    """float64 attention, BSHD, query i seeing keys i - left .. i + right."""
    q, k, v = (x.double().numpy() for x in (q, k, v))
    g = q.shape[2] // k.shape[2]
    k, v = np.repeat(k, g, 2), np.repeat(v, g, 2)
    s = np.einsum("bqhd,bkhd->bhqk", q, k) / math.sqrt(q.shape[-1])
    i, j = np.arange(q.shape[1])[:, None], np.arange(k.shape[1])[None, :]
    keep = np.ones(s.shape[-2:], bool)
    if left is not None:
        keep &= j >= i - left
    if right is not None:
        keep &= j <= i + right
    s = np.where(keep, s, -np.inf)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True) + 1e-6
    return np.einsum("bhqk,bkhd->bqhd", p, v)


SIZES = [  # B, H, H_kv, Sq, Sk
    (1, 2, 2, 1, 1), (1, 2, 1, 1, 2048), (2, 8, 2, 3, 700), (1, 4, 4, 31, 33), (1, 4, 4, 65, 127),
    (1, 8, 8, 64, 129), (1, 16, 16, 257, 257), (1, 4, 2, 300, 300), (2, 16, 16, 512, 512),
    (1, 16, 16, 1000, 1000), (1, 8, 8, 1025, 1025), (2, 8, 8, 130, 1100), (1, 3, 1, 777, 777),
]


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("causal", [True, False])
def test_dense(device, size, dtype, D, causal):
    B, H, H_kv, Sq, Sk = size
    q = rnd((B, Sq, H, D), 1, dtype)
    k, v = rnd((B, Sk, H_kv, D), 2, dtype), rnd((B, Sk, H_kv, D), 3, dtype)
    out = flash_attention(*(x.to(device) for x in (q, k, v)), causal=causal, enable_gqa=H != H_kv)
    want = dense(q, k, v, None, max(0, Sk - Sq) if causal else None)
    np.testing.assert_allclose(out.double().cpu().numpy(), want, rtol=0, atol=2e-2)


# A size for each form that _native.fwd_form names: key groups, whether the keys
# are split, and float32's order of two workgroups per CU.
FORMS = [  # dtype, D, (B, H, H_kv, Sq, Sk), causal, window, (groups, split, balanced)
    *((dt, D, *c) for dt in (torch.bfloat16, torch.float16) for D in (64, 128) for c in (
        ((1, 2, 2, 1, 1), True, None, (2 if D == 64 else 1, False, False)),
        ((1, 4, 4, 3, 300), True, None, (4, False, False)),
        ((1, 2, 1, 1, 2048), True, None, (4, True, False)),
        ((1, 96, 48, 129, 129), True, None, (2, False, False)),
        ((1, 96, 96, 129, 129), False, None, (2, False, False)),
        ((1, 5, 1, 65, 16384), True, None, (2, True, False)),
        ((1, 5, 5, 65, 16384), False, None, (2, True, False)),
        ((1, 96, 96, 129, 129), True, 30, (2, False, False)),
        ((1, 12, 12, 1000, 1000), False, 500, (2, True, False)),
        ((1, 1, 1, 1000, 1000), False, 500, (4, True, False)),
        ((1, 96, 96, 257, 257), True, None, (1, False, False)))),
    *((torch.bfloat16, 128, *c) for c in (
        ((1, 32, 8, 777, 777), True, None, (2, False, False)),
        ((1, 24, 24, 1300, 1300), True, None, (2, False, False)),
        ((1, 24, 24, 129, 4065), True, None, (1, True, False)))),
    *((torch.float32, D, *c) for D in (32, 64) for c in (
        ((1, 8, 8, 33, 97), True, None, (2, False, False)),
        ((1, 2, 1, 1, 2048), False, None, (2, True, False)),
        ((1, 12, 12, 65, 4096), True, None, (1, True, False)),
        ((1, 64, 32, 257, 257), True, None, (2, False, True)),   # 40 q-tiles on each XCD
        ((1, 64, 64, 257, 257), False, None, (1, False, False)))),
]


def form_of(dtype, D, size, causal, W):
    B, H, _, Sq, Sk = size
    if W is not None:
        mask = (causal, W, -1 if causal else W)
    else:
        mask = (False, -1, Sk - Sq) if causal and Sk > Sq else (causal, -1, -1)
    groups, splits, balanced = _native.fwd_form(B, H, Sq, Sk, D, *mask, dtype)
    return groups, splits > 1, balanced


@pytest.mark.parametrize("dtype,D,size,causal,W,form", FORMS)
def test_each_form(device, dtype, D, size, causal, W, form):
    assert form_of(dtype, D, size, causal, W) == form
    B, H, H_kv, Sq, Sk = size
    q = rnd((B, Sq, H, D), 1, dtype)
    k, v = rnd((B, Sk, H_kv, D), 2, dtype), rnd((B, Sk, H_kv, D), 3, dtype)
    qd, kd, vd = (x.to(device) for x in (q, k, v))
    if W is None:
        out = flash_attention(qd, kd, vd, causal=causal, enable_gqa=H != H_kv)
        want = dense(q, k, v, None, max(0, Sk - Sq) if causal else None)
    else:
        out = sliding_window_attention(qd, kd, vd, W, causal=causal)
        want = dense(q, k, v, W, 0 if causal else W)
    rtol, atol = (1e-4, 1e-5) if dtype == torch.float32 else (0, 2e-2)
    np.testing.assert_allclose(out.double().cpu().numpy(), want, rtol=rtol, atol=atol)


@pytest.mark.parametrize("dtype,D,size", [
    (torch.bfloat16, 64, (1, 4, 4, 3, 300)), (torch.float16, 128, (1, 4, 4, 3, 300)),
    (torch.bfloat16, 128, (1, 4, 4, 3, 2048)), (torch.bfloat16, 128, (1, 96, 96, 129, 129)),
    (torch.float32, 64, (1, 4, 4, 3, 300)), (torch.float32, 32, (1, 2, 2, 1, 2048))])
@pytest.mark.parametrize("causal", [True, False])
def test_infinities_and_nan_across_groups(device, dtype, D, size, causal):
    # Keys of some groups of a tile score -inf or NaN, or +inf (a NaN row, inf -
    # inf), as the query's first dimension is negative or positive: the same rows
    # are NaN as in float64, the others agree.
    B, H, _, Sq, Sk = size
    assert form_of(dtype, D, size, causal, None)[0] > 1
    for inf, nan in ((range(32, 64), ()), (range(0, 128), ()), ((5, 70, 127), ()),
                     ((), (100,)), (range(16, 32), (3,))):
        q, k, v = (rnd((B, n, H, D), i, dtype) for i, n in enumerate((Sq, Sk, Sk)))
        q[:, ::2, :, 0] = -q[:, ::2, :, 0].abs() - 1   # even rows: -inf
        k[:, list(inf), :, 0] = math.inf
        k[:, list(nan), 0] = math.nan                  # in the first head
        out = flash_attention(*(x.to(device) for x in (q, k, v)), causal=causal)
        with np.errstate(invalid="ignore"):
            want = dense(q, k, v, None, Sk - Sq if causal else None)
        got = out.double().cpu().numpy()
        # (a row whose every visible key scores -inf: NaN in the closed form, a
        # row without keys, 0, in the kernels)
        blind = np.isnan(want) & (got == 0)
        if blind.any():
            assert Sq == Sk and causal and len(inf) >= 32 and not blind[:, 128:].any()
        assert (np.isnan(got) == np.isnan(want) & ~blind).all()
        rtol, atol = (1e-4, 1e-5) if dtype == torch.float32 else (0, 2e-2)
        seen = ~np.isnan(want)
        np.testing.assert_allclose(got[seen], want[seen], rtol=rtol, atol=atol)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("S,W,causal", [(700, 0, True), (700, 30, True), (1000, 63, False),
                                        (513, 200, True), (300, 299, False)])
def test_window(device, S, W, causal, D):
    q, k, v = (rnd((1, S, 12, D), i, torch.bfloat16) for i in range(3))
    out = sliding_window_attention(*(x.to(device) for x in (q, k, v)), W, causal=causal)
    np.testing.assert_allclose(out.double().cpu().numpy(),
                               dense(q, k, v, W, 0 if causal else W), rtol=0, atol=2e-2)


@pytest.mark.parametrize("D,scale,mult", [(128, -0.2, 1.0), (64, 0.125, 3.0), (128, 0.001, 1.0)])
def test_scales(device, D, scale, mult):
    # Negative, larger and near-zero scores. The kernels round Q times the scale
    # to bfloat16, an error of 2^-9 / sqrt(3) of a score's spread, which is at
    # most 3 here: 3.4e-3 of a weight, well inside the bar. (A spread of 80, D =
    # 64 at scale 1 and inputs times 10, moves weights by a third with any tile.)
    q, k, v = (rnd((1, 400, 8, D), i + 5, torch.bfloat16) for i in range(3))
    q = q * mult
    out = flash_attention(*(x.to(device) for x in (q, k, v)), scale=scale, causal=True)
    want = oa.flash_attention(*(x.double().numpy() for x in (q, k, v)), scale=scale, causal=True)
    np.testing.assert_allclose(out.double().cpu().numpy(), want, rtol=0, atol=2e-2)


def test_one_group_dominates(device):
    # All the weight on one key, in each 32-key part of the tile in turn: the
    # merge rescales the other groups' sums to nothing.
    S, D = 512, 128
    for at in (0, 33, 70, 127, 128, 255, 511):
        k = torch.zeros(1, S, 4, D)
        k[:, at] = 30.0
        q = torch.ones(1, S, 4, D)
        v = rnd((1, S, 4, D), at, torch.float16)
        out = flash_attention(*(x.half().to(device) for x in (q, k, v)), causal=False)
        want = v[:, at:at + 1].expand(1, S, 4, D)
        assert float((out.cpu().float() - want.float()).abs().max()) <= 2e-3, at


@pytest.mark.parametrize("bs", [16, 24, 64])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("alibi", [False, True])
def test_paged_prefill_missing_pages(device, D, bs, alibi):
    B, Sq, H, H_kv = 3, 400, 8, 4
    lens = [400, 333, 0]
    pages = -(-Sq // bs) + 1
    g = torch.Generator().manual_seed(bs)
    tables = torch.randperm(B * pages, generator=g).to(torch.int32).reshape(B, pages)
    tables[0, 1] = -1             # one page of the first tile
    tables[1, 128 // bs] = B * pages + 7  # an id past the pool in the second tile
    q = rnd((B, Sq, H, D), 1, torch.float16)
    kp, vp = (rnd((B * pages, bs, H_kv, D), s, torch.float16) for s in (2, 3))
    cl = torch.tensor(lens, dtype=torch.int32)
    slopes = torch.rand(H, generator=g) * 0.1 if alibi else None
    out = paged_attention(*(x.to(device) for x in (q, kp, vp, tables, cl)), block_size=bs,
                          alibi_slopes=None if slopes is None else slopes.to(device),
                          enable_gqa=True)
    tb = tables.clone()
    tb[tb >= B * pages] = -1
    rep = lambda x: x.double().repeat_interleave(H // H_kv, dim=2).numpy()
    want = op.paged_attention_prefill(q.double().numpy(), rep(kp), rep(vp), tb.numpy(), cl.numpy(),
                                      1 / math.sqrt(D), bs, True,
                                      None if slopes is None else slopes.double().numpy())
    got = out.double().cpu().numpy()
    assert (np.isnan(got) == np.isnan(want)).all() and np.isnan(got[2]).all()
    np.testing.assert_allclose(got[:2], want[:2], rtol=0, atol=2e-2)


@pytest.mark.parametrize("D,H,S,bs,form", [
    (128, 2, 1, 16, (1, False)), (128, 1, 257, 16, (4, False)), (128, 1, 1000, 16, (4, True)),
    (128, 12, 1000, 16, (2, True)), (128, 1, 129, 24, (2, False)), (128, 1, 512, 24, (2, True)),
    (64, 1, 129, 16, (2, False)), (64, 1, 512, 16, (2, True)), (64, 48, 512, 16, (1, True))])
def test_each_paged_form(device, D, H, S, bs, form):
    pages = -(-S // bs)
    got = _native.fwd_form(1, H, max(S, 2), pages * bs, D, True, -1, -1, torch.bfloat16, bs)
    assert (got[0], got[1] > 1) == form
    Sq = max(S, 2)   # (one query is a decode)
    tables = torch.randperm(pages, generator=torch.Generator().manual_seed(1)).to(torch.int32)[None]
    q = rnd((1, Sq, H, D), 1, torch.bfloat16)
    kp, vp = (rnd((pages, bs, H, D), s, torch.bfloat16) for s in (2, 3))
    cl = torch.tensor([S], dtype=torch.int32)
    out = paged_attention(*(x.to(device) for x in (q, kp, vp, tables, cl)), block_size=bs)
    want = op.paged_attention_prefill(*(x.double().numpy() for x in (q, kp, vp)), tables.numpy(),
                                      cl.numpy(), 1 / math.sqrt(D), bs, True, None)
    np.testing.assert_allclose(out.double().cpu().numpy(), want, rtol=0, atol=2e-2)


@pytest.mark.parametrize("D", [64, 128])
def test_rope_on_load_equals_rope_first(device, D):
    # Q rotated by every key group: bit-identical to rotating it first.
    q, k, v = (rnd((1, 300, 8, D), i, torch.bfloat16).to(device) for i in range(3))
    cos, sin = precompute_rope_cache(400, D, dtype=torch.bfloat16, device=device)
    out = fused_rope_attention(q, k, v, cos_cache=cos, sin_cache=sin, q_offset=40, kv_offset=40,
                               causal=True)
    want = flash_attention(rope(q, cos, sin, 40), rope(k, cos, sin, 40), v, causal=True)
    assert torch.equal(out, want)


@pytest.mark.parametrize("cache", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,Sq,Sk,q_off,kv_off,causal,groups", [
    (1, 4, 1, 700, 699, 0, True, 4), (2, 32, 65, 4065, 4000, 0, True, 2),
    (1, 8, 100, 129, 40, 40, False, 2), (1, 3, 33, 400, 369, 2, True, 4),
    (1, 4, 1, 257, 263, 7, True, 4), (1, 16, 200, 200, 0, 0, True, 2),
    (1, 96, 129, 129, 5, 5, True, 2)])
def test_k_rotated_in_the_kernel_equals_rope_first(device, B, H, Sq, Sk, q_off, kv_off, causal,
                                                   groups, cache):
    # The same bits as rotating Q and K first: tiles past the last key, offsets
    # on either side, splits of the keys, 2 and 4 key groups.
    D, dtype = 128, torch.bfloat16
    q = rnd((B, Sq, H, D), 1, dtype).to(device)
    k, v = (rnd((B, Sk, H, D), s, dtype).to(device) for s in (2, 3))
    # (the tables end at the last key or query)
    cos, sin = precompute_rope_cache(max(Sq + q_off, Sk + kv_off), D, dtype=cache, device=device)
    wr = q_off - kv_off if causal else -1
    mask = (False, -1, wr) if wr else (True, -1, -1)
    assert _native.rope_qk_preferred(B, H, Sq, Sk, D, *mask, dtype, cache)
    assert _native.fwd_form(B, H, Sq, Sk, D, *mask, dtype)[0] == groups
    out = fused_rope_attention(q, k, v, cos_cache=cos, sin_cache=sin, q_offset=q_off,
                               kv_offset=kv_off, causal=causal)
    o = torch.empty_like(q)
    qr, kr = rope(q, cos, sin, q_off), rope(k, cos, sin, kv_off)
    bhs = lambda x: (x.stride(0), x.stride(2), x.stride(1))
    _native.attn_fwd(qr, kr, v, o, bhs(q), bhs(k), bhs(v), bhs(o), B, H, Sq, Sk, D, D ** -0.5,
                     *mask)
    assert torch.equal(out, o)


@pytest.mark.parametrize("offset", [40.0, np.float32(40), np.int64(40), torch.tensor(40)])
def test_offsets_as_int_reads_them(device, offset):
    # Where K is rotated in the kernel (Sq = 3) and where it is not (Sq = 700).
    cos, sin = precompute_rope_cache(800, 128, dtype=torch.bfloat16, device=device)
    k, v = (rnd((1, 700, 4, 128), s, torch.bfloat16).to(device) for s in (2, 3))
    for Sq in (3, 700):
        q = rnd((1, Sq, 4, 128), 1, torch.bfloat16).to(device)
        a, b = (fused_rope_attention(q, k, v, cos_cache=cos, sin_cache=sin, q_offset=o,
                                     kv_offset=0, causal=True) for o in (offset, 40))
        assert torch.equal(a, b)


def test_k_rotation_left_to_its_own_pass():
    # full launches, float32 tables, other inputs and head dims
    pref = _native.rope_qk_preferred
    b, f = torch.bfloat16, torch.float32
    assert not pref(2, 32, 65, 4065, 128, False, -1, 4000, torch.float16, b)
    assert not pref(4, 32, 4096, 4096, 128, True, -1, -1, b, b)
    assert not pref(2, 32, 65, 4065, 128, False, -1, 4000, b, f)
    assert not pref(2, 32, 65, 4065, 64, False, -1, 4000, b, b)
    assert not pref(2, 32, 65, 4065, 128, False, -1, 4000, f, b)


@pytest.mark.parametrize("S,H", [(300, 8), (1000, 16), (777, 12), (129, 96)])
def test_lse_of_key_groups(device, S, H):
    # The saved log-sum-exp (base 2) does not depend on the groups: lse against
    # float64.
    D = 128
    q, k, v = (rnd((1, S, H, D), i, torch.float16).to(device) for i in range(3))
    o, lse = torch.empty_like(q), torch.empty(1, H, S, device=device)
    bhs = lambda x: (x.stride(0), x.stride(2), x.stride(1))
    _native.attn_fwd(q, k, v, o, bhs(q), bhs(k), bhs(v), bhs(o), 1, H, S, S, D, D ** -0.5, True,
                     lse=lse)
    s = torch.einsum("bqhd,bkhd->bhqk", q.double().cpu(), k.double().cpu()) * D ** -0.5
    s.masked_fill_(~torch.ones(S, S, dtype=torch.bool).tril(), -math.inf)
    want = torch.logsumexp(s, -1) / math.log(2)
    # scores of products of float16: Q times the scale is rounded to float16 (2^-11 of ~5)
    assert float((lse.double().cpu() - want).abs().max()) <= 1e-2


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("B,H,H_kv,Sq,Sk,causal,W", [
    (1, 8, 8, 1, 300, False, None), (1, 8, 8, 33, 97, True, None), (1, 8, 2, 300, 300, True, None),
    (1, 8, 8, 700, 700, True, 100), (2, 16, 16, 300, 300, True, None),  # 10 tiles per XCD
    (1, 16, 16, 1300, 1300, True, None),
    (2, 12, 12, 1024, 1024, True, None),   # 48, the training case
    (1, 3, 1, 500, 500, False, None)])
def test_float32_key_groups(device, B, H, H_kv, Sq, Sk, causal, W, D):
    q = rnd((B, Sq, H, D), 1, torch.float32)
    k, v = rnd((B, Sk, H_kv, D), 2, torch.float32), rnd((B, Sk, H_kv, D), 3, torch.float32)
    qd, kd, vd = (x.to(device) for x in (q, k, v))
    if W is None:
        out = flash_attention(qd, kd, vd, causal=causal, enable_gqa=H != H_kv)
    else:
        out = sliding_window_attention(qd, kd, vd, W, causal=causal)
    want = dense(q, k, v, W, max(0, Sk - Sq) if causal else None)
    # the repository's float32 forward bar
    np.testing.assert_allclose(out.double().cpu().numpy(), want, rtol=1e-4, atol=1e-5)
