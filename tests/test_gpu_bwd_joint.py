"""GPU parity of the joint backward launch (dQ and dK/dV tiles in one grid) and
of the grouped backward that cuts a K/V head's query heads into parts, at the
sizes where their launch rules and tile orders change: gradients against a
float64 evaluation of the closed form, itself pinned to the oracle on the CPU.

Tolerance: normwise ||g - ref|| / ||ref||, 2e-3 (float16), 1.5e-2 (bfloat16)
and 2e-5 (float32), the bars of test_gpu_attention_bwd.py (a few units of the
rounding of P, dS and the result to dtype; float32 sums).
"""

import math

import numpy as np
import pytest
import torch

from mlx_primitives import _native
from mlx_primitives.attention import _launch, flash_attention, sliding_window_attention
from mlx_primitives.constants import Layout
from oracle import attention_grad as oag
from oracle import dropout as od

NREL = {torch.float16: 2e-3, torch.bfloat16: 1.5e-2, torch.float32: 2e-5}


def rnd(shape, seed, dtype):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(shape, generator=g).to(dtype)


def grads64(q, k, v, dout, scale, left, right):
    """dq, dk, dv (BSHD, float64) with query i seeing keys i - left .. i + right
    (None: no limit); every query sees a key."""
    B, Sq, H, D = q.shape
    Sk, Hk = k.shape[1], k.shape[2]
    out = [torch.zeros(x.shape, dtype=torch.float64, device=q.device) for x in (q, k, v)]
    i = torch.arange(Sq, device=q.device)[:, None]
    j = torch.arange(Sk, device=q.device)[None, :]
    for b in range(B):
        for h in range(H):
            q1, k1, v1, d1 = (x.double().contiguous() for x in (
                q[b, :, h], k[b, :, h // (H // Hk)], v[b, :, h // (H // Hk)], dout[b, :, h]))
            s = (q1 @ k1.t()) * scale
            if left is not None:
                s.masked_fill_(j < i - left, -math.inf)
            if right is not None:
                s.masked_fill_(j > i + right, -math.inf)
            p = torch.exp(s - s.amax(1, keepdim=True))
            p = p / (p.sum(1, keepdim=True) + 1e-6)
            ds = p * (d1 @ v1.t() - (d1 * (p @ v1)).sum(1, keepdim=True)) * scale
            out[0][b, :, h] = ds @ k1
            out[1][b, :, h // (H // Hk)] += ds.t() @ q1
            out[2][b, :, h // (H // Hk)] += p.t() @ d1
    return out


@pytest.mark.parametrize("left,right", [(None, 0), (None, None), (5, 0), (None, 20)])
def test_reference_matches_oracle(left, right):
    q, d = rnd((2, 20, 4, 8), 0, torch.float32), rnd((2, 20, 4, 8), 1, torch.float32)
    k, v = rnd((2, 40, 2, 8), 2, torch.float32), rnd((2, 40, 2, 8), 3, torch.float32)
    want = oag.attention_grad(*(x.double().numpy() for x in (q, k, v, d)), 0.3, False,
                              -1 if left is None else left, -1 if right is None else right)
    for g, w in zip(grads64(q, k, v, d, 0.3, left, right), want):
        np.testing.assert_allclose(g.numpy(), w, rtol=1e-9, atol=1e-11)


def run(device, q, k, v, d, causal=True, window=None, dropout=0.0):
    q, k, v = (x.to(device).requires_grad_(True) for x in (q, k, v))
    if window is None:
        out = flash_attention(q, k, v, causal=causal, dropout_p=dropout,
                              enable_gqa=q.shape[2] != k.shape[2])
    else:
        out = sliding_window_attention(q, k, v, window, causal=causal)
    return torch.autograd.grad(out, (q, k, v), d.to(device))


CASES = [
    # B, H, H_kv, Sq, Sk, D, causal, window
    (1, 1, 1, 1, 1, 128, True, None),
    (1, 1, 1, 2, 128, 64, False, None),
    (1, 8, 8, 129, 257, 128, False, None),       # 8 heads: one per XCD
    (1, 3, 3, 257, 129, 128, True, None),        # queries past the last key tile
    (1, 8, 1, 130, 70, 128, True, None),         # 8 parts of one head
    (2, 16, 4, 300, 300, 128, True, None),       # 4 parts
    (1, 12, 4, 200, 333, 64, False, None),       # group of 3
    (3, 6, 6, 260, 260, 64, True, 75),           # window, heads not a multiple of 8
    (1, 8, 8, 400, 400, 128, False, 60),
    (1, 1, 1, 128, 16256, 128, False, None),     # 1 + 127 tiles: the longest order
    (1, 1, 1, 128, 16257, 128, False, None),     # 1 + 128: two launches
    (1, 1, 1, 16129, 100, 64, True, None),       # 127 + 1
    (4, 8, 8, 4096, 4096, 64, True, None),       # chunks of 16 heads per XCD
    (2, 16, 16, 4096, 200, 128, False, None),    # 32 x 34 tiles: joint
    (1, 32, 4, 4096, 4096, 128, True, None),     # 2048 tiles: paired, 4 parts
    (1, 31, 31, 4100, 4100, 128, True, None),    # 2046 tiles: joint
    (1, 20, 4, 2048, 16384, 128, True, None),    # 5 heads in 4 parts: paired tiles
    (1, 33, 3, 1300, 16384, 64, False, None),    # 11 in 10, two launches at D = 64
    (1, 4, 2, 1300, 16384, 64, True, None),      # 2 parts of one head, two launches
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES)
def test_joint_backward(device, dtype, case):
    B, H, H_kv, Sq, Sk, D, causal, W = case
    q, d = rnd((B, Sq, H, D), Sq, dtype), rnd((B, Sq, H, D), Sq + 1, dtype)
    k, v = rnd((B, Sk, H_kv, D), Sk + 2, dtype), rnd((B, Sk, H_kv, D), Sk + 3, dtype)
    got = run(device, q, k, v, d, causal, W)
    left = W
    right = (0 if causal else W) if W is not None else (max(0, Sk - Sq) if causal else None)
    want = grads64(*(x.to(device) for x in (q, k, v, d)), 1 / math.sqrt(D), left, right)
    for name, g, w in zip(("dq", "dk", "dv"), got, want):
        assert torch.isfinite(g).all(), name
        err = float((g.double() - w).norm())
        # (one visible key: dq and dk vanish, rounding noise is left)
        assert err <= NREL[dtype] * float(w.norm()) + 1e-2 * (Sk == 1), (name, err)


CASES32 = [  # float32: tiles of 64 rows, two key groups of 32
    (1, 1, 1, 1, 1, 64, True, None),
    (1, 3, 3, 31, 33, 64, False, None),
    (1, 8, 8, 65, 97, 128, False, None),
    (2, 4, 4, 97, 65, 64, True, None),
    (1, 8, 2, 130, 200, 128, False, None),       # 4 parts
    (1, 6, 2, 257, 257, 64, True, None),         # group of 3
    (1, 5, 5, 300, 300, 128, True, 40),
    (2, 3, 3, 300, 300, 64, False, 33),
    (1, 1, 1, 64, 8128, 64, False, None),        # 1 + 127 tiles: the longest order
    (1, 1, 1, 64, 8129, 64, False, None),
    (1, 1, 1, 128, 4032, 128, False, None),      # 2 + 2 x 63 tiles
    (1, 4, 1, 64, 6000, 128, False, None),       # too many for an order: parts alone
    (1, 31, 31, 2112, 2112, 64, True, None),     # 2046 tiles: joint
    (1, 32, 8, 2048, 2048, 64, True, None),      # 2048: launches of their own, 4 parts
    (1, 74, 2, 64, 8256, 64, False, None),       # 37 heads in 31 parts, own launches
    (1, 34, 2, 64, 8256, 128, True, None),       # 17 in 15
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES32)
def test_joint_backward_float32(device, case):
    test_joint_backward(device, torch.float32, case)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,D,stored", [
    (torch.bfloat16, 64, None), (torch.float16, 128, False), (torch.bfloat16, 128, None),
    (torch.float32, 64, None), (torch.float32, 128, None)])
@pytest.mark.parametrize("long,p,causal,wl,H_kv", [
    ("keys", 0.0, False, 300, 4), ("keys", 0.3, True, -1, 4), ("keys", 0.3, False, 300, 2),
    ("queries", 0.0, True, -1, 4), ("queries", 0.3, False, -1, 2), ("queries", 0.3, False, 300, 4)])
def test_launches_of_their_own(device, monkeypatch, dtype, D, stored, p, causal, wl, H_kv, long):
    # A side of 129 tiles is no joint launch at any size: the dQ and dK/dV
    # launches (paired at D = 128, an odd count), with the masks and the keep
    # mask; without groups and with them (parts on the side of the keys). At D =
    # 128 the dropout backward stores dS by default; False recomputes.
    monkeypatch.setattr(_launch, "BWD_STORED_DS", stored)
    n = 16400 if dtype != torch.float32 else 8200
    Sq, Sk = (70, n) if long == "keys" else (n, 200)
    H, seed = 4, 0xABCDEF0123456789
    q, d = rnd((1, Sq, H, D), 1, dtype), rnd((1, Sq, H, D), 2, dtype)
    k, v = rnd((1, Sk, H_kv, D), 3, dtype), rnd((1, Sk, H_kv, D), 4, dtype)
    a = [x.to(device).requires_grad_(True) for x in (q, k, v)]
    out = _launch.run_attention(*a, Layout.BSHD, 1 / math.sqrt(D), causal, wl, -1, dropout_p=p,
                                dropout_seed_value=seed)
    got = torch.autograd.grad(out, a, d.to(device))
    want = od.attention_dropout_grad(*(x.double().numpy() for x in (q, k, v, d)), 1 / math.sqrt(D),
                                     causal, p, seed, wl, keep=None if p else np.ones((1, 1, 1, 1)))
    for name, g, w in zip(("dq", "dk", "dv"), got, want):
        err = np.linalg.norm(g.double().cpu().numpy() - w)
        assert err <= NREL[dtype] * np.linalg.norm(w), (name, err)


@pytest.mark.gpu
@pytest.mark.parametrize("H,H_kv,S", [(4, 4, 300), (8, 2, 257), (16, 16, 2000)])
def test_joint_dropout_agrees_with_stored_schedule(device, monkeypatch, H, H_kv, S):
    # Same keep mask from the same seed; the schedules differ in summation order
    # and rounding of the same 16-bit P and dS.
    q, d = rnd((1, S, H, 128), 1, torch.bfloat16), rnd((1, S, H, 128), 2, torch.bfloat16)
    k, v = rnd((1, S, H_kv, 128), 3, torch.bfloat16), rnd((1, S, H_kv, 128), 4, torch.bfloat16)
    got = {}
    for stored in (True, None):
        monkeypatch.setattr(_launch, "BWD_STORED_DS", stored)
        torch.manual_seed(5)
        got[stored] = run(device, q, k, v, d, dropout=0.2)
    for name, a, b in zip(("dq", "dk", "dv"), got[True], got[None]):
        rel = float((a.double() - b.double()).norm() / a.double().norm())
        assert rel <= 4e-3, (name, rel)


@pytest.mark.gpu
def test_uneven_parts_with_dropout(device, monkeypatch):
    # The keep mask of every head where one part holds a head more than the
    # others, against the stored-dS schedule, which has no parts.
    H, H_kv, Sq, Sk = 20, 4, 2048, 16384
    q, d = rnd((1, Sq, H, 128), 1, torch.bfloat16), rnd((1, Sq, H, 128), 2, torch.bfloat16)
    k, v = rnd((1, Sk, H_kv, 128), 3, torch.bfloat16), rnd((1, Sk, H_kv, 128), 4, torch.bfloat16)
    got = {}
    for stored in (True, None):
        monkeypatch.setattr(_launch, "BWD_STORED_DS", stored)
        torch.manual_seed(5)
        got[stored] = run(device, q, k, v, d, causal=False, dropout=0.2)
    for name, a, b in zip(("dq", "dk", "dv"), got[True], got[None]):
        rel = float((a.double() - b.double()).norm() / a.double().norm())
        assert rel <= 4e-3, (name, rel)


@pytest.mark.gpu
def test_grouped_backward_without_room_for_parts(device):
    # A workspace for Dvec alone: each group is one part, the same gradients up
    # to summation order.
    B, H, H_kv, S, D = 1, 8, 2, 300, 128
    q, d = rnd((B, S, H, D), 1, torch.float16).to(device), rnd((B, S, H, D), 2, torch.float16).to(device)
    k, v = (rnd((B, S, H_kv, D), s, torch.float16).to(device) for s in (3, 4))
    lib = _native.load()
    want = run(device, q, k, v, d)
    o, lse = torch.empty_like(q), torch.empty(B, H, S, device=device)
    bhs = lambda x: (x.stride(0), x.stride(2), x.stride(1))
    _native.attn_fwd(q, k, v, o, bhs(q), bhs(k), bhs(v), bhs(o), B, H, S, S, D, D ** -0.5, True,
                     H_kv=H_kv, lse=lse)
    got = [torch.empty_like(x) for x in (q, k, v)]
    ws = torch.empty(lib.mpx_attn_bwd_workspace_bytes(B, H, S), dtype=torch.uint8, device=device)
    rc = lib.mpx_attn_bwd_grouped(
        *(x.data_ptr() for x in (q, k, v, o, d, lse, *got)),
        *(_native._strides(bhs(x)) for x in (q, k, v, o, d, *got)), B, H, H_kv, S, S, D,
        D ** -0.5, 1, -1, -1, _native.dtype_code(q.dtype), 0.0, 0, ws.data_ptr(), ws.numel(),
        _native._stream_ptr(device))
    assert rc == _native.MPX_OK
    for a, b in zip(got, want):
        assert float((a.double() - b.double()).norm() / b.double().norm()) <= 1e-3


@pytest.mark.gpu
@pytest.mark.parametrize("H_kv", [8, 2, 1])
@pytest.mark.parametrize("Sq,Sk,stored", [(64, 16384, True), (64, 1000, False)])
def test_dropout_entry_stores_ds_in_large_launches(device, H_kv, Sq, Sk, stored):
    # mpx_attn_bwd_dropout with the stored-dS workspace, with and without groups:
    # the bits of mpx_attn_bwd_stored and its dS blocks where the launch is not a
    # joint one, else nothing but Dvec written.
    B, H, D = 1, 8, 128
    q, d = (rnd((B, Sq, H, D), s, torch.bfloat16).to(device) for s in (1, 2))
    k, v = (rnd((B, Sk, H_kv, D), s, torch.bfloat16).to(device) for s in (3, 4))
    lib = _native.load()
    o, lse = torch.empty_like(q), torch.empty(B, H, Sq, device=device)
    bhs = lambda x: (x.stride(0), x.stride(2), x.stride(1))
    _native.attn_fwd(q, k, v, o, bhs(q), bhs(k), bhs(v), bhs(o), B, H, Sq, Sk, D, D ** -0.5, False,
                     H_kv=H_kv, lse=lse, dropout=(0.2, 7))
    nbytes = lib.mpx_attn_bwd_ds_workspace_bytes(B, H, Sq, Sk, D, 2, 0, -1, -1)
    outs, left = {}, {}
    for entry in ("mpx_attn_bwd_dropout", "mpx_attn_bwd_stored"):
        got = [torch.empty_like(x) for x in (q, k, v)]
        ws = torch.full((nbytes,), 0xA5, dtype=torch.uint8, device=device)
        rc = getattr(lib, entry)(
            *(x.data_ptr() for x in (q, k, v, o, d, lse, *got)),
            *(_native._strides(bhs(x)) for x in (q, k, v, o, d, *got)), B, H, H_kv, Sq, Sk, D,
            D ** -0.5, 0, -1, -1, 2, 0.2, 7, ws.data_ptr(), ws.numel(),
            _native._stream_ptr(device))
        assert rc == _native.MPX_OK
        outs[entry] = got
        left[entry] = int((ws[lib.mpx_attn_bwd_workspace_bytes(B, H, Sq):] == 0xA5).sum())
    a, b = outs.values()
    if stored:
        assert all(torch.equal(x, y) for x, y in zip(a, b))
        assert left["mpx_attn_bwd_dropout"] == left["mpx_attn_bwd_stored"] < nbytes // 2
    else:
        assert left["mpx_attn_bwd_stored"] < nbytes // 2 < left["mpx_attn_bwd_dropout"]
        for x, y in zip(a, b):
            assert float((x.double() - y.double()).norm() / y.double().norm()) <= 4e-3


def test_grouped_workspace_bytes():
    lib = _native.load()
    ws = lib.mpx_attn_bwd_grouped_workspace_bytes
    plain = lib.mpx_attn_bwd_workspace_bytes(1, 8, 300)
    assert ws(1, 8, 8, 300, 300, 128, 2, -1) == plain       # no groups
    assert ws(1, 8, 2, 300, 300, 256, 2, -1) == plain       # no parts at head dim 256
    # float32: tiles of 64 keys, parts up to 256 workgroups
    assert ws(1, 8, 2, 300, 300, 128, 0, -1) == -(-plain // 256) * 256 + 2 * 8 * 300 * 128 * 4
    assert ws(8, 8, 4, 512, 512, 64, 0, -1) == lib.mpx_attn_bwd_workspace_bytes(8, 8, 512)
    # 4 parts of 2 K/V heads, dK and dV sums in float32
    assert ws(1, 8, 2, 300, 300, 128, 2, -1) == -(-plain // 256) * 256 + 2 * 8 * 300 * 128 * 4
    assert ws(1, 8, 3, 300, 300, 128, 2, -1) == 0
    # parts stop at one workgroup per slot of the chip
    assert ws(4, 32, 8, 4096, 4096, 128, 2, -1) == lib.mpx_attn_bwd_workspace_bytes(4, 32, 4096)


@pytest.mark.parametrize("group", [2, 3, 4, 5, 6, 7, 8, 11, 12, 28, 31, 64, 71])
def test_grouped_workspace_is_bounded(group):
    # also where the group has no divisor near the count that fills the chip
    lib = _native.load()
    most = 0
    for B in (1, 2, 3, 4, 7, 8, 15, 16):
        for H_kv in (1, 2, 4, 8):
            for S in (64, 300, 1024, 2048, 4000, 4096, 4608, 8192, 16384, 32768, 65000):
                for D in (64, 128):
                    for dtype in (0, 2):
                        need = lib.mpx_attn_bwd_grouped_workspace_bytes(
                            B, H_kv * group, H_kv, S, S, D, dtype, -1)
                        plain = lib.mpx_attn_bwd_workspace_bytes(B, H_kv * group, S)
                        most = max(most, need - -(-plain // 256) * 256)
    assert most <= 256 << 20


@pytest.mark.parametrize("B,H,H_kv,Sq,Sk,D,dtype,parts", [
    # the parts that the cases above mean
    (1, 20, 4, 2048, 16384, 128, 2, 4), (1, 33, 3, 1300, 16384, 64, 2, 10),
    (1, 4, 2, 1300, 16384, 64, 2, 2), (1, 74, 2, 64, 8256, 64, 0, 31),
    (1, 34, 2, 64, 8256, 128, 0, 15), (1, 8, 1, 130, 70, 128, 2, 8), (1, 12, 4, 200, 333, 64, 2, 3),
    (1, 32, 4, 4096, 4096, 128, 2, 8), (1, 32, 8, 2048, 2048, 64, 0, 4),
    # short queries, where parts cost more than the chains they cut
    # (forward and backward whole and in all parts: 203 / 539 us, 35 / 63, 36 / 45)
    (4, 216, 27, 18, 847, 128, 2, 1), (2, 100, 20, 32, 783, 64, 2, 1), (8, 54, 18, 4, 56, 128, 2, 1),
    # full launches (152 / 203 and 404 / 514)
    (6, 108, 27, 378, 378, 64, 2, 1), (4, 84, 21, 781, 781, 128, 2, 1)])
def test_parts_of_a_group(B, H, H_kv, Sq, Sk, D, dtype, parts):
    lib = _native.load()
    plain = -(-lib.mpx_attn_bwd_workspace_bytes(B, H, Sq) // 256) * 256
    got = lib.mpx_attn_bwd_grouped_workspace_bytes(B, H, H_kv, Sq, Sk, D, dtype, -1)
    assert max(0, got - plain) == (2 * B * H_kv * parts * Sk * D * 4 if parts > 1 else 0)
