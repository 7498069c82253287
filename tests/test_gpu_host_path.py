"""The native host path (_mpx_host) against the general Python path: the same
calls with the extension answering None give the same bits, over the layouts
that it takes and those that it leaves."""

import struct

import numpy as np
import pytest
import torch

from mlx_primitives import _native
from mlx_primitives.attention import flash_attention, sliding_window_attention
from mlx_primitives.cache import get_alibi_slopes, paged_attention, store_kv
from mlx_primitives.cache.kv_store import _i32
from mlx_primitives.kernels import precompute_rope_cache, rope_at


class _Sub(torch.Tensor):
    pass


class _Off:
    """A host extension that leaves every call to the general path."""

    def __getattr__(self, name):
        return lambda *args: None


def both(monkeypatch, fn):
    _native.load()
    native = fn()
    with monkeypatch.context() as m:
        m.setattr(_native, "_host", _Off())
        general = fn()
    for a, b in zip(native, general):
        assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride()
        assert torch.equal(a.nan_to_num(), b.nan_to_num())
    return native


def counted(monkeypatch):
    """How often the extension answered itself: name -> [taken, left]."""
    seen, real = {}, _native.host()

    class Spy:
        def __getattr__(self, name):
            def f(*args):
                r = getattr(real, name)(*args)
                seen.setdefault(name, [0, 0])[r is None] += 1
                return r
            return f
    monkeypatch.setattr(_native, "_host", Spy())
    return seen


def rnd(*shape, dtype=torch.bfloat16, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return torch.randn(shape, generator=g).to(dtype)


def test_entries_are_the_librarys():
    lib = _native.load()
    names = _native.host().entries()
    assert len(names) == len(set(names)) and all(hasattr(lib, n) for n in names)
    # host tensors, other objects and wrong counts
    t = torch.zeros(1, 2, 3, 64)
    assert _native.host().rope_at(t, t, t, t, t, 0) is None
    assert _native.host().rope_at(None, 1, "x", t, t, 0) is None
    with pytest.raises(TypeError):
        _native.host().attn_fwd(t, t)
    with pytest.raises(KeyError):
        _native.host().init({})
    assert _native._load_host(lib) is not None  # (binds the entries again)


def test_extension_has_no_thread_local_storage():
    # (a segment of type PT_TLS slows every thread-local access of the process)
    data = open(_native._HOST_PATH, "rb").read()
    assert data[:5] == b"\x7fELF\x02"
    off, size, count = struct.unpack_from("<Q", data, 32)[0], *struct.unpack_from("<HH", data, 54)
    assert 7 not in [struct.unpack_from("<I", data, off + i * size)[0] for i in range(count)]


@pytest.mark.parametrize("content", [None, b"", b"\x7fELF of another torch"])
def test_package_loads_without_the_extension(monkeypatch, tmp_path, content):
    # missing, empty or unreadable: a warning, and every call left to the Python path
    path = tmp_path / "_mpx_host.so"
    if content is not None:
        path.write_bytes(content)
    monkeypatch.setattr(_native, "_HOST_PATH", str(path))
    monkeypatch.setattr(_native, "_lib", None)
    monkeypatch.setattr(_native, "_host", None)
    with pytest.warns(RuntimeWarning, match="Python path"):
        assert _native.load().mpx_version() > 0
    assert _native.host().rope_at(None, None, None, None, None, 0) is None


@pytest.mark.parametrize("x", [2**31 - 1, -2**31, 2**31, 2**63, -2**31 - 1, True])
@pytest.mark.parametrize("n", [0, 1, 3])
def test_int_positions_are_refused_as_as_tensor_does(x, n):
    def general():
        t = torch.as_tensor(x, dtype=torch.int32).reshape(-1)
        t = t.expand(n) if n > 1 else t
        if t.numel() != n:
            raise ValueError
        return t
    try:
        want = general()
    except Exception as e:
        with pytest.raises(type(e)):
            _i32(x, "cpu", n, "x")
    else:
        got = _i32(x, "cpu", n, "x")
        assert got.dtype == torch.int32 and got.tolist() == want.tolist()


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["plain", "heads_first_view", "offset", "parameter", "subclass",
                                  "last_strided"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("D", [64, 80, 128])
def test_forward_and_gradients(device, monkeypatch, form, dtype, D):
    def make(seed, H=4):
        x = rnd(2, 70, H, D, dtype=dtype, seed=seed).to(device)
        if form == "heads_first_view":
            x = x.transpose(1, 2).contiguous().transpose(1, 2)
        elif form == "offset":      # 2 or 4 bytes past an aligned address
            x = torch.cat([x.new_zeros(1), x.reshape(-1)])[1:].reshape(x.shape)
        elif form == "last_strided":
            x = x.transpose(2, 3).contiguous().transpose(2, 3)
        elif form == "parameter":
            x = torch.nn.Parameter(x)
        elif form == "subclass":
            x = x.as_subclass(_Sub)
        return x
    q, k, v, d = make(1), make(2, 2), make(3, 2), make(4).detach()

    def fn():
        a, b, c = (x.detach().requires_grad_(True) for x in (q, k, v))
        out = flash_attention(a, b, c, causal=True, enable_gqa=True)
        with torch.no_grad():
            plain = flash_attention(q, k, v, causal=False, enable_gqa=True)
        # an expanded cotangent (zero strides) beside the dense one
        g0 = torch.autograd.grad(out, (a, b, c), d, retain_graph=True)
        g1 = torch.autograd.grad(out.sum(), (a, b, c))
        return [x.as_subclass(torch.Tensor) for x in (out.detach(), plain.detach(), *g0, *g1)]

    def refused():
        with pytest.raises(ValueError, match="16-byte aligned"):
            fn()
        return []
    # (a contiguous tensor off a 16-byte boundary is refused, unless padding copies it)
    both(monkeypatch, refused if form == "offset" and D != 80 else fn)


@pytest.mark.gpu
def test_which_calls_are_taken(device, monkeypatch):
    seen = counted(monkeypatch)
    q = rnd(1, 64, 2, 128).to(device).requires_grad_(True)
    out = flash_attention(q, q, q)
    out.backward(torch.ones_like(out))
    assert seen == {"attn_fwd": [1, 0], "attn_bwd": [1, 0]}
    flash_attention(*(q.detach()[..., :80],) * 3)          # padded: general
    assert seen["attn_fwd"] == [1, 0]
    flash_attention(*(q.detach()[..., ::2],) * 3)          # strided last dim: left
    assert seen["attn_fwd"] == [1, 1]


@pytest.mark.gpu
def test_tensors_that_refuse_their_address(device, monkeypatch):
    # data_ptr() throws while the GIL is released: the general path's error
    q = rnd(1, 1, 2, 128).to(device)
    kp, vp = (rnd(4, 16, 2, 128, seed=s).to(device) for s in (1, 2))
    torch._C._set_throw_on_mutable_data_ptr(vp)
    tables = torch.zeros(1, 1, dtype=torch.int32, device=device)
    lens = torch.ones(1, dtype=torch.int32, device=device)

    def fn():
        with pytest.raises(RuntimeError, match="data pointer"):
            paged_attention(q, kp, vp, tables, lens)
        return []
    both(monkeypatch, fn)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["BSHD", "BHSD"])
def test_dropout_window_and_second_derivative(device, monkeypatch, layout):
    q, k, v = (rnd(1, 130, 8, 64, seed=s).to(device) for s in range(3))

    def fn():
        torch.manual_seed(3)
        a, b, c = (x.detach().requires_grad_(True) for x in (q, k, v))
        o = flash_attention(a, b, c, dropout_p=0.3, layout=layout)
        w = sliding_window_attention(q, k, v, 20)
        return [o.detach(), w, *torch.autograd.grad(o, (a, b, c), torch.ones_like(o))]
    both(monkeypatch, fn)
    a = q.detach().requires_grad_(True)
    (g,) = torch.autograd.grad(flash_attention(a, k, v).float().square().sum(), a,
                               create_graph=True)
    with pytest.raises(RuntimeError):
        g.sum().backward()


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 80])
def test_windows_and_masks_as_int_reads_them(device, monkeypatch, D):
    # whatever int(...) takes, with its value: floats, numpy scalars, 0-dim
    # tensors; what int(...) refuses is refused
    q, k, v = (rnd(1, 70, 4, D, seed=s).to(device) for s in range(3))
    want = sliding_window_attention(q, k, v, 20)

    for W in (20.0, 20.9, np.float32(20), np.int64(20), torch.tensor(20)):
        def fn():
            a = q.detach().requires_grad_(True)
            o = sliding_window_attention(a, k, v, W)
            return [sliding_window_attention(q, k, v, W), o.detach(),
                    *torch.autograd.grad(o, a, torch.ones_like(o))]
        assert torch.equal(both(monkeypatch, fn)[0], want)
    for causal in (1.0, 2, np.True_, 0.5, np.float64(0.5), 0, "1"):
        (out,) = both(monkeypatch, lambda: [flash_attention(q, k, v, causal=causal)])
        assert torch.equal(out, flash_attention(q, k, v, causal=int(causal) != 0))
    for bad in (None, [], "x"):
        def refused():
            with pytest.raises((TypeError, ValueError)):
                flash_attention(q, k, v, causal=bad)
            return []
        both(monkeypatch, refused)


@pytest.mark.gpu
def test_paged_masks_as_int_reads_them(device, monkeypatch):
    kp, vp, q = (rnd(*n, 2, 64, seed=1).to(device) for n in ((3, 16), (3, 16), (1, 40)))
    tables = torch.tensor([[0, 2, 1]], dtype=torch.int32, device=device)
    lens = torch.tensor([40], dtype=torch.int32, device=device)
    for causal in (1.0, 2, np.True_, 0.5, 0):
        (out,) = both(monkeypatch,
                      lambda: [paged_attention(q, kp, vp, tables, lens, causal=causal)])
        assert torch.equal(out, paged_attention(q, kp, vp, tables, lens,
                                                causal=int(causal) != 0))
    # decode ignores it
    both(monkeypatch, lambda: [paged_attention(q[:, :1], kp, vp, tables, lens, causal=None)])

    def refused():
        with pytest.raises(TypeError):
            paged_attention(q, kp, vp, tables, lens, causal=None)
        return []
    both(monkeypatch, refused)


@pytest.mark.gpu
@pytest.mark.parametrize("H,H_kv,D,dtype", [(8, 2, 128, torch.bfloat16), (4, 4, 64, torch.float32),
                                            (4, 4, 72, torch.float16), (4, 2, 20, torch.float32)])
@pytest.mark.parametrize("alibi", [False, True])
def test_decode(device, monkeypatch, H, H_kv, D, dtype, alibi):
    kp, vp = (rnd(9, 16, H_kv, D, dtype=dtype, seed=s).to(device) for s in (1, 2))
    q = rnd(3, 1, H, D, dtype=dtype, seed=3).to(device)
    tables = torch.tensor([[0, 3, 5], [1, 2, -1], [4, 8, 7]], device=device)
    lens = torch.tensor([40, 0, 33], device=device)
    slopes = get_alibi_slopes(H, device=device) if alibi else None
    for it in (torch.int32, torch.int64):
        for view in (lambda x: x, lambda x: x.transpose(1, 2).contiguous().transpose(1, 2)):
            both(monkeypatch, lambda: [paged_attention(view(q), kp, vp, tables.to(it), lens.to(it),
                                                       alibi_slopes=slopes, enable_gqa=True)])


@pytest.mark.gpu
@pytest.mark.parametrize("H,H_kv,D,dtype", [(8, 2, 128, torch.bfloat16), (4, 4, 64, torch.float32),
                                            (4, 4, 72, torch.float16)])
@pytest.mark.parametrize("causal,alibi", [(True, False), (False, True)])
@pytest.mark.parametrize("S", [0, 2, 40])
def test_prefill(device, monkeypatch, H, H_kv, D, dtype, causal, alibi, S):
    kp, vp = (rnd(9, 16, H_kv, D, dtype=dtype, seed=s).to(device) for s in (1, 2))
    q = rnd(3, S, H, D, dtype=dtype, seed=3).to(device)
    tables = torch.tensor([[0, 3, 5], [1, 2, -1], [4, 8, 7]], device=device)
    lens = torch.tensor([40, 0, 33], device=device)
    slopes = get_alibi_slopes(H, device=device) if alibi else None
    for it in (torch.int32, torch.int64):
        for view in (lambda x: x, lambda x: x.transpose(1, 2).contiguous().transpose(1, 2)):
            both(monkeypatch, lambda: [paged_attention(view(q), kp, vp, tables.to(it), lens.to(it),
                                                       causal=causal, alibi_slopes=slopes,
                                                       enable_gqa=True)])


@pytest.mark.gpu
@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("counts", [None, 1, "tensor"])
def test_append_and_rope_at(device, monkeypatch, rope, counts):
    D, B, T = 64, 2, 3
    k, v = (rnd(B, T, 2, D, seed=s).to(device) for s in (1, 2))
    cos, sin = precompute_rope_cache(20, D, device=device)
    tables = torch.tensor([[0, 2], [1, 9]], dtype=torch.int32, device=device)
    starts = torch.tensor([14, 15], device=device)      # sequence 1 runs into a bad page
    n = torch.tensor([2, 3], device=device) if counts == "tensor" else counts

    def fn():
        kp, vp = (torch.zeros(4, 16, 2, D, dtype=k.dtype, device=device) for _ in range(2))
        err = torch.full((4 if rope else 3,), 7, dtype=torch.int32, device=device)
        got = store_kv(kp, vp, tables, k, v, starts, n, check=False, errors=err,
                       rope=(cos, sin) if rope else None)
        own = store_kv(kp, vp, tables, k, v, 15, n, check=False,
                       rope=(cos, sin) if rope else None)
        e1 = torch.full((1,), 7, dtype=torch.int32, device=device)
        x = rope_at(k, cos, sin, torch.tensor([1, 9], device=device), check=False, errors=e1)
        y = rope_at(k, cos, sin, [0, 2])
        return [kp, vp, got.clone(), own, x, e1, y]
    out = both(monkeypatch, fn)
    if counts != 1:
        assert out[2].tolist()[2] == 1
    with pytest.raises(ValueError):
        rope_at(k, cos, sin, [0, 19])
    with pytest.raises((ValueError, RuntimeError)):
        store_kv(torch.zeros(4, 16, 2, D, dtype=k.dtype, device=device),
                 torch.zeros(4, 16, 2, D, dtype=k.dtype, device=device), tables, k, v, starts)
