"""The native call path of the step / hand-over wrappers (csrc/sq_host.cpp) against the Python one: same bytes for the
calls it takes, None -- and therefore the Python path's own answer -- for every other call."""
import copy
import sys
import time
import types

import pytest
import torch

import statequant_amd as sq
from statequant_amd.kernels import (KDASlotLayout, Mamba2SlotLayout, PackedGDNState, PackedKDAState,
                                    PackedMamba2State, SlotLayout, _hip)
from statequant_amd.kernels.gga import GGAPacked, GGAPlan


class _Declines:
    """Answers every call as the native path answers one that is not ordinary."""

    def __getattr__(self, name):
        return lambda *a: None


class _Counts:
    """The native path, counting what it took."""

    def __init__(self):
        self.taken = 0

    def __getattr__(self, name):
        def call(*a):
            r = getattr(_sqhost(), name)(*a)
            self.taken += r is not None
            return r
        return call


def _sqhost():
    _hip.lib()
    from statequant_amd import _sqhost as m
    return m


def test_cpu_tensors_and_wrong_objects_are_declined():
    lay = SlotLayout(sq.Quantizer(8, 'k', 32), 4, 2, 64, 64)
    V = lay.views(lay.alloc(3, 'cpu'))
    st = lay._layout_struct()
    x, idx = torch.zeros(1, 2, 64), torch.ones(1, dtype=torch.int32)
    h = _hip.host()
    out = torch.zeros(1, 4, 64)
    for views, lay_ in ((V, st), ({}, st), (None, st), (V, b'short'), (V, None)):
        assert h.gdn_step(lay_, views, idx, x, x, out, out, 1.0, None, None, None, None) is None
    assert h.read(st, V, idx, False) is None and h.write(st, V, idx, torch.zeros(1, 4, 64, 64)) is None
    with pytest.raises(TypeError):
        h.gdn_step(st, V)
    with pytest.raises(RuntimeError, match='GPU'):
        lay.step(V, idx, x, x, out, out, 1.0, g=out[..., 0], beta=out[..., 0])


@pytest.mark.parametrize('other', ['missing', 'of another torch'])
def test_without_a_native_call_path_every_call_goes_the_python_way(other, monkeypatch):
    """The library needs no torch headers; the extension in front of it does.  Where it is missing or was built against
    another torch, nothing of it is called (its functions would raise here) and the Python path does every call."""
    import statequant_amd
    module = None if other == 'missing' else types.SimpleNamespace(TORCH='0.0')
    monkeypatch.setitem(sys.modules, 'statequant_amd._sqhost', module)
    monkeypatch.setattr(statequant_amd, '_sqhost', module, raising=False)
    if module is None:
        monkeypatch.delattr(statequant_amd, '_sqhost')
    monkeypatch.setattr(_hip, '_host', None)
    lay = SlotLayout(sq.Quantizer(8, 'k', 32), 4, 2, 64, 64)
    V = lay.views(lay.alloc(3, 'cpu'))
    lay._conv = lay._lay = lay._layout_struct()
    idx, x = torch.ones(1, dtype=torch.int32), torch.randn(1, 4, 64, 64)
    with pytest.warns(UserWarning, match='no native call path'):
        lay.write(V, idx, x)
    assert torch.allclose(lay.read(V, idx), x, atol=0.05)
    q, out = torch.zeros(1, 2, 64), torch.zeros(1, 4, 64)
    with pytest.raises(RuntimeError, match='GPU'):
        lay.step(V, idx, q, q, out, out, 1.0, g=out[..., 0], beta=out[..., 0])
    assert _hip.host().gdn_step(*range(12)) is None


def test_the_extension_is_rebuilt_for_another_torch(monkeypatch):
    from statequant_amd.csrc import build
    stamp = build._host_stamp()
    monkeypatch.setattr(torch, '__version__', '0.0')
    assert build._host_stamp() != stamp


def test_a_declined_call_costs_little():
    """The Python path follows a declined call, so declining must not add to it noticeably: 0.15 us, where an unwound C++
    exception took 3.6 (the Python path itself takes 17)."""
    lay = SlotLayout(sq.Quantizer(8, 'k', 32), 4, 2, 64, 64)
    V = lay.views(lay.alloc(3, 'cpu'))
    st, h, idx, n = lay._layout_struct(), _hip.host(), torch.ones(1, dtype=torch.int32), 2000
    best = float('inf')
    for _ in range(7):                                  # the least of several: the machine may be busy
        t = time.perf_counter()
        for _ in range(n):
            h.read(st, V, idx, False)
        best = min(best, (time.perf_counter() - t) / n)
    assert best < 2e-6, best


def _slot_case(family, fmt, gate, rows, gen, dev):
    HV, HK, D = 4, 4 if family == 'kda' else 2, 64
    q8 = sq.Quantizer(*fmt) if fmt else 'bf16'
    cls = {'gdn': SlotLayout, 'mamba2': Mamba2SlotLayout}.get(family)
    lay = KDASlotLayout(q8, HV, D, D) if family == 'kda' else cls(q8, HV, HK, D, D)
    r = lambda *s: torch.randn(*s, device=dev, generator=gen)                     # noqa: E731
    idx = torch.tensor([2, 0, 4, 1, 3][:rows], dtype=torch.int32, device=dev)
    S = r(rows, HV, D, D)
    x = r(rows, 2 * HK * D + HV * D).bfloat16()
    q, k, v = x[:, :HK * D].unflatten(1, (HK, D)), x[:, HK * D:2 * HK * D].unflatten(1, (HK, D)), x[:, 2 * HK * D:].unflatten(1, (HV, D))
    order = torch.arange(rows, dtype=torch.int32, device=dev).flip(0).contiguous()
    if family == 'mamba2':
        args = (v, r(rows, HV).bfloat16(), q, k)
        kw = dict(A=-r(HV).abs(), D=r(HV), dt_bias=r(HV), dt_limit=(0.01, 2.0) if gate else (0., float('inf')), order=order)
    elif family == 'kda':
        args, kw = (q, k, v, -r(rows, HV, D).abs(), torch.sigmoid(r(rows, HV))), dict(order=order)
    else:
        args = (q, k, v)
        kw = dict(gate=(r(rows, HV).bfloat16(), r(rows, HV).bfloat16(), r(HV), r(HV))) if gate else \
            dict(g=-r(rows, HV).abs(), beta=torch.sigmoid(r(rows, HV)))
        kw.update(order=order)

    def step(V, out):
        if family == 'gdn':
            return lay.step(V, idx, *args, out, D ** -0.5, **kw)
        if family == 'kda':
            return lay.step(V, idx, *args, out, **kw)
        return lay.step(V, idx, *args, out, **kw)
    return lay, idx, S, step, (rows, HV, D)


@pytest.mark.gpu
@pytest.mark.parametrize('family', ['gdn', 'kda', 'mamba2'])
@pytest.mark.parametrize('fmt,gate', [((8, 'k', 32), False), ((4, 'v', 32), True), (None, False)])
def test_slot_calls_are_the_python_paths(family, fmt, gate, monkeypatch):
    dev, rows = 'cuda', 5
    got = []
    for native in (True, False):
        gen = torch.Generator(device=dev).manual_seed(3)
        lay, idx, S, step, shape = _slot_case(family, fmt, gate, rows, gen, dev)
        V = lay.views(lay.alloc(6, dev))
        lay.write(V, idx, S * 0.5)                     # the first calls of a layout go the Python way
        out = torch.full(shape, 7.0, device=dev, dtype=torch.bfloat16)
        lay.read(V, idx)
        step(V, out)
        host = _Counts() if native else _Declines()
        monkeypatch.setattr(_hip, 'host', lambda: host)
        for _ in range(9):
            step(V, out)
        read = lay.read(V, idx)
        lay.write(V, idx[:2], S[:2].contiguous())
        monkeypatch.undo()
        if native:
            assert host.taken == 11
        got.append([out.clone(), read, *(V[k].clone() for k in sorted(V))])
    for a, b in zip(*got):
        assert a.dtype == b.dtype and torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


@pytest.mark.gpu
@pytest.mark.parametrize('family', ['gdn', 'kda', 'mamba2'])
def test_lockstep_and_mixed_width_calls_are_the_python_paths(family, monkeypatch):
    dev, B, H, D = 'cuda', 3, 4, 64
    got = []
    for native in (True, False):
        gen = torch.Generator(device=dev).manual_seed(4)
        r = lambda *s: torch.randn(*s, device=dev, generator=gen)                 # noqa: E731
        host = _Counts() if native else _Declines()
        q, k, v = r(B * H, D).bfloat16(), r(B * H, D).bfloat16(), r(B * H, D).bfloat16()
        S = r(B, H, D, D) * 0.3
        cls = dict(gdn=PackedGDNState, kda=PackedKDAState, mamba2=PackedMamba2State)[family]
        st = cls(S, sq.Quantizer(8, 'k', 32), hv=H)
        g = -r(B, H, D).abs() if family == 'kda' else -r(B * H).abs()
        beta = torch.sigmoid(r(B * H))
        lay = GGAPacked(GGAPlan({0: ([2, 4, 8, 16], torch.linspace(0.5, 1.5, H * D).view(H, D))}), H, H, D, D, pw=True)
        V = lay.views(lay.alloc(B + 1, dev))
        lay.prepare(V['blob'].device)
        idx = torch.arange(1, B + 1, dtype=torch.int32, device=dev)
        V['blob'].zero_()
        out = torch.zeros(B, H, D, device=dev, dtype=torch.bfloat16)
        monkeypatch.setattr(_hip, 'host', lambda: host)
        for _ in range(9):
            if family == 'mamba2':
                st.step(v, beta.view(B, H), k.view(B, H, D), q.view(B, H, D), -beta[:H].contiguous())
            else:
                st.step(q, k, v, g, beta, D ** -0.5)
            lay.step(V, idx, q.view(B, H, D), k.view(B, H, D), v.view(B, H, D), out, D ** -0.5,
                     g=-beta.view(B, H), beta=beta.view(B, H), layer=0)
        monkeypatch.undo()
        if native:
            assert host.taken == 18
        copy.deepcopy(lay._geometry)
        got.append([st.O.clone(), out, V['blob'].clone(), *(st.T[f].clone() for f in sorted(st.T))])
    for a, b in zip(*got):
        assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


@pytest.mark.gpu
def test_calls_out_of_the_ordinary_are_declined():
    """Other classes, transforms, devices, dtypes and strides: None, whatever the Python path then makes of them."""
    dev, rows = 'cuda', 3
    gen = torch.Generator(device=dev).manual_seed(5)
    lay, idx, S, step, shape = _slot_case('gdn', (8, 'k', 32), False, rows, gen, dev)
    V = lay.views(lay.alloc(6, dev))
    st = lay._layout_struct()
    h = _hip.host()
    x = torch.randn(rows, 8, 64, device=dev).bfloat16()
    q, v, gb = x[:, :2], x[:, 4:], torch.rand(rows, 4, device=dev)
    out = torch.zeros(shape, device=dev, dtype=torch.bfloat16)

    class Sub(torch.Tensor):
        pass
    base = dict(lay=st, views=V, idx=idx, q=q, k=q, v=v, out=out, scale=0.1, g=gb, beta=gb, gate=None, order=None)
    assert h.gdn_step(*base.values()) == 0
    for change in (dict(q=q.as_subclass(Sub)), dict(q=q.float().cpu()), dict(q=q.double()), dict(q=x[:, :2, ::2]),
                   dict(q=q.transpose(0, 1)), dict(q=q[0]), dict(idx=idx.long()), dict(idx=idx.cpu()), dict(idx=idx[:0]),
                   dict(out=out[:2]), dict(out=out.transpose(0, 1)), dict(g=None), dict(gate=(gb, gb, gb[0], gb[0])),
                   dict(gate=[gb] * 4, g=None, beta=None), dict(scale=torch.tensor(0.1)), dict(order=idx[:2]),
                   dict(order=idx.long()), dict(views={**V, 'S': V['S'].cpu()}), dict(views={k: t for k, t in V.items() if k != 'KB'}),
                   dict(q=torch._neg_view(q)), dict(lay=None)):
        assert h.gdn_step(*{**base, **change}.values()) is None, change.keys()

    def under_vmap(t):
        assert h.gdn_step(*{**base, 'beta': t}.values()) is None
        return t
    torch.vmap(under_vmap)(torch.rand(2, rows, 4, device=dev))


@pytest.mark.gpu
@pytest.mark.parametrize('fmt', [(4, 'k', 32), (8, 'v', 32), None])
def test_views_cut_natively_are_the_views_the_python_code_cuts(fmt, monkeypatch):
    """Same geometry, dtype, memory and base, for a blob of its own, a part of one and one with wider slots; what the
    Python code refuses stays refused."""
    for family in ('gdn', 'kda', 'mamba2'):
        lay = _slot_case(family, fmt, False, 3, torch.Generator(device='cuda').manual_seed(1), 'cuda')[0]
        big = torch.zeros(9, lay.nbytes + 32, dtype=torch.uint8, device='cuda')
        lay._layout_struct()
        for blob in (lay.alloc(5), big, big[2:7], big[:, 16:], big[::2], lay.alloc(1)):
            got = _hip.host().views(blob, lay.fields, lay.nbytes)
            with monkeypatch.context() as m:
                m.setattr(_hip, '_host', _Declines())
                want = lay.views(blob)
            assert list(got) == list(want) == list(lay.fields)
            for k in want:
                a, b = got[k], want[k]
                assert (a.shape, a.stride(), a.dtype, a.data_ptr(), a.storage_offset()) == \
                    (b.shape, b.stride(), b.dtype, b.data_ptr(), b.storage_offset())
                assert (a._version, a._base.shape, a._base.dtype) == (b._version, b._base.shape, b._base.dtype)
        for blob in (big[:, 8:], big[:, :lay.nbytes - 16], big.t(), big.view(torch.int8), big[0], lay.alloc(2, 'cpu')):
            assert _hip.host().views(blob, lay.fields, lay.nbytes) is None
        for blob in (big[:, 8:], big[:, :lay.nbytes - 16]):
            with pytest.raises(AssertionError):
                lay.views(blob)
