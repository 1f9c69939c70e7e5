"""The workgroup step kernels against the one-wavefront kernels on the same state, token by token, for the formats and
shapes at the edges of what the workgroup kernels serve.  Both kinds are held to the oracle elsewhere; here every step
of one starts from the other's state, so a difference is one step's.

Bounds: the two kinds add the same fp32 products in another order -- outputs within d_k 2^-24 of the largest one (1e-5
for d_k = 128); a stored or buffered value may come out one step off where it lies within that of a rounding boundary,
a scale one fp16 number off likewise (1e-4 of them, and the entries of a re-scaled vector)."""
import pytest
import torch

import statequant_amd as sq
from _util import code_diff
from statequant_amd.kernels import KDASlotLayout, Mamba2SlotLayout, SlotLayout, _hip

pytestmark = pytest.mark.gpu
DEV = 'cuda'

CASES = [
    # value-axis groups of one row block: one / two row blocks per wavefront, both buffers, short and long periods
    ('gdn', (4, 'v', 32), (4, 2, 128, 128), 8, 8), ('gdn', (8, 'v', 32), (4, 2, 128, 128), 8, 8),
    ('gdn', (4, 'v', 32), (3, 3, 128, 128), 1, 16), ('gdn', (8, 'v', 32), (6, 2, 64, 64), 16, 16),
    ('gdn', (4, 'v', 32), (4, 2, 64, 64), 4, 8), ('gdn', (8, 'v', 32), (2, 1, 128, 256), 2, 8),
    ('mamba2', (4, 'v', 32), (8, 2, 128, 64), 8, 8), ('mamba2', (8, 'v', 32), (6, 2, 128, 64), 4, 16),
    ('mamba2', (8, 'v', 32), (4, 1, 128, 128), 16, 8), ('mamba2', (4, 'v', 32), (3, 3, 64, 64), 1, 8),
    # KDA: one to eight wavefronts per head, key- and value-axis groups
    ('kda', (4, 'k', 32), (3, 3, 128, 128), 8, 8), ('kda', (8, 'k', 128), (2, 2, 128, 128), 8, 16),
    ('kda', (8, 'k', 32), (5, 5, 64, 32), 4, 8), ('kda', (4, 'k', 64), (2, 2, 64, 64), 16, 16),
    ('kda', (8, 'k', 64), (2, 2, 128, 256), 1, 8), ('kda', (4, 'v', 32), (3, 3, 128, 128), 8, 8),
    ('kda', (8, 'v', 32), (2, 2, 128, 128), 16, 16), ('kda', (8, 'v', 32), (3, 3, 64, 32), 2, 8),
    # d_k 96: rows padded to 128 columns in LDS, one to four scale groups, the last one ragged, half empty or whole
    ('gdn', (4, 'k', 64), (5, 5, 96, 192), 8, 8), ('gdn', (4, 'k', 32), (4, 2, 96, 192), 16, 16),
    ('gdn', (8, 'k', 128), (3, 3, 96, 96), 4, 8), ('gdn', (8, 'k', 32), (6, 2, 96, 192), 8, 16),
    ('gdn', (8, 'k', 64), (2, 2, 96, 96), 1, 8), ('gdn', (4, 'v', 32), (3, 3, 96, 192), 8, 8),
    ('gdn', (8, 'v', 32), (2, 1, 96, 96), 2, 16), ('kda', (4, 'k', 32), (5, 5, 96, 96), 8, 8),
    ('kda', (8, 'k', 32), (2, 2, 96, 96), 16, 16), ('kda', (4, 'v', 32), (3, 3, 96, 96), 4, 8),
    ('kda', (8, 'v', 32), (2, 2, 96, 96), 8, 16),
    # the bf16 state
    ('gdn', 'bf16', (4, 2, 128, 128), 8, 8), ('gdn', 'bf16', (6, 3, 64, 64), 16, 16), ('gdn', 'bf16', (3, 3, 96, 192), 8, 8),
    ('gdn', 'bf16', (2, 1, 96, 96), 1, 16), ('kda', 'bf16', (3, 3, 128, 128), 8, 8), ('kda', 'bf16', (2, 2, 96, 96), 4, 16),
    ('kda', 'bf16', (5, 5, 64, 32), 8, 8), ('mamba2', 'bf16', (8, 2, 128, 64), 8, 8),
    ('mamba2', 'bf16', (4, 1, 128, 128), 16, 16), ('mamba2', 'bf16', (6, 6, 64, 64), 2, 8),
    # d_v 80: the last row block half empty
    ('mamba2', (8, 'k', 128), (6, 2, 128, 80), 8, 8), ('mamba2', (4, 'k', 64), (4, 1, 128, 80), 16, 16),
    ('mamba2', (8, 'k', 32), (12, 4, 96, 80), 4, 8), ('mamba2', (4, 'k', 32), (3, 3, 96, 80), 1, 8),
    ('mamba2', 'bf16', (4, 1, 128, 80), 8, 8), ('mamba2', 'bf16', (6, 6, 96, 80), 2, 16),
]


def _layout(family, fmt, shape, m, bb):
    hv, hk, dk, dv = shape
    fmt = fmt if isinstance(fmt, str) else sq.Quantizer(*fmt)
    if family == 'kda':
        return KDASlotLayout(fmt, hv, dk, dv, m=m, buffer_bits=bb)
    cls = {'gdn': SlotLayout, 'mamba2': Mamba2SlotLayout}[family]
    return cls(fmt, hv, hk, dk, dv, m=m, buffer_bits=bb)


def _token(family, gen, rows, shape):
    hv, hk, dk, dv = shape
    r = lambda *s: torch.randn(*s, generator=gen).to(DEV)          # noqa: E731
    if family == 'mamba2':
        return dict(x=r(rows, hv, dv), dt=r(rows, hv), B=r(rows, hk, dk), C=r(rows, hk, dk))
    g = r(rows, hv, dk) if family == 'kda' else r(rows, hv)
    return dict(q=r(rows, hk, dk), k=r(rows, hk, dk), v=r(rows, hv, dv), g=-torch.nn.functional.softplus(g),
                beta=torch.sigmoid(r(rows, hv)))


def _step(family, lay, V, idx, t, out, model, order=None):
    if family == 'mamba2':
        lay.step(V, idx, t['x'], t['dt'], t['B'], t['C'], out, *model, order=order)
    elif family == 'kda':
        lay.step(V, idx, t['q'], t['k'], t['v'], t['g'], t['beta'], out, order=order)
    else:
        lay.step(V, idx, t['q'], t['k'], t['v'], out, lay.DK ** -0.5, g=t['g'], beta=t['beta'], order=order)


def _compare(family, fmt, shape, m, bb, idx):
    hv, hk, dk, dv = shape
    lay = _layout(family, fmt, shape, m, bb)
    gen = torch.Generator().manual_seed(5)
    rows = idx.shape[0]
    live = idx > 0
    blob = lay.alloc(int(idx.max()) + 1, DEV)
    V = lay.views(blob)
    S0 = torch.randn(rows, hv, dv, dk, generator=gen).to(DEV) * 0.4
    S0[0] = 0.0                                                     # a fresh sequence: its first fold is the exact one
    lay.write(V, idx, S0)
    r = lambda *s: torch.randn(*s, generator=gen).to(DEV)          # noqa: E731
    model = (-torch.exp(r(hv)), r(hv), r(hv)) if family == 'mamba2' else None
    codes = off = entries = flips = scales = scales_off = 0
    for step in range(2 * m + 3):
        if step == 1 and m > 1:                                     # from here on the sequences are out of step
            lay.write(V, idx[3:5], S0[3:5])
        t = _token(family, gen, rows, shape)
        twin = blob.clone()
        W = lay.views(twin)
        outs = [torch.full((rows, hv, dv), 3.0, device=DEV) for _ in range(2)]
        _step(family, lay, V, idx, t, outs[0], model)
        _hip.select_instances(no_group_kernel=True)
        try:
            _step(family, lay, W, idx, t, outs[1], model)
        finally:
            _hip.select_instances()
        assert torch.equal(outs[0][~live], torch.zeros_like(outs[0][~live]))
        assert ((outs[0] - outs[1]).abs().max() / outs[1].abs().max()).item() <= 1e-5, step
        for name in V:
            a, b = V[name], W[name]
            if name == 'NPTR':
                assert torch.equal(a, b)
            elif name == 'S' and lay.bits == 16:                    # a bf16 value next to a rounding boundary
                d = (a.view(torch.int16).int() - b.view(torch.int16).int()).abs()
                big = b.float().abs() > 1e-3                        # (below, sums cancel and steps are smaller than their error)
                assert d[big].max().item() <= 1 and torch.allclose(a.float(), b.float(), rtol=2 ** -7, atol=1e-5)
                codes, off = codes + d.numel(), off + int((d > 0).sum())
            elif name == 'S':
                mism, far, n = code_diff(a.cpu(), b.cpu(), lay.bits)
                assert far == 0
                codes, off = codes + n, off + mism
            elif name in ('SC', 'KBS', 'UBS'):
                d = (a.view(torch.int16).int() - b.view(torch.int16).int()).abs()
                assert d.max().item() <= 1
                scales, scales_off = scales + d.numel(), scales_off + int((d > 0).sum())
            elif name in ('KB', 'UB'):
                entries, flips = entries + a.numel(), flips + int((a != b).sum())
            else:
                assert torch.allclose(a, b, rtol=1e-6, atol=1e-7), name
    # bf16 steps are 2^-8 of a value; the two sums of up to 17 terms differ by some 2^-23 of it, and by more where they cancel
    assert off <= (2e-3 if lay.bits == 16 else 1e-4) * codes and scales_off <= 1e-4 * scales + 2, (off, codes, scales_off, scales)
    assert flips <= 1e-4 * entries + 2 * max(dk, dv), (flips, entries)


@pytest.mark.parametrize('family,fmt,shape,m,bb', CASES)
def test_group_kernel_matches_the_one_wavefront_kernel(family, fmt, shape, m, bb):
    _compare(family, fmt, shape, m, bb, torch.tensor([3, 1, 0, 9, 4, -1, 6], dtype=torch.int32, device=DEV))


@pytest.mark.parametrize('family,fmt,shape,m,bb,rows', [
    ('gdn', (8, 'v', 32), (32, 16, 64, 64), 8, 16, 34), ('gdn', (4, 'v', 32), (32, 16, 64, 64), 16, 8, 34),
    ('mamba2', (8, 'v', 32), (64, 8, 64, 64), 16, 16, 18), ('mamba2', (4, 'v', 32), (64, 8, 64, 64), 4, 16, 18),
    ('kda', (8, 'k', 32), (32, 32, 64, 32), 4, 8, 10), ('kda', (8, 'v', 32), (32, 32, 64, 32), 2, 16, 10),
    ('kda', (4, 'k', 64), (32, 32, 64, 32), 16, 8, 14), ('kda', 'bf16', (32, 32, 64, 32), 8, 8, 10)])
def test_group_kernels_that_serve_larger_launches_only(family, fmt, shape, m, bb, rows):
    idx = torch.randperm(rows, generator=torch.Generator().manual_seed(1)).to(torch.int32).to(DEV)      # one padding row
    _compare(family, fmt, shape, m, bb, idx)


@pytest.mark.parametrize('family,fmt,shape,m,bb,rows', [
    ('kda', (4, 'k', 64), (32, 32, 64, 64), 2, 8, 160), ('kda', (8, 'v', 32), (32, 32, 64, 64), 16, 16, 128),
    ('kda', (8, 'k', 32), (32, 32, 64, 32), 16, 8, 128), ('kda', (8, 'k', 32), (32, 32, 128, 128), 16, 8, 128),
    ('kda', 'bf16', (32, 32, 64, 32), 2, 8, 128),
    ('gdn', (4, 'k', 64), (20, 20, 96, 96), 4, 8, 176), ('gdn', 'bf16', (30, 30, 96, 192), 2, 16, 88),
    ('mamba2', 'bf16', (96, 8, 96, 80), 2, 8, 88),
    # ... or from one row block per wavefront to two
    ('gdn', (4, 'v', 32), (32, 16, 128, 128), 4, 8, 96), ('gdn', (8, 'v', 32), (32, 16, 128, 128), 8, 8, 104),
    ('gdn', (4, 'v', 32), (32, 16, 128, 128), 4, 8, 136), ('gdn', (8, 'k', 32), (32, 16, 128, 128), 2, 8, 72),
    ('gdn', (4, 'k', 64), (32, 16, 128, 128), 4, 8, 88), ('gdn', (4, 'k', 64), (20, 20, 96, 96), 4, 8, 184),
    ('mamba2', (8, 'k', 128), (96, 8, 128, 80), 4, 8, 72), ('mamba2', (4, 'k', 64), (96, 8, 128, 80), 2, 8, 56)])
def test_a_dispatch_order_that_changes_the_kernel(family, fmt, shape, m, bb, rows):
    """Launches of so many heads that a dispatch order moves them to the one-wavefront kernel (bounds as above)."""
    hv, hk, dk, dv = shape
    lay = _layout(family, fmt, shape, m, bb)
    gen = torch.Generator().manual_seed(8)
    blobs = [lay.alloc(rows + 1, DEV) for _ in range(2)]
    V = [lay.views(b) for b in blobs]
    idx = torch.arange(1, rows + 1, dtype=torch.int32, device=DEV)
    order = torch.randperm(rows, generator=gen).to(torch.int32).to(DEV)
    S0 = torch.randn(8, hv, dv, dk, generator=gen).to(DEV) * 0.4
    lay.write(V[0], idx, S0.repeat(rows // 8, 1, 1, 1))
    r = lambda *s: torch.randn(*s, generator=gen).to(DEV)          # noqa: E731
    model = (-torch.exp(r(hv)), r(hv), r(hv)) if family == 'mamba2' else None
    for step in range(m + 1):
        blobs[1].copy_(blobs[0])
        t = _token(family, gen, rows, shape)
        outs = [torch.zeros(rows, hv, dv, device=DEV) for _ in range(2)]
        for W, o, ordered in zip(V, outs, (None, order)):
            _step(family, lay, W, idx, t, o, model, order=ordered)
        assert ((outs[0] - outs[1]).abs().max() / outs[0].abs().max()).item() <= 1e-5, step
        assert torch.equal(V[0]['NPTR'], V[1]['NPTR'])
        # this token's entry of the buffer: a value one step off moves its whole row of the state by that step times the
        # key -- more than a code step where the row's value was near zero -- and a key or a scale that differs, the head
        off = lambda name: (V[0][name] != V[1][name])[1:].flatten(2).any(2)        # noqa: E731
        heads = off('KB').repeat_interleave(hv // hk, 1)
        if 'UBS' in V[0]:
            heads |= off('UBS') | off('KBS').repeat_interleave(hv // hk, 1)
        rows_off = (V[0]['UB'] != V[1]['UB'])[1:].any(2) | heads[..., None]
        assert rows_off.float().mean().item() <= 1e-3
        A, B = (W['S'][1:][~rows_off].cpu() for W in V)
        mism, far, n = code_diff(A, B, lay.bits)
        assert far == 0 and mism <= (2e-3 if lay.bits == 16 else 1e-4) * n


@pytest.mark.parametrize('family,fmt,shape,rows', [
    # workgroup / one-wavefront kernel
    ('gdn', (4, 'k', 64), (40, 40, 96, 96), 128), ('kda', (4, 'k', 32), (40, 40, 96, 96), 128),
    ('mamba2', (8, 'k', 32), (40, 8, 128, 80), 128),
    # one / two row blocks per wavefront
    ('gdn', (8, 'k', 32), (32, 16, 128, 128), 64), ('gdn', (4, 'k', 64), (32, 16, 128, 128), 64),
    ('gdn', (8, 'k', 128), (32, 8, 128, 128), 64), ('gdn', (4, 'v', 32), (32, 16, 128, 128), 96),
    ('gdn', (8, 'v', 32), (24, 24, 128, 128), 128), ('gdn', (4, 'v', 32), (32, 16, 128, 128), 104),
    ('gdn', (8, 'v', 32), (32, 16, 128, 128), 192), ('gdn', (8, 'k', 64), (30, 30, 96, 192), 26),
    ('mamba2', (8, 'k', 128), (128, 8, 128, 64), 6), ('mamba2', (4, 'k', 32), (96, 8, 128, 64), 8),
    ('gdn', (4, 'k', 64), (32, 16, 128, 128), 72), ('gdn', (8, 'k', 32), (32, 16, 128, 128), 96),
    ('gdn', (4, 'v', 32), (32, 16, 128, 128), 200), ('gdn', (8, 'v', 32), (32, 16, 128, 128), 256),
    ('mamba2', (8, 'k', 128), (128, 8, 128, 64), 14), ('mamba2', (4, 'k', 32), (128, 8, 128, 64), 19),
    # workgroup / one-wavefront kernel again
    ('mamba2', (4, 'k', 64), (96, 8, 128, 80), 120), ('mamba2', (4, 'k', 32), (96, 8, 96, 80), 64)])
def test_launches_either_side_of_a_head_count_agree(family, fmt, shape, rows):
    """A launch at the number of heads where another kernel takes over, and the same launch one sequence shorter (bounds
    as above)."""
    hv, hk, dk, dv = shape
    lay = _layout(family, fmt, shape, 4, 8)
    gen = torch.Generator().manual_seed(6)
    blobs = [lay.alloc(rows + 1, DEV) for _ in range(2)]
    V = [lay.views(b) for b in blobs]
    idx = torch.arange(1, rows + 1, dtype=torch.int32, device=DEV)
    lay.write(V[0], idx, torch.randn(rows, hv, dv, dk, generator=gen).to(DEV) * 0.4)
    r = lambda *s: torch.randn(*s, generator=gen).to(DEV)          # noqa: E731
    model = (-torch.exp(r(hv)), r(hv), r(hv)) if family == 'mamba2' else None
    for step in range(5):
        blobs[1].copy_(blobs[0])
        t = _token(family, gen, rows, shape)
        outs = [torch.zeros(rows, hv, dv, device=DEV) for _ in range(2)]
        _step(family, lay, V[0], idx, t, outs[0], model)
        _step(family, lay, V[1], idx[:-1], {k: x[:-1] for k, x in t.items()}, outs[1], model)
        assert ((outs[0] - outs[1])[:-1].abs().max() / outs[0].abs().max()).item() <= 1e-5, step
        mism, far, n = code_diff(V[0]['S'][1:rows].cpu(), V[1]['S'][1:rows].cpu(), lay.bits)
        assert far == 0 and mism <= 1e-4 * n


@pytest.mark.parametrize('family,fmt,shape', [('gdn', (4, 'k', 64), (4, 2, 128, 128)), ('gdn', (4, 'v', 32), (4, 2, 96, 96)),
                                              ('kda', (4, 'k', 32), (3, 3, 128, 128)), ('mamba2', (4, 'k', 32), (4, 2, 128, 80))])
def test_int4_states_aligned_to_8_bytes(family, fmt, shape):
    """The C ABI's alignment for int4 codes (the slot layouts give 16): the same tokens on a state 8 bytes off, which the
    16-byte accesses of the workgroup kernels do not take (bounds as above)."""
    hv, hk, dk, dv = shape
    lay = _layout(family, fmt, shape, 2, 8)
    gen = torch.Generator().manual_seed(7)
    rows, idx = 3, torch.tensor([2, 1, 4], dtype=torch.int32, device=DEV)
    V = [lay.views(lay.alloc(5, DEV)) for _ in range(2)]
    odd = torch.zeros(5 * V[0]['S'][0].numel() + 8, dtype=torch.uint8, device=DEV)[8:]
    V[1]['S'] = odd.view(5, *V[0]['S'].shape[1:])
    assert V[1]['S'].data_ptr() % 16 == 8
    S0 = torch.randn(rows, hv, dv, dk, generator=gen).to(DEV) * 0.4
    r = lambda *s: torch.randn(*s, generator=gen).to(DEV)          # noqa: E731
    model = (-torch.exp(r(hv)), r(hv), r(hv)) if family == 'mamba2' else None
    for W in V:
        lay.write(W, idx, S0)
    assert torch.equal(lay.read(V[0], idx), lay.read(V[1], idx))
    for step in range(5):
        t = _token(family, gen, rows, shape)
        outs = [torch.zeros(rows, hv, dv, device=DEV) for _ in range(2)]
        for W, o in zip(V, outs):
            _step(family, lay, W, idx, t, o, model)
        assert ((outs[0] - outs[1]).abs().max() / outs[0].abs().max()).item() <= 1e-5, step
        mism, far, n = code_diff(V[0]['S'].cpu(), V[1]['S'].cpu(), 4)
        assert far == 0 and mism <= 1e-4 * n
        for name in V[0]:                                           # a tie that went the other way is not carried on
            V[1][name].copy_(V[0][name])


@pytest.mark.parametrize('family,fmt,shape,rows,form', [
    # GDN: g and beta, or the gate in the kernel; head counts that are powers of two and not, one and two row blocks per
    # wavefront, the one-wavefront kernel of launches of many 96-wide heads
    ('gdn', (8, 'k', 32), (32, 16, 128, 128), 5, 'gate'), ('gdn', (8, 'k', 128), (32, 16, 128, 128), 70, 'plain'),
    ('gdn', (4, 'k', 64), (32, 16, 128, 128), 70, 'gate'), ('gdn', (4, 'v', 32), (32, 16, 128, 128), 5, 'gate'),
    ('gdn', (8, 'v', 32), (32, 16, 128, 128), 200, 'plain'), ('gdn', 'bf16', (32, 16, 128, 128), 5, 'gate'),
    ('gdn', (4, 'k', 64), (30, 30, 96, 192), 5, 'gate'), ('gdn', (8, 'k', 32), (30, 30, 96, 192), 40, 'plain'),
    ('gdn', 'bf16', (30, 30, 96, 192), 5, 'plain'), ('gdn', (4, 'k', 64), (40, 40, 96, 96), 130, 'gate'),
    # KDA: fp32 g and beta
    ('kda', (4, 'k', 32), (32, 32, 128, 128), 5, 'plain'), ('kda', (8, 'v', 32), (32, 32, 128, 128), 5, 'plain'),
    ('kda', (4, 'k', 32), (20, 20, 96, 96), 5, 'plain'), ('kda', 'bf16', (20, 20, 96, 96), 5, 'plain'),
    ('kda', (8, 'k', 32), (32, 32, 64, 32), 5, 'plain'), ('kda', (8, 'k', 32), (32, 32, 64, 32), 10, 'plain'),
    # Mamba2: dt of either type, head counts that are powers of two and not
    ('mamba2', (8, 'k', 128), (128, 8, 128, 64), 5, 'bf16 dt'), ('mamba2', (8, 'k', 128), (128, 8, 128, 64), 9, 'fp32 dt'),
    ('mamba2', (4, 'k', 64), (112, 8, 128, 64), 9, 'bf16 dt'), ('mamba2', (4, 'v', 32), (96, 8, 128, 64), 5, 'fp32 dt'),
    ('mamba2', (8, 'k', 128), (96, 8, 128, 80), 5, 'bf16 dt'), ('mamba2', 'bf16', (96, 8, 128, 80), 5, 'bf16 dt')])
def test_serving_case_instances_leave_the_bytes_of_the_general_one(family, fmt, shape, rows, form):
    """The tokens as serving layers hand them over (bf16, fp32 gates) through the instances with that compiled in and
    through the general one, two fold periods of sequences out of step, a padding row: the same bytes throughout."""
    hv, hk, dk, dv = shape
    lay = _layout(family, fmt, shape, 8, 8)
    gen = torch.Generator(device=DEV).manual_seed(9)
    r = lambda *s: torch.randn(*s, device=DEV, generator=gen)      # noqa: E731
    blobs = [lay.alloc(rows, DEV) for _ in range(2)]
    V = [lay.views(b) for b in blobs]
    idx = torch.randperm(rows, device=DEV, generator=gen).to(torch.int32)
    lay.write(V[0], idx, r(rows, hv, dv, dk) * 0.4)
    blobs[1].copy_(blobs[0])
    for step in range(17):
        if step in (3, 6):
            for W in V:
                lay.write(W, idx[:rows // 2], torch.ones(rows // 2, hv, dv, dk, device=DEV) * 0.1)
        x = r(rows, 2 * hk * dk + hv * dv).bfloat16()
        q, k, v = (x[:, lo:hi].unflatten(1, (h, d)) for lo, hi, h, d in (
            (0, hk * dk, hk, dk), (hk * dk, 2 * hk * dk, hk, dk), (2 * hk * dk, 2 * hk * dk + hv * dv, hv, dv)))
        g = -torch.nn.functional.softplus(r(rows, hv, dk) if family == 'kda' else r(rows, hv))
        beta, raw, model = torch.sigmoid(r(rows, hv)), r(rows, hv).bfloat16(), (r(hv) * 0.3, r(hv) * 0.3, r(hv))
        outs = [torch.full((rows, hv, dv), 3.0, device=DEV, dtype=torch.bfloat16) for _ in range(2)]
        for i, (W, out) in enumerate(zip(V, outs)):
            _hip.select_instances(no_specialised=i == 1)
            try:
                if family == 'mamba2':
                    lay.step(W, idx, v, raw if form == 'bf16 dt' else raw.float(), q, k, out, -torch.exp(model[0]), *model[1:])
                elif family == 'kda':
                    lay.step(W, idx, q, k, v, g, beta, out)
                elif form == 'gate':
                    lay.step(W, idx, q, k, v, out, dk ** -0.5, gate=(raw, raw.flip(0), *model[:2]))
                else:
                    lay.step(W, idx, q, k, v, out, dk ** -0.5, g=g, beta=beta)
            finally:
                _hip.select_instances()
        assert torch.equal(outs[0], outs[1]) and torch.equal(blobs[0], blobs[1]), step


@pytest.mark.parametrize('huge', ['q', 'k'])
@pytest.mark.parametrize('family,fmt,shape', [('gdn', (8, 'k', 128), (2, 2, 128, 128)), ('gdn', (4, 'v', 32), (4, 2, 64, 64)),
                                              ('gdn', 'bf16', (2, 1, 96, 96)), ('kda', (4, 'k', 32), (2, 2, 128, 128))])
def test_a_norm_that_overflows_leaves_a_vector_of_zeros(family, fmt, shape, huge):
    """q or k whose sum of squares is an infinity in fp32: divided by it, its finite entries are 0, in both kinds."""
    hv, hk, dk, dv = shape
    lay = _layout(family, fmt, shape, 8, 8)
    gen = torch.Generator().manual_seed(11)
    idx = torch.tensor([2, 1], dtype=torch.int32, device=DEV)
    blob = lay.alloc(3, DEV)
    lay.write(lay.views(blob), idx, torch.randn(2, hv, dv, dk, generator=gen).to(DEV))
    t = _token(family, gen, 2, shape)
    big = torch.randn(hk, dk, generator=gen).to(DEV) * 1e37
    big[0, 0] = 3e38
    t[huge][1] = big
    twin, outs = blob.clone(), []
    for group in (True, False):
        out = torch.full((2, hv, dv), 3.0, device=DEV)
        V = lay.views(blob if group else twin)
        _hip.select_instances(no_group_kernel=not group)
        try:
            _step(family, lay, V, idx, t, out, None)
        finally:
            _hip.select_instances()
        if huge == 'q':
            assert (out[1] == 0).all() and (out[0] != 0).any()
        else:
            assert (V['KB'][1, :, 0] == 0).all()                     # the key of the row's slot, as buffered
        outs.append(out)
    assert (outs[0] - outs[1]).abs().max() <= 1e-5 * outs[1].abs().max()
