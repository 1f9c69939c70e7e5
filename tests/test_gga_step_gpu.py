"""The mixed-width step's one launch: the slot's counters, which its last head advances, and the instances with the serving
case's types compiled in against the general one."""
import pytest
import torch

from statequant_amd.kernels.gga import GGAPacked, GGAPlan

pytestmark = pytest.mark.gpu
DEV = 'cuda'


def _case(hv, hk, d, m, rows, seed=0, pw=True):
    gen = torch.Generator().manual_seed(seed)
    widths = torch.tensor(([2, 4, 6, 8, 16] * hv)[:hv])
    lay = GGAPacked(GGAPlan({0: (widths, torch.rand(hv, d, generator=gen) + 0.5)}), hv, hk, d, d, pw=pw, m=m)
    views = lay.views(lay.alloc(rows + 3, DEV))
    idx = (torch.randperm(rows + 2, generator=gen)[:rows] + 1).to(torch.int32).to(DEV)
    lay.write(views, idx, (torch.randn(rows, hv, d, d, generator=gen) * 0.3).to(DEV), layer=0)
    return lay.prepare(DEV), views, idx, gen


def _token(gen, rows, hv, hk, d):
    r = lambda *s: torch.randn(*s, generator=gen).bfloat16().to(DEV)         # noqa: E731
    return r(rows, hk, d), r(rows, hk, d), r(rows, hv, d), r(rows, hv), r(rows, hv)


@pytest.mark.parametrize('hv, hk, d, m, rows', [(1, 1, 64, 1, 1), (3, 3, 64, 8, 5), (5, 5, 128, 3, 2), (32, 16, 64, 8, 40)])
def test_counters_advance_once_a_step(hv, hk, d, m, rows):
    lay, views, idx, gen = _case(hv, hk, d, m, rows)
    blob = views['blob']
    blob[:, 8:16] = 0xA5                                                     # not the step's to write
    idx[rows // 2] = 0 if rows > 1 else idx[0]                               # padding
    live = idx[idx > 0].long()
    A, bias = torch.randn(hv, generator=gen).to(DEV) * 0.3, torch.randn(hv, generator=gen).to(DEV) * 0.3
    out = torch.zeros(rows, hv, d, dtype=torch.bfloat16, device=DEV)
    want = torch.zeros(blob.shape[0], 2, dtype=torch.int32)
    for t in range(2 * m + 3):
        q, k, v, a, b = _token(gen, rows, hv, hk, d)
        lay.step(views, idx, q, k, v, out, d ** -0.5, gate=(a, b, A, bias), layer=0)
        for s in live.tolist():
            n, head = want[s].tolist()
            want[s] = torch.tensor([min(n + 1, m), (head + 1) % m if n == m else head])
        assert torch.equal(blob[:, :8].cpu().view(torch.int32), want), t
        assert (blob[:, 8:16] == 0xA5).all()


@pytest.mark.parametrize('hv, hk, rows, twice', [(1, 1, 2, [(0, 1)]), (5, 5, 6, [(0, 2), (1, 4), (1, 5)]),
                                                 (32, 16, 40, [(3, 39)]), (3, 3, 130, [(0, 64), (0, 129), (70, 71)])])
def test_a_slot_named_twice_advances_once_and_leaves_nothing_behind(hv, hk, rows, twice):
    """What such a launch leaves of the state is in no order; the slot's counters move on by one token, and the steps after
    it, which name every slot once, find them as they should be."""
    lay, views, idx, gen = _case(hv, hk, 64, 3, rows)
    blob = views['blob']
    doubled = idx.clone()
    for a, b in twice:
        doubled[b] = idx[a]
    A, bias = torch.randn(hv, generator=gen).to(DEV) * 0.3, torch.randn(hv, generator=gen).to(DEV) * 0.3
    out = torch.zeros(rows, hv, 64, dtype=torch.bfloat16, device=DEV)
    want = torch.zeros(blob.shape[0], 2, dtype=torch.int32)
    for t in range(9):
        rows_now = doubled if t in (0, 1, 4) else idx
        q, k, v, a, b = _token(gen, rows, hv, hk, 64)
        lay.step(views, rows_now, q, k, v, out, 0.125, gate=(a, b, A, bias), layer=0)
        for s in set(rows_now.tolist()):
            n, head = want[s].tolist()
            want[s] = torch.tensor([min(n + 1, 3), (head + 1) % 3 if n == 3 else head])
        assert torch.equal(blob[:, :8].cpu().view(torch.int32), want), t


def test_more_heads_than_a_launch_dimension_takes():
    """65 601 heads of one slot: those on either side of the launch's dimensions step like the same heads in a small slot."""
    hv, d, picked = 65601, 64, [0, 32767, 32768, 65535, 65536, 65600]
    gen = torch.Generator(device=DEV).manual_seed(4)
    w = torch.rand(hv, d, device=DEV, generator=gen).cpu() + 0.5
    widths = torch.full((hv,), 2)
    widths[picked] = torch.tensor([4, 2, 8, 6, 2, 16])
    S = torch.randn(1, hv, d, d, device=DEV, generator=gen) * 0.3
    r = lambda *s: torch.randn(*s, device=DEV, generator=gen).bfloat16()         # noqa: E731
    tokens = [(r(1, 1, d), r(1, 1, d), r(1, hv, d), r(1, hv), r(1, hv)) for _ in range(4)]
    A, bias = torch.randn(hv, device=DEV, generator=gen) * 0.3, torch.randn(hv, device=DEV, generator=gen) * 0.3
    idx = torch.ones(1, dtype=torch.int32, device=DEV)

    def outputs(sel):
        lay = GGAPacked(GGAPlan({0: (widths[sel], w[sel])}), len(sel), 1, d, d, pw=True, m=3)
        views = lay.views(lay.alloc(2, DEV))
        lay.write(views, idx, S[:, sel], layer=0)
        outs = []
        for q, k, v, a, b in tokens:
            o = torch.zeros(1, len(sel), d, dtype=torch.bfloat16, device=DEV)
            outs.append(lay.step(views, idx, q, k, v[:, sel].contiguous(), o, 0.125, layer=0,
                                 gate=(a[:, sel].contiguous(), b[:, sel].contiguous(), A[sel], bias[sel])))
        return torch.stack(outs), views['blob'][1, :8].view(torch.int32).tolist()

    many, counters = outputs(list(range(hv)))
    few, want = outputs(picked)
    assert counters == want == [3, 1]
    assert torch.equal(many[:, :, picked], few)


@pytest.mark.parametrize('gate', [True, False])
@pytest.mark.parametrize('hv, hk, d, pw', [(5, 5, 64, True), (8, 4, 128, True), (6, 2, 128, False)])
def test_serving_instances_equal_the_general_one(gate, hv, hk, d, pw):
    rows = 3
    lay, views, idx, gen = _case(hv, hk, d, 8, rows, pw=pw)
    twin = lay.views(views['blob'].clone())
    A, bias = torch.randn(hv, generator=gen).to(DEV) * 0.3, torch.randn(hv, generator=gen).to(DEV) * 0.3
    o16 = torch.zeros(rows, hv, d, dtype=torch.bfloat16, device=DEV)
    o32 = torch.zeros(rows, hv, d, device=DEV)
    for t in range(11):
        q, k, v, a, b = _token(gen, rows, hv, hk, d)
        if gate:
            one, two = dict(gate=(a, b, A, bias)), dict(gate=(a.float(), b.float(), A, bias))
        else:
            g, beta = -torch.nn.functional.softplus(a.float()), torch.sigmoid(b.float())
            one = two = dict(g=g, beta=beta)
        lay.step(views, idx, q, k, v, o16, d ** -0.5, layer=0, **one)
        lay.step(twin, idx, q.float(), k.float(), v.float(), o32, d ** -0.5, layer=0, **two)      # fp32: the general instance
        assert torch.equal(o16, o32.bfloat16()), t
        assert torch.equal(views['blob'], twin['blob']), t
