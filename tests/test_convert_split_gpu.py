"""A hand-over of a few sequences splits every head's rows over several wavefronts; one of many does not.  Both give the
same bytes: rows, scales, counters and read-outs of a sequence written (read) alone against the same one among hundreds."""
import pytest
import torch

import statequant_amd as sq
from statequant_amd.kernels import KDASlotLayout, Mamba2SlotLayout, SlotLayout

pytestmark = pytest.mark.gpu
DEV = 'cuda'


@pytest.mark.parametrize('family,fmt,hv,dk,dv,few', [
    ('gdn', (8, 'k', 32), 32, 128, 128, 1), ('gdn', (4, 'k', 64), 30, 96, 192, 3), ('gdn', (4, 'v', 32), 4, 128, 256, 2),
    ('gdn', 'bf16', 4, 64, 64, 5), ('kda', (8, 'k', 32), 5, 64, 32, 1), ('kda', (4, 'v', 32), 4, 96, 96, 2),
    ('mamba2', (8, 'k', 32), 8, 96, 80, 3), ('mamba2', (4, 'k', 32), 8, 256, 64, 1), ('mamba2', (8, 'v', 16), 8, 128, 80, 2)])
def test_split_rows_give_the_same_bytes(family, fmt, hv, dk, dv, few):
    fmt = fmt if isinstance(fmt, str) else sq.Quantizer(*fmt)
    lay = KDASlotLayout(fmt, hv, dk, dv) if family == 'kda' else \
        {'gdn': SlotLayout, 'mamba2': Mamba2SlotLayout}[family](fmt, hv, hv // 2, dk, dv)
    many = 4096 // hv + 1                                            # from here on a head is one wavefront
    gen = torch.Generator(device=DEV).manual_seed(2)
    S = torch.randn(few, hv, dv, dk, device=DEV, generator=gen)
    S[:, 0, 1] = 0.0
    lots = S.repeat(-(-many // few), 1, 1, 1)[:many].contiguous()
    got = []
    for states in (S, lots):
        n = states.shape[0]
        blob = lay.alloc(n + 1, DEV)
        V = lay.views(blob)
        V['NPTR'].fill_(77)
        idx = torch.arange(1, n + 1, dtype=torch.int32, device=DEV)
        lay.write(V, idx, states)
        written = blob[1:few + 1].clone()
        # a half-full decode buffer, the same for every sequence
        fill = torch.Generator(device=DEV).manual_seed(3)
        for f in ('KB', 'UB'):
            V[f][:] = torch.randint(-127, 128, V[f].shape[1:], device=DEV, generator=fill).to(V[f].dtype)
            V[f + 'S'][:] = 0.01
        for f in ('GB', 'GCUR'):
            V[f][:] = -torch.rand(V[f].shape[1:], device=DEV, generator=fill)
        V['NPTR'].fill_(5)
        got.append((written, lay.read(V, idx)[:few]))
    assert torch.equal(got[0][0], got[1][0])
    assert torch.equal(got[0][1], got[1][1])
