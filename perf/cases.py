"""What the speed of this package is judged by: the calls a serving or generation program makes every token, and the
state hand-over around a prefill.

A case is one decode step of a stack of recurrent layers (``layers`` independent layer states, one launch each), or
one hand-over of a few sequences' states to and from a prefill for every layer of the stack.  All calls are made as a
program makes them: the slot layouts with a table of slot indices, the tokens' q / k / v as column ranges of one fused
buffer, the sequences at different points of their fold period, the dispatch order from 64 sequences on (what the
package's own serving forwards do), tokens in bf16.  Head shapes and formats are those of bench.py and of the serving
presets.
"""
import math

import torch

import statequant_amd as sq
from statequant_amd.kernels import KDASlotLayout, Mamba2SlotLayout, PackedGDNState, PackedKDAState, SlotLayout
from statequant_amd.kernels.gga import GGAPacked, GGAPlan, head_bytes

DEV = 'cuda'
LAYERS = 24
TOKENS = 8                     # different tokens that a state cycles through (layer L reads token (step + L) % TOKENS)
MAX_BYTES = 4.0e9              # a drawn case moves no more than the largest listed one

# family -> the head shapes drawn from: (value heads, key heads / groups, d_k / d_state, d_v / head_dim)
SHAPES = {
    'gdn': [(32, 16, 128, 128), (32, 16, 128, 128), (30, 30, 96, 192), (16, 16, 128, 128)],
    'kda': [(32, 32, 128, 128), (32, 32, 128, 128), (20, 20, 96, 96)],
    'mamba2': [(128, 8, 128, 64), (112, 8, 128, 64), (96, 8, 128, 80)],
}
# formats drawn from: the serving presets int8k, int4k, int4v, int8v and bf16, and the other groups of bench.py
FORMATS = ['int8k32', 'int8k32', 'int8k128', 'int4k64', 'int4k64', 'int4k32', 'int4v32', 'int8v32', 'bf16']


def _case(name, kind, family, fmt, shape, rows, gate=False, buffer_bits=8, m=8, layers=LAYERS):
    hv, hk, dk, dv = shape
    return dict(name=name, kind=kind, family=family, fmt=fmt, hv=hv, hk=hk, dk=dk, dv=dv, rows=rows, layers=layers,
                gate=gate, buffer_bits=buffer_bits, m=m)


def listed():
    qwen = (32, 16, 128, 128)
    return [
        # one sequence being generated: 24 launches of a few microseconds each
        _case('gdn-int8k-1', 'step', 'gdn', 'int8k32', qwen, 1, gate=True),
        # a small interactive batch, a count that divides nothing, the 4-bit preset
        _case('gdn-int4k-13', 'step', 'gdn', 'int4k64', qwen, 13, gate=True),
        # the headline of the benchmark: a full serving batch, int8, one scale per state row
        _case('gdn-int8k-256', 'step', 'gdn', 'int8k128', qwen, 256),
        # the same batch in the 4-bit preset, the gate formed in the kernel
        _case('gdn-int4k-256', 'step', 'gdn', 'int4k64', qwen, 256, gate=True),
        # a medium ragged batch in the preset whose scales run along the value axis
        _case('gdn-int4v-100', 'step', 'gdn', 'int4v32', qwen, 100, gate=True),
        # heads that are no power of two wide
        _case('gdn-96x192-int4k-64', 'step', 'gdn', 'int4k64', (30, 30, 96, 192), 64, gate=True),
        # the unquantized state, which every deployment starts from
        _case('gdn-bf16-40', 'step', 'gdn', 'bf16', qwen, 40, gate=True),
        # decays per key channel
        _case('kda-int4k-128', 'step', 'kda', 'int4k32', (32, 32, 128, 128), 128),
        # state-space layers at their serving batch
        _case('mamba2-int8k-128', 'step', 'mamba2', 'int8k128', (128, 8, 128, 64), 128),
        # the mixed-width slot, whose heads are re-fitted at every token
        _case('gga-32', 'gga', 'gdn', 'mixed', qwen, 32, gate=True),
        # six sequences between two chunks of their prefill: states read, and the new ones written
        _case('handover-int8k-6', 'handover', 'gdn', 'int8k32', qwen, 6),
        # generation without a serving engine: a batch of equal lengths in lockstep
        _case('lockstep-kda-int8k-9', 'lockstep', 'kda', 'int8k32', (32, 32, 128, 128), 9, layers=6),
    ]


def draw(rng):
    """A case of the same ranges: any family, format and head shape, 1 to 256 sequences (mixed-width slots to 32,
    hand-overs to 12), now and then the bf16 decode buffer."""
    kind = rng.choices(['step', 'gga', 'handover', 'lockstep'], [14, 2, 2, 2])[0]
    family = 'gdn' if kind == 'gga' else rng.choices(['gdn', 'kda', 'mamba2'], [2, 1, 1])[0]
    if kind == 'lockstep':
        family = rng.choice(['gdn', 'kda'])
    shape = rng.choice(SHAPES[family])
    fmt = rng.choice(FORMATS)
    if kind == 'gga':
        shape, fmt = (32, 16, 128, 128), 'mixed'
    if fmt in ('int4v32', 'int8v32') and shape[3] % 32:
        fmt = fmt[:4] + 'k32'
    if fmt == 'int4k64' and shape[2] % 64 and family != 'gdn':
        fmt = 'int4k32'
    if fmt == 'int8k128' and shape[2] % 128 and family != 'gdn':
        fmt = 'int8k32'
    top = {'step': 256, 'gga': 32, 'handover': 12, 'lockstep': 64}[kind]
    rows = int(round(math.exp(rng.uniform(0.0, math.log(top)))))
    c = _case('', kind, family, fmt, shape, rows, gate=family == 'gdn' and kind in ('step', 'gga') and rng.random() < 0.7,
              buffer_bits=16 if kind in ('step', 'lockstep') and rng.random() < 0.1 else 8,
              layers=6 if kind == 'lockstep' else LAYERS)
    del c['name']
    while c['rows'] > 1 and work(c)['bytes'] > MAX_BYTES:
        c['rows'] -= 1
    return c


# ------------------------------------------------------------------------------------------------------------------
def _format(c):
    f = c['fmt']
    return f if f == 'bf16' else sq.Quantizer(int(f[3]), f[4], int(f[5:]))


def _gga_plan(c):
    """Mean width 4 bits with one fp16 pivot per layer, shuffled per layer: part of the model, the same for all seeds."""
    gen = torch.Generator().manual_seed(0)
    base = torch.tensor(([2] * 12 + [4] * 11 + [6] * 6 + [8] * 2 + [16]) * (-(-c['hv'] // 32)))[:c['hv']]
    return GGAPlan({L: (base[torch.randperm(c['hv'], generator=gen)], torch.rand(c['hv'], c['dk'], generator=gen) + 0.5)
                    for L in range(c['layers'])})


def _layout(c):
    if c['kind'] == 'gga':
        return GGAPacked(_gga_plan(c), c['hv'], c['hk'], c['dk'], c['dv'], pw=True, m=c['m'])
    kw = dict(m=c['m'], buffer_bits=c['buffer_bits'])
    if c['family'] == 'kda':
        return KDASlotLayout(_format(c), c['hv'], c['dk'], c['dv'], **kw)
    cls = SlotLayout if c['family'] == 'gdn' else Mamba2SlotLayout
    return cls(_format(c), c['hv'], c['hk'], c['dk'], c['dv'], **kw)


def _randn(gen, *shape):
    return torch.randn(*shape, device=DEV, generator=gen)


def _tokens(c, gen):
    """What the layers in front of the step hand over for one token of every sequence, TOKENS times."""
    rows, hv, hk, dk, dv = (c[k] for k in ('rows', 'hv', 'hk', 'dk', 'dv'))
    softplus = torch.nn.functional.softplus
    out = []
    for _ in range(TOKENS):
        if c['family'] == 'mamba2':
            x = _randn(gen, rows, hv * dv + 2 * hk * dk).bfloat16()              # x | B | C of one conv output
            out.append(dict(x=x[:, :hv * dv].unflatten(1, (hv, dv)), B=x[:, hv * dv:-hk * dk].unflatten(1, (hk, dk)),
                            C=x[:, -hk * dk:].unflatten(1, (hk, dk)), dt=(_randn(gen, rows, hv) * 0.5 - 2).bfloat16()))
            continue
        if c['kind'] == 'lockstep':
            t = dict(q=_randn(gen, rows * hk, dk).bfloat16(), k=_randn(gen, rows * hk, dk).bfloat16(),
                     v=_randn(gen, rows * hv, dv).bfloat16())
        elif c['family'] == 'kda':
            t = dict(q=_randn(gen, rows, hk, dk).bfloat16(), k=_randn(gen, rows, hk, dk).bfloat16(),
                     v=_randn(gen, rows, hv, dv).bfloat16())
        else:
            x = _randn(gen, rows, 2 * hk * dk + hv * dv).bfloat16()              # q | k | v of one conv output
            t = dict(q=x[:, :hk * dk].unflatten(1, (hk, dk)), k=x[:, hk * dk:2 * hk * dk].unflatten(1, (hk, dk)),
                     v=x[:, 2 * hk * dk:].unflatten(1, (hv, dv)))
        if c['family'] == 'kda':
            t.update(g=-softplus(_randn(gen, rows, hv, dk) - 1.0), beta=torch.sigmoid(_randn(gen, rows, hv)))
        elif c['gate']:
            t.update(a=_randn(gen, rows, hv).bfloat16(), b=_randn(gen, rows, hv).bfloat16())
        else:
            t.update(g=-softplus(_randn(gen, rows, hv) - 1.0), beta=torch.sigmoid(_randn(gen, rows, hv)))
        if c['kind'] == 'lockstep' and c['family'] == 'gdn':
            t.update(g=t['g'].reshape(-1), beta=t['beta'].reshape(-1))
        out.append(t)
    return out


def _rounded(x, dtype, scale):
    """x in the decode buffer's type: int8 against an fp16 scale per vector (stored in ``scale``), or bf16."""
    if dtype != torch.int8:
        return x.to(dtype)
    s = (x.abs().amax(-1) / 127.0).half()
    scale.copy_(s.reshape(scale.shape))
    return torch.round(x / s.float().unsqueeze(-1)).clamp_(-127, 127).to(torch.int8)


def _fill_buffer(c, F, at, n, gen):
    """Decode buffers in mid-period: the entries at ``at`` of the fields F hold keys, values and decays of the last
    tokens, ``n`` (one per sequence) of them live."""
    rows, hv, hk, dk, dv, m = (c[k] for k in ('rows', 'hv', 'hk', 'dk', 'dv', 'm'))
    key = _randn(gen, rows, hk, m, dk)
    if c['family'] != 'mamba2':
        key = torch.nn.functional.normalize(key, dim=-1)
    val = _randn(gen, rows, hv, m, dv) * (0.1 if c['family'] == 'mamba2' else 0.5)
    per_channel = (dk,) if c['family'] == 'kda' else ()
    decay = (-torch.nn.functional.softplus(_randn(gen, rows, hv, m, *per_channel) - 1.0)).cumsum(2)
    now = decay[torch.arange(rows, device=DEV), :, (n - 1).clamp(min=0)]          # the decay up to the last live token
    now[n == 0] = 0.0
    for x, name in ((key, 'KB'), (val, 'UB')):
        scale = torch.empty(x.shape[:-1], dtype=torch.float16, device=DEV)
        F[name][at] = _rounded(x, F[name].dtype, scale).view(rows, *F[name].shape[1:])
        if F[name].dtype == torch.int8:
            F[name + 'S'][at] = scale.view(rows, *F[name + 'S'].shape[1:])
    F['GB'][at] = decay.view(rows, *F['GB'].shape[1:])
    F['GCUR'][at] = now.reshape(rows, *F['GCUR'].shape[1:])
    F['NPTR'][at] = n.to(torch.int32).view(rows, 1).expand(rows, F['NPTR'].shape[1])


def _fill_windows(c, lay, blob, at, gen):
    """Full FP8 windows (every sequence of more than m tokens has one), their oldest entry anywhere in the ring."""
    rows, hv, m, dk, dv = (c[k] for k in ('rows', 'hv', 'm', 'dk', 'dv'))
    win = torch.empty(rows, hv, lay.QSZ, dtype=torch.uint8, device=DEV)
    scales = torch.empty(rows, hv, 2, m, device=DEV)
    for i, (lo, d, size) in enumerate(((0, dk, 0.05), (m * dk, dv, 1.0))):
        x = _randn(gen, rows, hv, m, d) * size
        s = x.abs().amax(-1) / 448.0
        scales[:, :, i] = s
        win[:, :, lo:lo + m * d] = (x / s.unsqueeze(-1)).to(torch.float8_e4m3fn).view(torch.uint8).flatten(2)
    win[:, :, m * (dk + dv):] = scales.flatten(2).view(torch.uint8)
    blob[at, lay.QOFF:lay.QOFF + hv * lay.QSZ] = win.flatten(1)
    count = torch.full((rows, 2), m, dtype=torch.int32, device=DEV)
    count[:, 1] = torch.randint(m, (rows,), generator=gen, device=DEV)
    blob[at, :8] = count.view(torch.uint8)


def _lockstep(c, gen):
    """Layer states that a program filled from a prefill and stepped for a part of a fold period."""
    rows, hv, hk, dk, dv = (c[k] for k in ('rows', 'hv', 'hk', 'dk', 'dv'))
    states = []
    for L in range(c['layers']):
        kw = dict(m=c['m'], hv=hv, buffer_bits=c['buffer_bits'])
        if c['family'] == 'kda':
            st = PackedKDAState(_randn(gen, rows, hv, dv, dk) * 0.3, _format(c), **kw)
        else:
            st = PackedGDNState(_randn(gen, rows, hv, dk, dv) * 0.3, _format(c), hk=hk, **kw)
        F = {k: t.view(rows, -1, *t.shape[1:]) if k != 'NPTR' else t for k, t in st.T.items() if k not in ('S', 'SC')}
        n = torch.full((rows,), c['m'] - 1, device=DEV)                            # all fold on the coming token
        _fill_buffer(c, F, torch.arange(rows, device=DEV), n, gen)
        states.append(st)
    return states


def prepare(case, seed):
    c = dict(case)
    gen = torch.Generator(device=DEV).manual_seed(seed)
    st = dict(c=c, t=0, tokens=_tokens(c, gen))
    rows, hv, hk, dk, dv, layers = (c[k] for k in ('rows', 'hv', 'hk', 'dk', 'dv', 'layers'))
    if c['family'] == 'mamba2':
        st['model'] = (-torch.exp(torch.rand(hv, device=DEV, generator=gen) * 2), _randn(gen, hv), _randn(gen, hv) * 0.1)
    else:
        st['model'] = (_randn(gen, hv) * 0.3, _randn(gen, hv) * 0.3)             # A_log, dt_bias of the gate
    st['out'] = torch.zeros(layers, rows, hv, dv, dtype=torch.bfloat16, device=DEV)
    if c['kind'] == 'lockstep':
        st['states'] = _lockstep(c, gen)
        return st
    lay = st['lay'] = _layout(c)
    slots = rows + 1 + rows // 4                                                 # slot 0 is nobody's; some are free
    st['idx'] = idx = (torch.randperm(slots - 1, device=DEV, generator=gen)[:rows] + 1).to(torch.int32)
    blob = st['blob'] = lay.alloc(layers * slots, DEV)
    st['views'] = [lay.views(blob[L * slots:(L + 1) * slots]) for L in range(layers)]
    n = torch.randint(c['m'], (rows,), generator=gen, device=DEV)                # the same fill in every layer
    at = idx.long()
    for L in range(layers):
        S = _randn(gen, rows, hv, dv, dk) * 0.3
        kw = dict(layer=L) if c['kind'] == 'gga' else {}
        lay.write(st['views'][L], idx, S, **kw)
        if c['kind'] == 'gga':
            _fill_windows(c, lay, blob[L * slots:(L + 1) * slots], at, gen)
        else:
            _fill_buffer(c, st['views'][L], at, n, gen)
    if c['kind'] == 'gga':
        lay.prepare(DEV)
    if c['kind'] == 'handover':
        st['final'] = [_randn(gen, rows, hv, dv, dk) * 0.3 for _ in range(4)]    # a prefill's final states
    return st


def run(st):
    c, T = st['c'], st['tokens']
    t0 = st['t']
    st['t'] = (t0 + 1) % TOKENS
    scale = c['dk'] ** -0.5
    if c['kind'] == 'lockstep':
        out = []
        for L, S in enumerate(st['states']):
            t = T[(t0 + L) % TOKENS]
            out.append(S.step(t['q'], t['k'], t['v'], t['g'], t['beta'], scale))
        return dict(out=out, state=[[S.T[k] for k in sorted(S.T)] for S in st['states']])
    lay, idx, views, out = st['lay'], st['idx'], st['views'], st['out']
    if c['kind'] == 'handover':
        init = []
        for L, V in enumerate(views):
            init.append(lay.read(V, idx))
            lay.write(V, idx, st['final'][(t0 + L) % 4])
        return dict(init=init, state=_fields(lay, st['blob']))
    A_log, dt_bias = st['model'][:2]
    if c['kind'] == 'gga':
        for L, V in enumerate(views):
            t = T[(t0 + L) % TOKENS]
            gate = dict(gate=(t['a'], t['b'], A_log, dt_bias)) if c['gate'] else dict(g=t['g'], beta=t['beta'])
            lay.step(V, idx, t['q'], t['k'], t['v'], out[L], scale, layer=L, **gate)
        return dict(out=out, state=st['blob'])
    order = lay.fold_order(views[0], idx) if c['rows'] >= 64 and c['rows'] % 8 == 0 else None
    for L, V in enumerate(views):
        t = T[(t0 + L) % TOKENS]
        if c['family'] == 'mamba2':
            A, D, bias = st['model']
            lay.step(V, idx, t['x'], t['dt'], t['B'], t['C'], out[L], A, D, bias, dt_softplus=True, order=order)
        elif c['family'] == 'kda':
            lay.step(V, idx, t['q'], t['k'], t['v'], t['g'], t['beta'], out[L], scale, order=order)
        else:
            gate = dict(gate=(t['a'], t['b'], A_log, dt_bias)) if c['gate'] else dict(g=t['g'], beta=t['beta'])
            lay.step(V, idx, t['q'], t['k'], t['v'], out[L], scale, order=order, **gate)
    return dict(out=out, state=_fields(lay, st['blob']))


def _fields(lay, blob):
    """The updated state, field by field, of all layers' slots."""
    V = lay.views(blob)
    return [V[k] for k in sorted(V)]


# ------------------------------------------------------------------------------------------------------------------
def _stored(c):
    """Bytes of one sequence's stored state in one layer (codes and scales)."""
    hv, dk, dv = c['hv'], c['dk'], c['dv']
    if c['fmt'] == 'bf16':
        return hv * dk * dv * 2
    f = _format(c)
    return hv * dk * dv * f.bits // 8 + hv * 2 * (dv * -(-dk // f.group) if f.axis == 'k' else dv // f.group * dk)


def work(case):
    """State read whole and, one step in m, written back; the live half of the decode buffer; the append; the token's
    inputs and output.  Mixed-width slots: every head read and written, the window read, its left factors written.
    A hand-over: stored state and buffer read, fp32 states out and in, codes written."""
    c = dict(case)
    rows, hv, hk, dk, dv, m, layers = (c[k] for k in ('rows', 'hv', 'hk', 'dk', 'dv', 'm', 'layers'))
    token = 2 * hk * dk * 2 + 2 * hv * dv * 2 + hv * 4 * (dk if c['family'] == 'kda' else 2)
    values = hv * dk * dv
    if c['kind'] == 'gga':
        widths = [2] * 12 + [4] * 11 + [6] * 6 + [8] * 2 + [16]
        state = 2 * sum(head_bytes(w, dk, dv) for w in widths)
        coded = sum(w != 16 for w in widths)
        state += coded * (m * (dk + dv + 8) + m * (dk + 4) + dk + dv + 8)
        return dict(bytes=float(rows * layers * (state + token)), flops=float(rows * layers * values * 24))
    be = c['buffer_bits'] // 8
    entry = (hv * dv + hk * dk) * be + (hv + hk) * 2 * (be == 1) + hv * 4 * (dk if c['family'] == 'kda' else 1)
    live = entry * (m - 1) / 2
    stored = _stored(c)
    if c['kind'] == 'handover':
        return dict(bytes=float(rows * layers * (2 * stored + live + 2 * values * 4)),
                    flops=float(rows * layers * values * (m + 4)))
    return dict(bytes=float(rows * layers * (stored * (1 + 1 / m) + live + entry + token)),
                flops=float(rows * layers * values * 6))


def tolerance(case):
    """Outputs are bf16 of fp32 sums whose order is free (measured on two kernels that sum differently: rel 2.4e-5,
    max 0.02); a stored code or a buffered int8 value moves by one step where the value rounded lies within the sums'
    error of a rounding boundary (1e-6 of them), and a vector whose fp16 scale falls on the other side of one re-rounds
    all its entries (one vector of the smallest case is 1.6e-4 of its entries).  Mixed-width slots are handed back as
    bytes, the low bytes of fp32 scales among them (0.3 % of a slot), and an FP8 tie moves a head's output by 2e-3."""
    if case['kind'] == 'handover':
        return {'rel': 1e-5, 'max': 1e-3, 'differ': 0.0}
    if case['kind'] == 'gga':
        return {'rel': 5e-4, 'max': 0.05, 'differ': 2e-3}
    return {'rel': 2e-4, 'max': 0.05, 'differ': 2e-4}
