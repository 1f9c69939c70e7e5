"""Build libsqhip.so (the C-ABI library of include/statequant_hip.h) for gfx950 with hipcc.

    python -m statequant_amd.csrc.build [-j N] [--force] [--timeline] [--resources [PATTERN]]

The step kernels are templates on (bits, d_k, d_v, group, int8-buffer, max m).  ``CASES`` below lists the instances
that are compiled; this script writes one small translation unit per chunk of instances plus the dispatch table into
``csrc/build/`` (not tracked), compiles them in parallel and links ``statequant_amd/libsqhip.so`` next to the Python
package, where the loader looks for it.  hipcc cross-compiles, so no GPU is needed to build.
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import hashlib
import itertools
import os
import re
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.dirname(HERE)
OUT = os.path.join(HERE, 'build')
LIB = os.path.join(PKG, 'libsqhip.so')
HOST = os.path.join(PKG, '_sqhost' + sysconfig.get_config_var('EXT_SUFFIX'))
ARCH = 'gfx950'

# -ffp-contract=off: every fused multiply-add in the kernels is written explicitly, as in the reference's kernels.
# The packed-fp32 target feature is switched off on purpose (plain v_fma / v_mul only).
HIPCC_FLAGS = ['--offload-arch=' + ARCH, '-O3', '-std=c++17', '-fPIC', '-ffp-contract=off',
               '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops', '-Wno-unused-command-line-argument',
               # scalar kernel arguments ahead of a parameter struct arrive in registers (no load at wave start)
               '-mllvm', '-amdgpu-kernarg-preload-count=16']

# Vectorized by the compiler, the comparisons over the mixed-width step's eight columns a lane (do two roundings agree, is a
# column certain) gather their results in lanes' bytes -- 390 16-bit shifts, 380 ors and as many selects more in the kernel --
# instead of or-ing masks in scalar registers: 15 000 -> 16 100 vector instructions.  us a layer, captured, with this flag /
# without: 32 sequences 27.6 / 30.8, 256 146.5 / 164.  (Registers do not decide it: 59 are spilled with it, 46 without.)
UNIT_FLAGS = {'inst_gga_': ['-fno-slp-vectorize']}


def _flags(src):
    base = os.path.basename(src)
    return HIPCC_FLAGS + [f for prefix, flags in UNIT_FLAGS.items() if base.startswith(prefix) for f in flags]


def _cases():
    """family -> [(bits, dk, dv, group, qbuf, mmax, axv)].  Shapes: Qwen3.5 GDN 128x128, small test heads 64x64,
    OLMo-Hybrid 96x192, a 96x96 head, 128x256 (the power-of-two problem that 96x192 pads to); Mamba2 d_state 128 /
    head_dim 64 (Nemotron-H), 128 x 128, 64 x 64, d_state 256 / head_dim 64 (Falcon-H1; key-axis groups and bf16 only), d_state 128 / head_dim 80 (Nemotron-3-Nano) and 96 / 80 (the
    reference tests' odd head);
    KDA 128x128, 96x96, 64x64, 128x256 and 64x32 (the reference tests' wide and small heads).  Key-axis groups: every power of two from 32 up to the padded d_k."""
    shapes = {
        'gdn': [(128, 128), (64, 64), (96, 192), (96, 96), (128, 256)],
        'mamba2': [(128, 64), (128, 128), (64, 64), (128, 80), (96, 80), (256, 64)],
        'kda': [(128, 128), (96, 96), (64, 64), (128, 256), (64, 32)],
    }
    out = {}
    for fam, shp in shapes.items():
        rows = []
        for (dk, dv), bits, qbuf in itertools.product(shp, (8, 4), (1, 0)):
            dkp = 1 << (dk - 1).bit_length()
            for group in (32, 64, 128):
                if group > dkp:
                    continue
                rows.append((bits, dk, dv, group, qbuf, 8, 0))
                rows.append((bits, dk, dv, group, qbuf, 16, 0))      # a buffer of up to 16 tokens
            for mmax in (8, 16) if dk <= 128 else ():                # value-axis groups: d_k up to 128
                if dv % 32 == 0:
                    rows.append((bits, dk, dv, 32, qbuf, mmax, 1))   # value-axis groups of 32 rows
                if dv % 64 == 0:
                    rows.append((bits, dk, dv, 64, qbuf, mmax, 1))   # ... of 64 rows
                if fam != 'gdn' or (dk, dv) in ((128, 128), (64, 64)):
                    rows.append((bits, dk, dv, 16, qbuf, mmax, 1))   # ... and of 16 (the reference's KDA / Mamba2 tests)
        for (dk, dv), qbuf in itertools.product(shp, (1, 0)):        # the unquantized control: bf16 (GDN also fp32) state
            for mmax in (8, 16):
                rows.append((16, dk, dv, dk, qbuf, mmax, 0))
                if fam == 'gdn':
                    rows.append((32, dk, dv, dk, qbuf, mmax, 0))
        out[fam] = rows
    return out


CASES = _cases()
GGA_SHAPES = [(128, 128), (64, 64)]                  # (d_k, d_v) of the mixed-width GGA / STEP slot (sq_gga.cuh)
PARAMS = {'gdn': 'GdnParams', 'kda': 'KdaParams', 'mamba2': 'Mamba2Params'}
# families with a workgroup-per-key-head kernel (sq_<family>_quad.cuh) -> value heads per workgroup that are built
QUAD_FAMILIES = {'gdn': (2, 1), 'mamba2': (4, 2, 1), 'kda': (1,)}
# compile-time specialisations of the step kernels (SPEC, sq_params.h), most specific first; 0: everything read from
# the arguments.  Built for the default buffer (int8, 8 tokens) only.
SPECS = {'gdn': (1, 2, 0), 'kda': (1, 0), 'mamba2': (1, 2, 0)}


def specs_of(fam, c, quad):
    """SPEC values an instance is built for: the workgroup-per-key-head kernels for every case they serve, the
    one-wavefront kernels for the cases that have no such kernel."""
    bits, dk, dv, group, qbuf, mmax, axv = c
    if not (qbuf and mmax == 8) or (not quad and quad_variants(fam, c) and not (fam == 'kda' and dk == 64)):
        return (0,)                                          # (KDA, d_k 64: the one-wavefront kernel serves launches of many heads)
    if not quad and fam != 'kda':
        # measured on the one-wavefront kernels: KDA int4 g32 40.0 -> 38.9 us, GDN value-axis int4 36.3 -> 35.1, but
        # value-axis int8 45.2 -> 48.4 and Mamba2 d_state 256 41.9 -> 48.1 (their register allocation tips over)
        return (0,)
    return SPECS[fam]
CHUNK = 6                                            # instances per translation unit


def _tile(c):
    bits, dk, dv, group, qbuf, mmax, axv = c
    return (f'Tile<{bits}, {dk}, {dv}, {group}, {"true" if qbuf else "false"}, {mmax}'
            + (', true>' if axv else '>'))


# Run-time conditions of the workgroup kernels, per family (part of the generated dispatch unit): vectors and rows of codes
# that 16-byte accesses can address.  (The C ABI asks int4 states for 8-byte alignment only: those that have no more go to
# the one-wavefront kernels, which read 8 bytes a lane.)
QUAD_OK = [
    'static bool rows16(const void* ptr, uint32_t stride, int dt) {',
    '    return reinterpret_cast<uintptr_t>(ptr) % 16 == 0 && (uint64_t(stride) * (dt == 0 ? 4 : 2)) % 16 == 0;',
    '}',
    'static bool codes16(const StatePtrs& st) { return reinterpret_cast<uintptr_t>(st.S) % 16 == 0 && st.sS % 16 == 0; }',
    '// q, k per key head (or ungrouped keys)',
    'static bool gdn_quad_ok(const GdnParams& p) {',
    '    return (p.qk_per_key_head || p.gqa == 1) && codes16(p.st) && rows16(p.q, p.s_q, p.q_dt) && rows16(p.k, p.s_k, p.k_dt);',
    '}',
    'static bool mamba2_quad_ok(const Mamba2Params& p) {',
    '    return codes16(p.st) && rows16(p.B, p.s_B, p.B_dt) && rows16(p.C, p.s_C, p.C_dt);',
    '}',
    'static bool kda_quad_ok(const KdaParams& p) {',
    '    return codes16(p.st) && rows16(p.q, p.s_q, p.q_dt) && rows16(p.k, p.s_k, p.k_dt) && rows16(p.g, p.s_g, p.g_dt);',
    '}']


def quad_variants(fam, c):
    """[(row blocks per wavefront, value heads per workgroup, wavefronts per SIMD the register allocation aims for,
    serving case, condition on the launch -- '': any)], small launches' first, then widest head group first, of the
    workgroup kernels (sq_quad.cuh) for a case; empty where only the one-wavefront kernels (sq_tile.cuh) serve it:
    value-axis groups other than 32 rows, the fp32 state, d_v that is no multiple of 32 (Mamba2: 16), d_k above 128, more
    than four scale groups per row, states beyond 64 KB."""
    bits, dk, dv, group, qbuf, mmax, axv = c
    if fam not in QUAD_FAMILIES or bits not in (4, 8, 16) or (axv and group != 32):
        return []
    flt = bits == 16
    dkp = 1 << (dk - 1).bit_length()
    rb = 1 << (dk * bits // 8 - 1).bit_length()              # LDS row: the next power of two
    if (dk * bits // 8) % 16 or not 32 <= rb <= 256 or dk > 128 or dv % 32 and (fam != 'mamba2' or dv % 16 or axv):
        return []
    if not axv and not flt and -(-dk // group) > 4:
        return []
    if fam == 'gdn' and (dk, dv, bits, axv) == (64, 64, 8, 1) and mmax > 8:      # (32 heads, workgroup / one wavefront) 16
        return []                                        # sequences 9.7 / 8.8 us per launch, 100: 15.2 / 14.6, 250: 23.7 / 23.4
    nrb = -(-dv // 32)                                       # the last one may be half empty (Mamba2)
    # row blocks per wavefront: one for the bf16 state, whose blocks are 8 KB each (a head of 128 x 128 on two wavefronts
    # leaves eight per compute unit)
    nb = 2 if nrb % 2 == 0 and fam != 'kda' and not flt else 1
    be = 1 if qbuf else 2
    out = []
    for gh in QUAD_FAMILIES[fam]:
        if dv % 32 and gh > 1:                               # d_v 80: a head a workgroup (96 heads, int8 g32; us per launch
            continue                                         # with one, two, four: 1 sequence 5.6, 5.8, 6.4, 48: 24.8, 31.8, 25.5)
        nw = gh * nrb // nb
        if nw > 16:
            continue
        lds = gh * nrb * 32 * rb + mmax * dkp * be + gh * mmax * dv * be + 2 * dkp * 4 + (0 if flt else dkp * 8) + 512
        if fam == 'kda':                                 # keys x decay ratio in fp32 (the raw ones stay in registers), decays
            lds += mmax * dkp * 4 + 2 * dkp * 4 + (2 * dkp * 4 if axv or flt else 0)
        if axv:                                          # a plane set per wavefront
            lds += nw * dkp * 6 - dkp * 8
        if lds > (40 * 1024 if flt and gh > 1 else 63 * 1024):      # heads share a workgroup only while four of them fit
            continue
        wgs = min(160 * 1024 // lds, 32 // nw)
        if wgs < 1:
            continue
        # register target: as many wavefronts per SIMD as LDS lets workgroups in, up to 6 (5 with the 16-token buffer and
        # for value-axis groups, which spill 10 registers at 80); asked for 7, the int4 kernels spill into scratch
        # memory inside the fold (measured: +60 % bytes written)
        wpe = max(1, min(6 if mmax <= 8 and not axv else 5, -(-wgs * nw // 4)))
        # the serving cases compiled in (SPEC of the kernels) for the default buffer: int8, 8 tokens
        for spec in SPECS[fam] if (qbuf and mmax == 8) else (0,):
            out.append((nb, gh, wpe, spec, ''))
    if small_when(fam, c):                               # the one-head entries again, a row block per wavefront
        out = [(1, 1, 6 if not axv else 5, spec, small_when(fam, c)) for spec in SPECS[fam]] + out
    return out


# Where a line lies for launches without a dispatch order.  Such a launch is a batch out of step or one in lockstep, whose
# heads fold all on the same step: no head is a straggler then, and the variants that shorten a fold are worth less.  From 64
# sequences on a serving engine orders a batch that is out of step where its count allows it, so there the line is where a
# batch in lockstep begins to lose; below, it is where what a batch out of step gains is what one in lockstep loses (a lockstep
# state, which is one for sure, has no slot indices: `p.idx` null).
#
# Launches that satisfy this take one row block per wavefront and one head per workgroup: twice the wavefronts on up to
# four times the compute units, so that a head's life -- which is all such a launch consists of, the fold's four half
# blocks in sequence above all -- gets shorter.  (One block per wavefront with two heads per workgroup gains nothing:
# the wavefronts then share the SIMDs they had.)  us per launch, two blocks and two heads / this, 16 layers captured, sequences
# out of step; in lockstep (ls); in order:
# GDN 128 x 128 (32 heads on 16 key heads) int4 g64 60 sequences 13.3 / 12.8, 64: 13.0 / 12.8 (ls 9.2 / 10.3), 71: 14.1 / 14.0 (10.3
# / 11.1), in order 64: 11.6 / 11.2, 96: 15.1 / 14.3, 104: 15.1 / 15.0, 112: 15.6 / 15.8; int8 g32 60: 15.6 / 15.2, 64, one full
# round of pairs: 15.1 / 15.3 (11.7 / 12.5), 66: 15.9 / 15.9 (12.9 / 13.0), 72: 16.6 / 16.1 (13.4 / 13.5), 90: 19.3 / 18.7 (15.1 / 15.6; g128
# 14.7 / 15.1), in order 64: 13.7 / 13.3, 72: 14.2 / 14.4.  Value-axis int4 104: 20.7 / 19.3 (14.0 / 15.0), 108: 22.5 / 21.7 (15.3 /
# 16.8), 128: 22.7 / 22.0 (16.2 / 17.9), 190: 28.7 / 29.1, in order 104: 16.2 / 15.9, 128: 17.7 / 17.9, 136: 19.0 / 19.3; int8 190:
# 33.6 / 31.5 (26.8 / 27.2), 200: 34.9 / 33.1 (28.2 / 28.1), 250: 40.7 / 39.4 (34.0 / 35.1), in order 120: 19.9 / 19.7, 128: 20.4 /
# 21.4.  Ungrouped heads (16 on 16), where the other side has one head a workgroup too, int4 128: 15.1 / 13.4 (10.2 / 10.5), 140:
# 16.1 / 14.1 (11.3 / 11.1), in order 208: 16.3 / 15.1; int8 136: 18.9 / 15.9 (14.5 / 13.2), 190: 22.5 / 19.7; value-axis int4 250:
# 25.4 / 21.9 (17.5 / 17.6), int8 256: 28.8 / 24.2 (22.0 / 20.3).  48 on 16 int4 44: 15.7 / 15.0 (11.3 / 12.7), int8 60: 22.7 /
# 20.6 (17.5 / 17.4).  96 x 192 int4 g64 (30 heads) 25: 11.4 / 11.0 (7.9 / 8.1), 26: 11.8 / 11.9, 40: 13.1 / 16.4, in order 64: 14.2 /
# 17.7, 128: 21.5 / 31.9; int8 g128 40: 14.2 / 17.0, in order 64: 16.2 / 18.6.  Mamba2 128 x 64 (128 heads) int8 g128 8: 7.7 / 7.5 (5.6
# / 5.8), 10: 9.4 / 8.7 (6.7 / 6.5), 12: 9.0 / 9.0 (6.8 / 7.1), 13: 9.8 / 9.7 (7.0 / 7.3); int4 g64 10: 8.9 / 8.1 (6.0 / 6.0), 14: 9.2 /
# 9.2 (6.2 / 6.8), 18: 10.5 / 10.1 (7.2 / 7.6); 112 heads 14: 9.9 / 9.2 (6.4 / 6.9).  The other shapes and buffers that have two
# blocks or several heads in a workgroup were not built this way: nothing is known about them.
def small_when(fam, c):
    bits, dk, dv, group, qbuf, mmax, axv = c
    if bits == 16 or not qbuf or mmax > 8:
        return ''
    gdn4 = 'heads < (p.order ? 3456 : p.gqa == 1 ? 2304 : 2048)'
    gdn8 = '(p.order ? heads < 2176 : p.gqa == 1 ? heads < 3072 : heads < 2560 && heads != 2048)'
    gdn4v = 'heads < (p.order ? 4224 : p.gqa == 1 ? 6400 : 3328)'
    gdn8v = 'heads < (p.order ? 3968 : p.gqa == 1 ? 8192 : 6912)'
    return {('gdn', 128, 128, 0): gdn4 if bits == 4 else gdn8, ('gdn', 128, 128, 1): gdn4v if bits == 4 else gdn8v,
            ('gdn', 96, 192, 0): 'heads < 768',
            ('mamba2', 128, 64, 0): f'heads < (p.idx ? {2432 if bits == 4 else 1664} : 768)'}.get((fam, dk, dv, axv), '')


# Heads per launch from which the one-wavefront kernel serves these cases again where nothing below has a line of its own:
# the buffers of 16 tokens or bf16, int8 value-axis groups of 96 x 96, and launches without an order whose lockstep batches
# lose from about there on.  Their workgroups waste something -- lanes and LDS on the columns between 96 and 128, a half empty
# row block (d_v 80) -- which does not matter while a launch is short of wavefronts and may once it has several rounds of them.
GROUP_HEADS = 5120


def group_when(fam, c):
    """The condition (C++, on `heads` of the launch and whether it has a dispatch order) under which a case's workgroup
    kernels serve; '' always.  What ends their lead is a launch with enough heads to fill the chip several times over:
    then a head costs its instructions and its LDS, not its length.  A dispatch order ends it earlier: the one-wavefront
    kernel's folding heads live three times as long as the others, and placed well they no longer decide when the launch
    ends.  Figures: us per launch, workgroup / one wavefront, sequences out of step (ls: in lockstep)."""
    bits, dk, dv, group, qbuf, mmax, axv = c
    flt, usual = bits == 16, qbuf and mmax == 8
    when = []
    if fam == 'mamba2':
        if dv % 32 and not flt:
            # a half empty row block.  128 x 80 (96 heads) int4 g64 52 sequences 22.3 / 24.7 (ls 17.6 / 17.3), 64: 24.8 / 27.7 (20.5 /
            # 19.2), 76: 27.2 / 29.4 (23.5 / 21.8), 80: 29.3 / 31.3 (24.4 / 22.1), 120: 39.8 / 39.9 (34.0 / 30.2), in order 64: 21.7 / 21.1;
            # int8 g128 52: 23.5 / 26.7 (18.8 / 19.3), 64: 26.2 / 29.5 (21.7 / 21.6), 128: 44.4 / 47.9 (38.3 / 36.9), 250: 78.5 / 82.3
            # (71.6 / 68.4), 400: 120.0 / 124.5 (112.0 / 107.4), in order 64: 23.0 / 23.7 (g32 128: 46.0 / 51.0, ls 40.5 / 39.3).
            # d_state 96, int4 34: 16.7 / 18.1 (13.2 / 12.8), 40: 18.7 / 18.7 (14.8 / 13.1), 64: 25.1 / 25.3 (20.9 / 18.3), in order 22.1 /
            # 19.7; int8 50: 22.1 / 24.0 (18.0 / 17.6), 72: 27.4 / 29.5 (23.9 / 22.0), 80: 30.5 / 31.8 (25.9 / 23.7), 150: 49.5 / 48.9, 250:
            # 75.9 / 70.9 (68.4 / 60.8), in order 64: 22.4 / 21.7
            line = {(4, 96): 3328, (8, 128): 6656 if usual and not axv else GROUP_HEADS}.get((bits, dk), GROUP_HEADS)
            when.append(f'heads < {line if mmax == 8 else GROUP_HEADS}')
        if flt and (dk, mmax) == (96, 8):                    # 64 sequences 33.7 / 34.3, 96 in order 47.3 / 43.1
            when.append('(!p.order || heads < 8192)')
    elif dk == 96 and not flt and (bits == 8 or not axv) and (fam == 'gdn' or (bits == 4 and not axv)):
        # a quarter of the lanes and of LDS on padded columns.  96 x 192 (30 heads) int4 g64 170 sequences 31.1 / 41.6 (ls 25.3 /
        # 27.5), 400: 60.1 / 69.5 (51.2 / 53.9), in order 256: 35.7 / 38.7, 400: 51.9 / 54.7; int8 g128 256: 48.8 / 58.6 (42.3 / 44.5), in
        # order 43.3 / 48.3, value-axis 50.1 / 67.0 (44.6 / 51.5), 44.8 / 53.2.  96 x 96 (20 heads) KDA int4 g32 200: 20.3 / 25.5 (17.1
        # / 18.0), 390: 30.7 / 37.6 (27.9 / 30.9), in order 256: 21.0 / 23.7, 400: 29.0 / 31.6; GDN, three wavefronts a head, int4 g64 160:
        # 18.0 / 20.1 (14.3 / 14.2), 256: 23.7 / 26.2 (19.9 / 18.6), 300: 26.6 / 28.5 (22.5 / 20.3), 400: 32.0 / 32.4 (28.1 / 24.5), in
        # order 160: 15.0 / 16.4, 192: 16.9 / 17.2, 256: 20.5 / 19.7; int8 g32 256: 24.8 / 28.6 (21.1 / 21.3), 400: 33.9 / 37.1 (30.1 /
        # 28.8), in order 256: 21.8 / 22.2, 400: 30.8 / 30.2
        if not usual or (axv and dv != 192):
            when.append(f'heads < {GROUP_HEADS}')
        elif fam == 'gdn' and dv == 192 and bits == 4:
            when.append('(!p.order || heads < 12288)')
        elif fam == 'gdn' and dv == 96:
            when.append(f'heads < (p.order ? 3680 : {GROUP_HEADS})' if bits == 4 else f'heads < (p.order ? {GROUP_HEADS} : 6400)')
        if fam == 'gdn' and dv == 96 and not axv and mmax == 8 and not qbuf:
            when.append('(!p.order || heads < 2880)')        # bf16 buffer 128: 14.7 / 15.2, 160: 17.0 / 16.0
    elif fam == 'gdn' and flt and (dk, dv) == (96, 192) and not usual:
        # two workgroups per compute unit (30 heads, 16-token buffer): 64 sequences in order 45.9 / 58.2, 96: 64.4 / 61.3,
        # 128: 80.6 / 64.8; 130, not in order, 81.3 / 87.5
        when.append('(!p.order || heads < 2560)')
    elif fam == 'kda' and dk == 64:
        # one or two wavefronts a head: little to deal out.  64 x 64 (32 heads) int4 g64 in order 128 sequences 9.6 / 10.8, 160:
        # 11.5 / 11.8, 256: 15.5 / 16.3, int8 g32 17.0 / 19.2; 16-token buffer int4 96: 11.6 / 12.2, 128: 13.5 / 12.8, int8 15.0 /
        # 13.7.  64 x 32 int4 g64 1 sequence 4.9 / 4.6, 8: 5.4 / 5.4, 16-token buffer 8: 6.2 / 6.2, 16: 6.9 / 7.1; bf16 state 100,
        # not in order, 11.1 / 11.7, 128 in order 11.7 / 11.1; 16-token bf16 buffer 64: 8.5 / 9.7, 130, not in order, int8 13.2 /
        # 13.1, value-axis 14.4 / 13.1
        if dv == 32 and not (flt and mmax > 8):
            when.append(f'heads >= {256 if mmax <= 8 else 384}')
        if not flt and mmax > 8:
            when.append('heads < 4096' if dv == 32 and not qbuf else '(!p.order || heads < 4096)')
        elif dv == 32 and mmax <= 8 and (flt or (bits == 8 and axv)):
            when.append('(!p.order || heads < 4096)')
        elif not flt and dv == 64 and (axv or not usual):
            when.append('(!p.order || heads < 5120)')
    elif fam == 'kda' and (dk, dv, bits, group, axv) == (128, 128, 8, 32, 0) and qbuf and mmax > 8:
        # 132 registers (32 heads): 96 sequences in order 27.4 / 29.4, 128: 34.5 / 32.7; 130, not in order, 37.7 / 44.8
        when.append('(!p.order || heads < 4096)')
    if axv and (dk, dv) == (64, 64) and fam != 'kda' and not usual:
        # one wavefront a head in both, and here the front end's barriers are what is left: GDN int8, bf16 buffer, 16
        # sequences 8.7 / 8.1, 64: 10.7 / 11.2; Mamba2 (64 heads) 8: 7.3 / 6.8, 16: 8.3 / 8.6
        when.append('heads >= 1024')
    return ' && '.join(when)


def _quad_name(fam, c, v):
    nb, gh, wpe, spec, _ = v
    return f'launch_{fam}_quad<{_tile(c)}, {nb}, {gh}, {wpe}, {spec}>'


def _write_if_changed(path, text):
    if os.path.exists(path) and open(path).read() == text:
        return
    with open(path, 'w') as f:
        f.write(text)


def generate():
    """Write the instance and dispatch translation units; returns their paths."""
    os.makedirs(OUT, exist_ok=True)
    units = []
    for fam, rows in CASES.items():
        insts = [(c, sp) for c in rows for sp in specs_of(fam, c, False)]
        for k in range(0, len(insts), CHUNK):
            body = ''.join(f'template int launch_{fam}<{_tile(c)}, {sp}>(const {PARAMS[fam]}&, hipStream_t);\n'
                           for c, sp in insts[k:k + CHUNK])
            path = os.path.join(OUT, f'inst_{fam}_{k // CHUNK:02d}.hip')
            _write_if_changed(path, f'// generated by build.py\n#include "../sq_{fam}.cuh"\nnamespace sq {{\n{body}}}\n')
            units.append(path)
    for fam, rows in CASES.items():
        qrows = [(c, v) for c in rows for v in quad_variants(fam, c)]
        for k in range(0, len(qrows), CHUNK):
            body = ''.join(f'template int {_quad_name(fam, c, v)}(const {PARAMS[fam]}&, hipStream_t);\n'
                           for c, v in qrows[k:k + CHUNK])
            path = os.path.join(OUT, f'inst_{fam}q_{k // CHUNK:02d}.hip')
            _write_if_changed(path, f'// generated by build.py\n#include "../sq_{fam}_quad.cuh"\nnamespace sq {{\n{body}}}\n')
            units.append(path)
    # pack / read: instances by (bits, d_k, group, value-axis[, buffer, per-channel decay]); d_v and m are run-time there
    rowfmt = sorted({(c[0], c[1], c[3], c[6]) for rows in CASES.values() for c in rows})
    kda_fmt = {(c[0], c[1], c[3], c[6]) for c in CASES['kda']}
    tf = lambda x: 'true' if x else 'false'                  # noqa: E731
    conv = [f'template int launch_pack<{b}, {dk}, {g}, {tf(v)}>(const PackParams&, hipStream_t);\n'
            for b, dk, g, v in rowfmt]
    reads = [(b, dk, g, v, q, k) for b, dk, g, v in rowfmt for q in (1, 0) for k in (0, 1)
             if not k or (b, dk, g, v) in kda_fmt]
    conv += [f'template int launch_read<{b}, {dk}, {g}, {tf(q)}, {tf(k)}, {tf(v)}>(const ReadParams&, hipStream_t);\n'
             for b, dk, g, v, q, k in reads]
    for k in range(0, len(conv), 2 * CHUNK):
        path = os.path.join(OUT, f'inst_convert_{k // (2 * CHUNK):02d}.hip')
        _write_if_changed(path, '// generated by build.py\n#include "../sq_convert.cuh"\nnamespace sq {\n'
                          + ''.join(conv[k:k + 2 * CHUNK]) + '}\n')
        units.append(path)
    path = os.path.join(OUT, 'inst_gga_00.hip')
    _write_if_changed(path, '// generated by build.py\n#include "../sq_gga.cuh"\nnamespace sq {\n'
                      + ''.join(f'template int launch_gga<GgaTile<{dk}, {dv}>>(const GgaParams&, int, hipStream_t);\n'
                                for dk, dv in GGA_SHAPES) + '}\n')
    units.append(path)
    d = ['// generated by build.py: layout -> compiled kernel instance', '#include <atomic>', '#include "../sq_convert.cuh"',
         'namespace sq {',
         '// Which instance serves a call when several could (results do not depend on it): set through sq_debug_select,',
         '// never read from the environment.',
         'static std::atomic<int> g_no_spec{0}, g_no_quad{0}, g_ghmax{64}, g_lds_pad{0};',
         'void select_instances(int no_spec, int no_quad, int ghmax, int lds_pad) {',
         '    g_no_spec.store(no_spec != 0);',
         '    g_no_quad.store(no_quad != 0);',
         '    g_ghmax.store(ghmax > 0 ? ghmax : 64);',
         '    g_lds_pad.store(lds_pad > 0 ? lds_pad : 0);',
         '}',
         'int quad_lds_pad() { return g_lds_pad.load(std::memory_order_relaxed); }', *QUAD_OK]
    for fam, rows in CASES.items():
        P = PARAMS[fam]
        d.append(f'template <class T, int SPEC> int launch_{fam}(const {P}&, hipStream_t);')
        if fam in QUAD_FAMILIES:
            d.append(f'template <class T, int NB, int GH, int WPE, int SPEC> int launch_{fam}_quad(const {P}&, hipStream_t);')
        d.append(f'int dispatch_{fam}(const {P}& p, hipStream_t stream, bool run) {{')
        d.append('    const int spec = (run && !g_no_spec.load(std::memory_order_relaxed)) ? serving_case(p) : 0;')
        if fam in QUAD_FAMILIES:
            d.append(f'    const bool quad = !g_no_quad.load(std::memory_order_relaxed) && (!run || {fam}_quad_ok(p));')
            d.append('    const int ghmax = g_ghmax.load(std::memory_order_relaxed);')
            d.append('    const int64_t heads = int64_t(p.rows) * p.hv;')
        # smallest sufficient buffer bound first
        for c in sorted(rows, key=lambda c: c[5]):
            bits, dk, dv, group, qbuf, mmax, axv = c
            cond = (f'p.bits == {bits} && p.dk == {dk} && p.dv == {dv} && p.group == {group} && p.axv == {axv} '
                    f'&& p.qbuf == {qbuf} && p.m <= {mmax}')
            for v in quad_variants(fam, c):
                want = f'spec == {v[3]} && ' if v[3] else ''             # the general instance takes whatever is left
                size = v[4] or group_when(fam, c)
                size = f'{size} && ' if size else ''
                d.append(f'    if (quad && {want}{size}p.gqa % {v[1]} == 0 && {v[1]} <= ghmax && {cond}) return run ? {_quad_name(fam, c, v)}(p, stream) : 0;')
            for sp in specs_of(fam, c, False):
                want = f'spec == {sp} && ' if sp else ''
                d.append(f'    if ({want}{cond}) return run ? launch_{fam}<{_tile(c)}, {sp}>(p, stream) : 0;')
        d.append('    return -1;\n}')
    d.append('template <int BITS, int DK, int GROUP, bool AXV> int launch_pack(const PackParams&, hipStream_t);')
    d.append('int dispatch_pack(const PackParams& p, hipStream_t stream, bool run) {')
    for b, dk, g, v in rowfmt:
        d.append(f'    if (p.bits == {b} && p.dk == {dk} && p.group == {g} && p.axv == {v}) '
                 f'return run ? launch_pack<{b}, {dk}, {g}, {tf(v)}>(p, stream) : 0;')
    d.append('    return -1;\n}')
    d.append('template <int BITS, int DK, int GROUP, bool QBUF, bool KDA, bool AXV> '
             'int launch_read(const ReadParams&, hipStream_t);')
    d.append('int dispatch_read(const ReadParams& p, hipStream_t stream, bool run) {')
    for b, dk, g, v, q, k in reads:
        d.append(f'    if (p.bits == {b} && p.dk == {dk} && p.group == {g} && p.axv == {v} && p.qbuf == {q} '
                 f'&& p.kda == {k}) return run ? '
                 f'launch_read<{b}, {dk}, {g}, {tf(q)}, {tf(k)}, {tf(v)}>(p, stream) : 0;')
    d.append('    return -1;\n}')
    d += ['int launch_fold_order(const int32_t* idx, const int32_t* NPTR, uint32_t sN, int m, int rows, int32_t* order,',
          '                      hipStream_t stream) {',
          '    hipLaunchKernelGGL((fold_order_kernel<FO_THREADS>), dim3(1), dim3(FO_THREADS), 0, stream, idx, NPTR, sN, m, rows, order);',
          '    return int(hipGetLastError());',
          '}']
    d.append('template <int DK, int DV> struct GgaTile;')
    d.append('template <class T> int launch_gga(const GgaParams&, int, hipStream_t);')
    d.append('int dispatch_gga(const GgaParams& p, int op, hipStream_t stream, bool run) {')
    for dk, dv in GGA_SHAPES:
        d.append(f'    if (p.dk == {dk} && p.dv == {dv} && p.m <= 8) '
                 f'return run ? launch_gga<GgaTile<{dk}, {dv}>>(p, op, stream) : 0;')
    d.append('    return -1;\n}')
    d.append('}  // namespace sq\n')
    path = os.path.join(OUT, 'dispatch.hip')
    _write_if_changed(path, '\n'.join(d))
    units.append(path)
    units.append(os.path.join(HERE, 'sq_api.hip'))
    return units


def _stamp():
    """Hash of every source that goes into the library (to skip a rebuild when nothing changed)."""
    h = hashlib.sha256()
    for name in sorted(os.listdir(HERE)):
        if name.endswith(('.cuh', '.h', '.hip', '.py')):
            h.update(open(os.path.join(HERE, name), 'rb').read())
    h.update(open(os.path.join(os.path.dirname(PKG), 'include', 'statequant_hip.h'), 'rb').read())
    h.update(' '.join(HIPCC_FLAGS).encode())
    return h.hexdigest()


_INCLUDE = re.compile(r'^\s*#\s*include\s+"([^"]+)"', re.M)


def _unit_hash(src, seen=None):
    """Hash of a translation unit with every header it includes by "quotes", transitively, and the flags."""
    seen = {} if seen is None else seen
    todo = [os.path.abspath(src)]
    while todo:
        path = todo.pop()
        if path in seen or not os.path.exists(path):
            continue
        text = open(path).read()
        seen[path] = text
        todo += [os.path.normpath(os.path.join(os.path.dirname(path), inc)) for inc in _INCLUDE.findall(text)]
    h = hashlib.sha256(' '.join(_flags(src)).encode())
    for path in sorted(seen):
        h.update(path.encode())
        h.update(seen[path].encode())
    return h.hexdigest()


_SREG = re.compile(r'\bs(\d+)\b|\bs\[(\d+):(\d+)\]')


def lint_counter_loads(asm_text):
    """The workgroup kernels fetch a slot's fill counter with a scalar load written in assembly and wait for it in a
    second assembly statement further down (sq_quad.cuh: quad_dma_counter / quad_dma_counter_wait).  Between the two
    the destination register holds nothing yet, and the compiler -- which believes the value is there -- must not have
    read, copied or spilled it.  This walks the device assembly of a unit and returns one message per violation
    (empty list: fine)."""
    problems, pending, in_asm, func = [], None, False, '?'
    for no, line in enumerate(asm_text.split('\n'), 1):
        t = line.strip()
        if t.endswith(':') and not t.startswith(('.', ';')):
            func = t[:-1]
        if t.startswith(';;#ASMSTART'):
            in_asm = True
            continue
        if t.startswith(';;#ASMEND'):
            in_asm = False
            continue
        if not t or t[0] in '.;' or t.endswith(':'):
            continue
        if t.startswith('s_endpgm') and pending is not None:    # a path that leaves before the wait never uses it
            continue
        if in_asm:
            m = re.match(r's_load_dword s(\d+), ', t)
            if m:
                if pending is not None:
                    problems.append(f'{func}: line {no}: a second counter load before the wait for s{pending}')
                pending = int(m.group(1))
                continue
            if pending is not None and t.startswith('s_waitcnt') and 'lgkmcnt(0)' in t:
                pending = None
                continue
        if pending is None:
            continue
        code = t.split(';')[0]
        for m in _SREG.finditer(code):
            lo, hi = (int(m.group(1)),) * 2 if m.group(1) else (int(m.group(2)), int(m.group(3)))
            if lo <= pending <= hi:
                problems.append(f'{func}: line {no}: `{code.strip()}` touches s{pending} before its load is waited for')
                break
    if pending is not None:
        problems.append(f'{func}: counter load into s{pending} is never waited for')
    return problems


def _compile(src, force=False):
    """Compile one unit unless its object is current (same sources, headers and flags as when it was built).  Units of
    the workgroup kernels keep their device assembly long enough for lint_counter_loads to read it."""
    base = os.path.splitext(os.path.basename(src))[0]
    obj = os.path.join(OUT, base + '.o')
    tag, want = obj + '.hash', _unit_hash(src)
    if not force and os.path.exists(obj) and os.path.exists(tag) and open(tag).read() == want:
        return obj
    lint = base.startswith(tuple(f'inst_{fam}q_' for fam in QUAD_FAMILIES))
    cmd = ['hipcc', *_flags(src), *(['--save-temps=obj'] if lint else []), '-c', src, '-o', obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode:
        raise RuntimeError(f'{" ".join(cmd)}\n{r.stdout}\n{r.stderr}')
    if lint:
        temps = [os.path.join(OUT, f) for f in os.listdir(OUT) if f.startswith(base + '-') or f.startswith(base + '.hip-')]
        asm = [f for f in temps if f.endswith(f'{ARCH}.s')]
        problems = lint_counter_loads(open(asm[0]).read()) if asm else [f'no device assembly kept for {src}']
        for f in temps:
            os.remove(f)
        if problems:
            os.remove(obj)
            raise RuntimeError(f'{src}: hand-placed scalar wait violated\n  ' + '\n  '.join(problems))
    with open(tag, 'w') as f:
        f.write(want)
    return obj


def _host_stamp():
    """What the extension depends on: its source, the C ABI, and the interpreter and torch whose headers it includes."""
    import torch
    h = hashlib.sha256()
    for path in (os.path.join(HERE, 'sq_host.cpp'), os.path.join(os.path.dirname(PKG), 'include', 'statequant_hip.h')):
        h.update(open(path, 'rb').read())
    h.update(repr((torch.__version__, torch._C._GLIBCXX_USE_CXX11_ABI, os.path.basename(HOST))).encode())
    return h.hexdigest()


def build_host(force=False):
    """Compile the Python extension of the step wrappers (sq_host.cpp: host code only, against this interpreter's and
    this torch's headers) next to the library, unless it is current."""
    import torch
    from torch.utils import cpp_extension
    stamp_path, stamp = os.path.join(OUT, 'host_stamp'), _host_stamp()
    if not force and os.path.exists(HOST) and os.path.exists(stamp_path) and open(stamp_path).read() == stamp:
        return HOST
    lib_dirs = cpp_extension.library_paths()
    cmd = ['g++', '-O2', '-std=c++17', '-fPIC', '-shared', '-D__HIP_PLATFORM_AMD__=1', '-DUSE_ROCM=1',
           f'-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}', f'-DSQ_TORCH="{torch.__version__}"',
           *(f'-I{p}' for p in cpp_extension.include_paths()), '-I' + sysconfig.get_paths()['include'],
           '-I' + os.path.join(os.environ.get('ROCM_PATH', '/opt/rocm'), 'include'),
           os.path.join(HERE, 'sq_host.cpp'), '-o', HOST, *(f'-L{p}' for p in lib_dirs),
           *(f'-Wl,-rpath,{p}' for p in lib_dirs), '-ltorch_python', '-ltorch_cpu', '-lc10', '-lc10_hip']
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode:
        raise RuntimeError(f'{" ".join(cmd)}\n{r.stdout}\n{r.stderr}')
    with open(stamp_path, 'w') as f:
        f.write(stamp)
    return HOST


def build(jobs=None, force=False, verbose=True):
    """Compile and link; returns the path of the library."""
    jobs = jobs or min(16, os.cpu_count() or 4)
    units = generate()
    stamp_path = os.path.join(OUT, 'stamp')
    stamp = _stamp()
    build_host(force)
    if not force and os.path.exists(LIB) and os.path.exists(stamp_path) and open(stamp_path).read() == stamp:
        if verbose:
            print(f'[build] {LIB} is up to date')
        return LIB
    if verbose:
        n = sum(len(specs_of(fam, c, False)) + len(quad_variants(fam, c)) for fam, r in CASES.items() for c in r)
        print(f'[build] hipcc {ARCH}: {n} step-kernel instances in {len(units)} translation units, {jobs} jobs')
    with cf.ThreadPoolExecutor(jobs) as ex:
        objs = list(ex.map(lambda u: _compile(u, force), units))
    cmd = ['hipcc', '--offload-arch=' + ARCH, '-shared', '-fPIC', '-o', LIB, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode:
        raise RuntimeError(f'{" ".join(cmd)}\n{r.stdout}\n{r.stderr}')
    with open(stamp_path, 'w') as f:
        f.write(stamp)
    if verbose:
        print(f'[build] wrote {LIB} ({os.path.getsize(LIB) / 1e6:.1f} MB)')
    return LIB


_REMARK = re.compile(r'remark: +(Function Name|VGPRs|AGPRs|SGPRs Spill|VGPRs Spill|ScratchSize \[bytes/lane\]|'
                     r'Occupancy \[waves/SIMD\]|LDS Size \[bytes/block\]): +(\S+)')


def resources(pattern='', jobs=None):
    """Print one line per compiled kernel: what the compiler's -Rpass-analysis=kernel-resource-usage remarks state
    for it (device pass only, nothing is linked).  VGPRs and AGPRs share one file of 512 registers per SIMD lane."""
    jobs = jobs or min(16, os.cpu_count() or 4)
    units = [u for u in generate() if not u.endswith(('dispatch.hip', 'sq_api.hip'))]

    def one(src):
        cmd = ['hipcc', *_flags(src), '--cuda-device-only', '-Rpass-analysis=kernel-resource-usage', '-c', src,
               '-o', os.devnull]
        r = subprocess.run(cmd, capture_output=True, text=True)
        rows, cur = [], None
        for key, val in _REMARK.findall(r.stderr):
            if key == 'Function Name':
                cur = {'name': val}
                rows.append(cur)
            elif cur is not None:
                cur[key] = val
        return rows

    with cf.ThreadPoolExecutor(jobs) as ex:
        rows = [r for unit in ex.map(one, units) for r in unit]
    demangle = subprocess.run(['c++filt'], input='\n'.join(r['name'] for r in rows), capture_output=True, text=True)
    names = demangle.stdout.split('\n') if demangle.returncode == 0 else [r['name'] for r in rows]
    print('VGPR AGPR spill(V/S) scratch occupancy   LDS  kernel')
    for r, n in sorted(zip(rows, names), key=lambda x: x[1]):
        n = n.replace('sq::', '').replace('void ', '')
        n = n[:n.index('>(') + 1] if '>(' in n else n
        if pattern in n:
            print(f"{r.get('VGPRs', '?'):>4} {r.get('AGPRs', '?'):>4} {r.get('VGPRs Spill', '?'):>5}/{r.get('SGPRs Spill', '?'):<3} "
                  f"{r.get('ScratchSize [bytes/lane]', '?'):>6} {r.get('Occupancy [waves/SIMD]', '?'):>8} "
                  f"{r.get('LDS Size [bytes/block]', '?'):>6}  {n}")


if __name__ == '__main__':
    ap = argparse.ArgumentParser()
    ap.add_argument('-j', type=int, default=None)
    ap.add_argument('--force', action='store_true')
    ap.add_argument('--timeline', action='store_true',
                    help='build libsqhip_timeline.so instead: the same library with the workgroup-per-key-head Gated '
                         'DeltaNet kernel instrumented (-DSQ_TIMELINE, see sq_gdn_quad.cuh); profile_timeline.py '
                         'loads it.  Objects go to csrc/build_timeline/')
    ap.add_argument('--resources', metavar='PATTERN', nargs='?', const='', default=None,
                    help="instead of building, print the compiler's resource usage (registers, spills, LDS, "
                         'occupancy) of every kernel whose name contains PATTERN')
    a = ap.parse_args()
    if a.timeline:
        OUT = os.path.join(HERE, 'build_timeline')
        LIB = os.path.join(PKG, 'libsqhip_timeline.so')
        HIPCC_FLAGS = HIPCC_FLAGS + ['-DSQ_TIMELINE']
    if a.resources is not None:
        resources(a.resources, a.j)
        sys.exit(0)
    try:
        build(a.j, a.force)
    except RuntimeError as e:
        print(e, file=sys.stderr)
        sys.exit(1)
