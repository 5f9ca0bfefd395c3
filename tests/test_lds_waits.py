"""Finds registers that are used before an LDS read has filled them, in the assembly of kernels whose LDS reads are placed by hand.

The compiler does not know that such a read (inline assembly) is still under way: it may copy the destination in front of the wait
that the source ties to it, and the copy then holds what was there before. LDS operations of a wave complete in order and
`s_waitcnt lgkmcnt(n)` leaves at most the n newest of them; every path through a kernel is followed with, for each register under
way, the fewest operations issued behind its own."""
import os
import re
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from hidet_amd import build

SOURCES = ['gemm_fp8', 'gemm_fp8_scaled', 'gemm_mid_fp8', 'gemm_mid_w4a16', 'gemm_mid_w8a16', 'gemm_w4a16', 'gemm_w8a16']

_LABEL = re.compile(r'^([.\w$]+):')
_VECTOR = re.compile(r'\b([va])(?:(\d+)|\[(\d+):(\d+)\])')
_LGKM = re.compile(r'lgkmcnt\((\d+)\)')
_MOST = 16  # the counter counts to 15: older operations than that are all alike


def _registers(text):
    for kind, one, first, last in _VECTOR.findall(text):
        for r in ([int(one)] if one else range(int(first), int(last) + 1)):
            yield kind, r


def _blocks(lines):
    """[(label, [(line, text)])] in order; a block ends behind a branch or in front of a label."""
    blocks, label, body = [], None, []
    for at, raw in enumerate(lines, 1):
        text = raw.split(';')[0].strip()
        found = _LABEL.match(text)
        if found:
            blocks.append((label, body))
            label, body = found.group(1), []
        elif text and not text.startswith('.'):
            body.append((at, text))
            if text.startswith(('s_branch', 's_cbranch', 's_endpgm')):
                blocks.append((label, body))
                label, body = None, []
    blocks.append((label, body))
    return blocks


def _walk(body, state, report):
    state = dict(state)
    for at, text in body:
        name, _, rest = text.partition(' ')
        if name == 's_waitcnt':
            left = _LGKM.search(rest)
            if left is None and 'cnt' not in rest:  # the number that the instruction holds
                left = (int(rest, 0) >> 8) & 15
            elif left is not None:
                left = int(left.group(1))
            if left is not None:
                state = {r: newer for r, newer in state.items() if newer < left}
            continue
        lds = name.startswith('ds_')
        operands = rest.split(',')
        filled = list(_registers(operands[0])) if name.startswith(('ds_read', 'ds_bpermute', 'ds_permute', 'ds_swizzle')) or '_rtn' in name else []
        for r in _registers(','.join(operands[1:]) if filled else rest):
            if r in state and report is not None:
                report.append((at, text, '%s%d' % r))
        if lds:
            state = {r: min(newer + 1, _MOST) for r, newer in state.items()}
            state.update((r, 0) for r in filled)
    return state


def early_uses(assembly):
    """{kernel: [(line, instruction, register)]} of every kernel; empty lists where there are none."""
    lines = assembly.splitlines()
    kernels = [m.group(1) for m in re.finditer(r'^\s*\.amdhsa_kernel\s+(\S+)', assembly, re.M)]
    starts = {l.split(':')[0]: i for i, l in enumerate(lines) if _LABEL.match(l)}
    out = {}
    for kernel in kernels:
        begin = starts[kernel]
        end = next(i for i in range(begin, len(lines)) if lines[i].startswith('.Lfunc_end'))
        blocks = _blocks(lines[begin:end])
        index = {label: i for i, (label, _) in enumerate(blocks) if label}

        def successors(i):
            last = blocks[i][1][-1][1] if blocks[i][1] else ''
            to = []
            if last.startswith(('s_branch', 's_cbranch')):
                to.append(index[last.split()[-1]])
            if not last.startswith(('s_branch', 's_endpgm')) and i + 1 < len(blocks):
                to.append(i + 1)
            return to

        entry, todo = {0: {}}, [0]
        while todo:
            i = todo.pop()
            after = _walk(blocks[i][1], entry[i], None)
            for j in successors(i):
                if j not in entry:
                    entry[j] = dict(after)
                    todo.append(j)
                    continue
                changed = False
                for r, newer in after.items():
                    if newer < entry[j].get(r, _MOST + 1):
                        entry[j][r] = newer
                        changed = True
                if changed:
                    todo.append(j)
        found = []
        for i, state in entry.items():
            _walk(blocks[i][1], state, found)
        out[kernel] = sorted((at + begin, text, r) for at, text, r in found)
    return out


def _loop(copy, wait):
    return """
kernel:
    ds_read_b32 v1, v0
    ds_read_b64 v[2:3], v0 offset:4
    {}
    s_cbranch_scc0 .L2
.L1:
    s_waitcnt lgkmcnt({})
    v_add_u32_e32 v4, v4, v1
    ds_read_b32 v1, v0
    s_cbranch_scc1 .L1
.L2:
    s_waitcnt vmcnt(0) lgkmcnt(0)
    v_add_u32_e32 v4, v3, v1
    s_endpgm
.Lfunc_end0:
    .amdhsa_kernel kernel
""".format(copy, wait)


@pytest.mark.parametrize('copy,wait,registers', [('s_nop 0', 0, []), ('s_nop 0', 1, ['v1']), ('v_mov_b32_e32 v5, v3', 0, ['v3']), ('v_mov_b32_e32 v2, 0', 0, ['v2']),
                                                 ('s_waitcnt lgkmcnt(1)\n v_mov_b32_e32 v5, v1', 0, []), ('s_waitcnt 0xc17f\n v_mov_b32_e32 v5, v2', 0, ['v2'])])
def test_what_is_found(copy, wait, registers):
    """(`wait` of 1: right for the first pass, with two reads under way, and not for the next ones, with one)"""
    assert [r for _, _, r in early_uses(_loop(copy, wait))['kernel']] == registers


def test_hand_placed_reads_are_waited_for(tmp_path):
    if not (shutil.which('hipcc') or os.path.exists('/opt/rocm/bin/hipcc')):
        pytest.skip('hipcc not available')

    def assembly(name):
        out = str(tmp_path / (name + '.s'))
        cmd = [build.hipcc()] + build.FLAGS + ['--offload-device-only', '-S', os.path.join(build.CSRC, name + '.hip'), '-o', out]
        r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        assert r.returncode == 0, r.stdout[-2000:]
        with open(out) as f:
            return f.read()

    with ThreadPoolExecutor(max_workers=4) as pool:
        found = {k: uses for text in pool.map(assembly, SOURCES) for k, uses in early_uses(text).items()}
    assert len(found) >= 4 * len(SOURCES)
    assert {k: uses[:3] for k, uses in found.items() if uses} == {}
