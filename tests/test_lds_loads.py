"""CPU checks of the built kernels: the wait states in front of the loads into LDS that are written as asm (csrc/lds_load.hpp),
where the compiler puts none, and no registers spilled where a reload would wait for those loads."""
import os
import re
import shutil
import subprocess
from pathlib import Path

import pytest

PKG = Path(__file__).resolve().parent.parent / 'cuda-agent_amd'
LIBRARIES = [PKG / 'lib' / 'libcuda_agent_amd.so', *(PKG / 'workspaces' / w / 'cuda_extension.so' for w in ('moe_fp8', 'sparse_mla'))]


def llvm(tool, *args, cwd=None):
    rocm = os.environ.get('ROCM_PATH') or '/opt/rocm'
    cmd = [shutil.which(tool) or f'{rocm}/llvm/bin/{tool}', *map(str, args)]
    return subprocess.run(cmd, cwd=cwd, check=True, capture_output=True, text=True).stdout


def code_objects(library, folder):
    """The gfx950 code objects of a library, written to `folder`."""
    assert library.exists(), 'build first: python __graft_entry__.py'
    llvm('llvm-objdump', '--offloading', shutil.copy(library, folder), cwd=folder)
    return sorted(folder.glob('*gfx950'))


def instructions(code_object):
    text = llvm('llvm-objdump', '-d', '--no-show-raw-insn', code_object)
    return [line.split('//')[0].strip() for line in text.splitlines() if line.startswith('\t')]


def before(code, i, states):
    """The instructions that can end less than `states` wait states before instruction i, in straight order."""
    passed = 0
    while i > 0 and passed < states:
        i -= 1
        if re.match(r's_(branch|endpgm|setpc)', code[i]):
            return
        nop = re.match(r's_nop (\w+)', code[i])
        yield code[i]
        passed += int(nop[1], 0) + 1 if nop else 1


def scalar_registers(operand):
    """Numbers of the scalar registers that `s7` or `s[6:7]` names (vcc, exec and anything else: none)."""
    m = re.fullmatch(r's(\d+)|s\[(\d+):(\d+)\]', operand)
    if m is None:
        return set()
    return {int(m[1])} if m[1] else set(range(int(m[2]), int(m[3]) + 1))


def written_by_vector_instruction(text):
    """Scalar registers among the results of a vector instruction (the first operand, and the second of a carry out)."""
    if not text.startswith('v_'):
        return set()
    operands = [o.strip() for o in text.split(None, 1)[1].split(',')] if ' ' in text else []
    results = operands[:2] if re.match(r'v_(add|sub|subrev|addc|subb|subbrev)_co_|v_mad_[iu]64|v_div_scale', text) else operands[:1]
    return set().union(*map(scalar_registers, results))


def faults(code):
    """The loads into LDS that come too soon after a write of what they read, and how many there are: 1 wait state behind a
    scalar write of M0, 5 behind a vector instruction's write of the scalar registers of the address."""
    loads = [i for i, text in enumerate(code) if '_load_lds_' in text]
    found = []
    for i in loads:
        found += [(code[i], text) for text in before(code, i, 1) if re.match(r's_\w+ m0\b', text)]
        read = set().union(*map(scalar_registers, re.findall(r's\[\d+:\d+\]|\bs\d+', code[i])))
        found += [(code[i], text) for text in before(code, i, 5) if read & written_by_vector_instruction(text)]
    return found, len(loads)


def test_scan_finds_what_it_looks_for():
    load = 'global_load_lds_dwordx4 v2, s[4:5]'
    assert faults(['s_mov_b32 m0, s7', load]) == ([(load, 's_mov_b32 m0, s7')], 1)
    assert faults(['s_mov_b32 m0, s7', 's_nop 0', load]) == ([], 1)
    assert faults(['s_mov_b32 m0, s7', 's_add_u32 s4, s4, s6', load]) == ([], 1)
    for write in ('v_readlane_b32 s5, v9, 3', 'v_readfirstlane_b32 s4, v1', 'v_cmp_gt_u32_e64 s[4:5], v1, v2',
                  'v_add_co_u32 v1, s[4:5], v2, v3'):
        assert faults([write, 's_mov_b32 m0, s7', 's_nop 2', load]) == ([(load, write)], 1)
        assert faults([write, 's_mov_b32 m0, s7', 's_nop 3', load]) == ([], 1)
    assert faults(['v_add_u32_e32 v1, s4, v2', 's_nop 0', load]) == ([], 1)


@pytest.mark.parametrize('library', LIBRARIES, ids=lambda p: p.parent.name)
def test_wait_states_before_loads_into_lds(library, tmp_path):
    loads = 0
    for code_object in code_objects(library, tmp_path):
        found, n = faults(instructions(code_object))
        assert not found, found[:5]
        loads += n
    assert loads > 100


def test_the_split_kernels_of_sparse_mla_spill_nothing(tmp_path):
    # two registers of the output's address, reloaded right before the output is stored, cost a single split over e4m3 rows 0.5 us
    notes = ''.join(llvm('llvm-readelf', '--notes', code_object) for code_object in code_objects(LIBRARIES[0], tmp_path))
    spilled = re.findall(r'\.name: +(\S*sparse_mla_split8_kernel\S*)\n.*?\.vgpr_spill_count: +(\d+)', notes, flags=re.S)
    assert len(spilled) == 2 and all(int(n) == 0 for _, n in spilled), spilled
