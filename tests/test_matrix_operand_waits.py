"""Wait states between a vector instruction and the matrix instruction that reads its result.

On gfx950 a v_mfma may not read a register in the two wait states after a (non-matrix) vector
instruction wrote it.  The compiler keeps them for its own instructions; it does not look
inside asm statements.  So the assembly of every kernel source with matrix instructions is
checked here as built."""
import os
import re
import subprocess

import pytest

from musc_hip import build

WAIT_STATES = 2


def _registers(operand: str) -> set[str]:
    m = re.fullmatch(r'([va])\[(\d+):(\d+)\]', operand)
    if m:
        return {m[1] + str(i) for i in range(int(m[2]), int(m[3]) + 1)}
    return {operand} if re.fullmatch(r'[va]\d+', operand) else set()


def _operands(ins: str) -> list[str]:
    parts = ins.split(None, 1)
    return [x.strip() for x in re.split(r',(?![^\[]*\])', parts[1])] if len(parts) > 1 else []


def too_close(assembly: str) -> list[tuple[str, str]]:
    """(writer, reader) pairs with fewer than WAIT_STATES wait states between them."""
    code = [line.split(';')[0].strip() for line in assembly.splitlines()]
    code = [x for x in code if x and not x.startswith(('.', '//')) and not x.endswith(':')]
    found = []
    for k, reader in enumerate(code):
        if not reader.startswith('v_mfma'):
            continue
        read = set().union(*map(_registers, (x.split()[0] for x in _operands(reader)[1:4])))
        waited, back = 0, k - 1
        while waited < WAIT_STATES and back >= 0 and not code[back].startswith(('s_branch', 's_endpgm', 's_setpc')):
            ins = code[back]
            if ins.startswith('v_') and not ins.startswith('v_mfma') and read & _registers(_operands(ins)[0]):
                found.append((ins, reader))
            waited += int(ins.split()[1], 0) + 1 if ins.startswith('s_nop') else 1
            back -= 1
    return found


def test_the_check_sees_a_short_wait():
    mfma = 'v_mfma_f32_32x32x16_f16 v[18:33], v[46:49], v[34:37], v[18:33]'
    write = 'v_fma_mixhi_f16 v37, v41, -1.0, v118 op_sel:[1,0,0] op_sel_hi:[1,0,0]'
    assert too_close(f'{write}\ns_waitcnt lgkmcnt(2)\n{mfma}') == [(write, mfma)]
    assert too_close(f'{write}\ns_nop 1\n{mfma}') == []
    assert too_close(f'{write}\n{mfma.replace("v[34:37]", "v[38:41]")}') == []


SOURCES = [s for s in sorted(os.listdir(build.CSRC)) if s.endswith('.hip')
           and 'builtin_amdgcn_mfma' in open(os.path.join(build.CSRC, s)).read()]


@pytest.mark.parametrize('source', SOURCES)
def test_matrix_operands_are_written_early_enough(source, tmp_path):
    out = tmp_path / 'kernels.s'
    subprocess.run([build.HIPCC] + build.COMMON + build.FILE_FLAGS.get(source, [])
                   + ['--cuda-device-only', '-S', os.path.join(build.CSRC, source), '-o', str(out)],
                   check=True, capture_output=True)
    assembly = out.read_text()
    assert assembly.count('v_mfma') > 0
    assert too_close(assembly) == []
