"""Waits that the compiler does not place for the library's own inline assembly, looked for in the machine code that was
built here (``libhla_s6.so``, disassembled with the toolchain's llvm-objdump), along every path through a kernel.

The compiler's hazard recognizer does not look inside inline assembly (csrc/common.h: the direct global -> LDS copies, the
maxima without quieting). On gfx950 it puts one wait state between a scalar write of M0 and a load with an LDS destination,
five between a vector instruction's write of a scalar register (``v_readfirstlane``) and a memory instruction that reads it,
and, after a matrix instruction, as many as its passes need before a vector instruction reads the result; around its own
assembly the library has to bring them by itself."""
import collections
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, 'hybrid-latent-attention_amd')
OBJDUMP = shutil.which('llvm-objdump') or '/opt/rocm/llvm/bin/llvm-objdump'


class Kernel:
    """Instructions ``(opcode, operands)`` in program order and each one's predecessors."""

    def __init__(self, lines):
        self.code, at, targets = [], {}, []
        for line in lines:
            text, _, note = line.partition('//')
            op, _, rest = text.strip().partition(' ')
            address = re.match(r'\s*([0-9A-F]+):', note)
            if not address or not re.match(r'[a-z]+_', op):
                continue
            at[int(address[1], 16)] = len(self.code)
            if 'branch' in op:
                step = int(rest.split()[0])
                targets.append((len(self.code), int(address[1], 16) + 4 + 4 * (step - 65536 if step > 32767 else step)))
            self.code.append((op, [rest] if op == 's_waitcnt' else
                              [o.strip().split(' ')[0] for o in re.split(r',\s*(?![^\[]*\])', rest)]))
        self.before = collections.defaultdict(list)
        for i, (op, _) in enumerate(self.code[:-1]):
            if op not in ('s_branch', 's_endpgm'):
                self.before[i + 1].append(i)
        for i, target in targets:
            self.before[at[target]].append(i)

    def writers(self, i, registers, states, writes):
        """Fewest wait states to instruction i, below ``states``, from one that writes any of ``registers`` by ``writes(op,
        operands)`` (the set it writes), over all paths on which nothing else has rewritten it: ``[(opcode, passed)]``."""
        found, best = [], {}
        stack = [(j, 0, frozenset(registers)) for j in self.before[i]]
        while stack:
            j, passed, left = stack.pop()
            op, operands = self.code[j]
            hit = writes(op, operands)
            if hit & left:
                found.append((op, passed))
            left -= hit | destination(op, operands)
            passed += int(operands[0]) + 1 if op == 's_nop' else 1
            if left and passed < states:
                for k in self.before[j]:
                    if best.get((k, left), states) > passed:
                        best[k, left] = passed
                        stack.append((k, passed, left))
        return found


def registers(operand):
    m = re.fullmatch(r'[-|]*([vas])\[(\d+):(\d+)\]\|?', operand)
    if m:
        return frozenset((m[1], r) for r in range(int(m[2]), int(m[3]) + 1))
    m = re.fullmatch(r'[-|]*([vas])(\d+)\|?', operand)
    return frozenset([(m[1], int(m[2]))]) if m else frozenset()


def destination(op, operands):
    if re.match(r'(global|buffer|scratch|flat)_(store|load_lds|atomic)|ds_write|s_waitcnt|s_nop|s_barrier|s_cmp|s_.*branch',
                op):
        return frozenset()
    return registers(operands[0]) if operands else frozenset()


@pytest.fixture(scope='module')
def kernels(tmp_path_factory):
    """{symbol: Kernel} of every gfx950 code object in the library."""
    if not os.path.exists(OBJDUMP):
        pytest.skip('llvm-objdump not found')
    lib = os.path.join(PKG, 'libhla_s6.so')
    if not os.path.exists(lib):
        spec = importlib.util.spec_from_file_location('hla_build', os.path.join(PKG, 'build.py'))
        build = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(build)
        build.build()
    tmp = tmp_path_factory.mktemp('code')
    shutil.copy(lib, tmp / 'lib.so')
    subprocess.run([OBJDUMP, '--offloading', 'lib.so'], cwd=tmp, check=True, capture_output=True)
    out = {}
    for obj in sorted(p for p in os.listdir(tmp) if p.endswith('gfx950')):
        text = subprocess.run([OBJDUMP, '-d', '--no-show-raw-insn', obj], cwd=tmp, check=True, capture_output=True,
                              text=True).stdout
        lines = []
        for line in text.splitlines():
            head = re.match(r'[0-9a-f]+ <(.*)>:', line)
            if head:
                lines = out.setdefault(head[1], [])
            else:
                lines.append(line)
    assert any('khop_dkdv4' in name for name in out), 'no kernel found in the library'
    return {name: Kernel(lines) for name, lines in out.items()}


def test_copies_to_lds_wait_for_m0(kernels):
    copies, short = 0, []
    for name, kernel in kernels.items():
        for i, (op, _) in enumerate(kernel.code):
            if '_load_lds_' in op:
                copies += 1
                for j in kernel.before[i]:
                    before, operands = kernel.code[j]
                    if before.startswith('s_') and operands[0] == 'm0':
                        short.append(name)
    assert copies > 100
    assert not short, f'{len(short)} of {copies} copies right behind their write of M0: {sorted(set(short))[:4]}'


def test_memory_instructions_wait_for_scalar_registers_written_by_vector_code(kernels):
    def vector(op, operands):
        return registers(operands[0]) if op.startswith('v_') else frozenset()

    short = []
    for name, kernel in kernels.items():
        for i, (op, operands) in enumerate(kernel.code):
            if re.match(r'(global|buffer|scratch|flat)_', op):
                need = frozenset(r for o in operands for r in registers(o) if r[0] == 's')
                short += [(name, *w) for w in kernel.writers(i, need, 5, vector)] if need else []
    assert not short, f'{len(short)} reads too soon: {sorted(set(short))[:4]}'


# Wait states before a vector instruction may read the result, as the compiler places them for its own instructions
MATRIX = {'v_mfma_f32_16x16x32_bf16': 8, 'v_mfma_f32_16x16x16_bf16': 8, 'v_mfma_f32_32x32x16_bf16': 12,
          'v_mfma_f32_16x16x4_f32': 10}


def test_maxima_wait_for_matrix_results(kernels):
    def matrix(op, operands):
        return registers(operands[0]) if op.startswith('v_mfma') else frozenset()

    short = []
    for name, kernel in kernels.items():
        if any(op.startswith('v_mfma') for op, _ in kernel.code):
            for i, (op, operands) in enumerate(kernel.code):
                if re.match(r'v_max3?_f32', op):
                    need = frozenset(r for o in operands[1:] for r in registers(o))
                    short += [(name, w) for w in kernel.writers(i, need, max(MATRIX.values()), matrix)
                              if w[1] < MATRIX[w[0]]]
    assert not short, f'{len(short)} reads too soon: {sorted(set(short))[:4]}'


def test_writer_ring_barrier_waits_for_the_reads_of_the_freed_stage(kernels):
    """The tiled writer's one barrier per step frees the stage read in the step before for the next copies: the reads'
    returns are waited for in the barrier's own block, not left to where the compiler puts their users."""
    tiled = {n: k.code for n, k in kernels.items() if 'writer_gemm' in n}
    assert tiled
    for name, code in tiled.items():
        barriers = [i for i, (op, _) in enumerate(code) if op == 's_barrier']
        assert barriers, name
        for i in barriers:
            waits = [args[0] for op, args in code[i - 8:i] if op == 's_waitcnt']   # with and without a copy to come
            assert code[i - 1][0] == 's_waitcnt' and all('lgkmcnt(0)' in w for w in waits), (name, waits)
