"""Waits that the compiler does not place for the library's own inline assembly, looked for in the machine code that was
built here (``libhla_s6.so``, disassembled with the toolchain's llvm-objdump).

The direct global -> LDS copies are inline assembly (csrc/common.h), inside which the compiler's hazard recognizer does
not look. On gfx950 it puts one wait state between a scalar write of M0 and a load with an LDS destination, and five
between a vector instruction's write of a scalar register (``v_readfirstlane``) and a memory instruction that reads it;
the assembly has to bring both by itself."""
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, 'hybrid-latent-attention_amd')
OBJDUMP = shutil.which('llvm-objdump') or '/opt/rocm/llvm/bin/llvm-objdump'


@pytest.fixture(scope='module')
def kernels(tmp_path_factory):
    """{kernel symbol: [(opcode, [operands]), ..]} of every gfx950 code object in the library, in program order."""
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
        body = []
        for line in text.splitlines():
            head = re.match(r'[0-9a-f]+ <(.*)>:', line)
            if head:
                body = out.setdefault(head[1], [])
                continue
            op, _, rest = line.split('//')[0].strip().partition(' ')
            if re.match(r'[a-z]+_', op):
                body.append((op, [rest] if op == 's_waitcnt' else [o.strip().split(' ')[0] for o in rest.split(',')]))
    assert any('khop_dkdv4' in name for name in out), 'no kernel found in the library'
    return out


def scalars(operand):
    m = re.fullmatch(r's\[(\d+):(\d+)\]', operand)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.fullmatch(r's(\d+)', operand)
    return {int(m[1])} if m else set()


def states(op, operands):
    """Wait states that an instruction between the two others stands for."""
    return int(operands[0]) + 1 if op == 's_nop' else 1


def test_copies_to_lds_wait_for_m0(kernels):
    copies, short = 0, []
    for name, body in kernels.items():
        for i, (op, _) in enumerate(body):
            if '_load_lds_' in op:
                copies += 1
                if i and body[i - 1][0].startswith('s_') and body[i - 1][1][0] == 'm0':
                    short.append(name)
    assert copies > 100
    assert not short, f'{len(short)} of {copies} copies right behind their write of M0: {sorted(set(short))[:4]}'


def test_memory_instructions_wait_for_scalar_registers_written_by_vector_code(kernels):
    short = []
    for name, body in kernels.items():
        for i, (op, operands) in enumerate(body):
            if not re.match(r'(global|buffer|scratch|flat)_', op):
                continue
            need = set().union(*(scalars(o) for o in operands))
            passed, j = 0, i - 1
            while need and j >= 0 and passed < 5:
                prev, args = body[j]
                if prev.startswith('v_') and scalars(args[0]) & need:
                    short.append((name, passed))
                    break
                passed += states(prev, args)
                j -= 1
    assert not short, f'{len(short)} reads too soon: {sorted(set(short))[:4]}'


def test_writer_ring_barrier_waits_for_the_reads_of_the_freed_stage(kernels):
    """The tiled writer's one barrier per step frees the stage read in the step before for the next copies: the reads'
    returns are waited for in the barrier's own block, not left to where the compiler puts their users."""
    tiled = {n: b for n, b in kernels.items() if 'writer_gemm' in n}
    assert tiled
    for name, body in tiled.items():
        barriers = [i for i, (op, _) in enumerate(body) if op == 's_barrier']
        assert barriers, name
        for i in barriers:
            waits = [args[0] for op, args in body[i - 8:i] if op == 's_waitcnt']   # with and without a copy to come
            assert body[i - 1][0] == 's_waitcnt' and all('lgkmcnt(0)' in w for w in waits), (name, waits)
