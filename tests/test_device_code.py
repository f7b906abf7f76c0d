"""Waits that the compiler does not place for the library's own inline assembly, looked for in the machine code that was
built here (``libhla_s6.so``, disassembled with the toolchain's llvm-objdump).

The direct global -> LDS copies are inline assembly (csrc/common.h), inside which the compiler's hazard recognizer does
not look. On gfx950 it puts one wait state between a scalar write of M0 and a load with an LDS destination; the assembly
has to bring it by itself."""
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
                body.append((op, [o.strip().split(' ')[0] for o in rest.split(',')]))
    assert any('khop_dkdv4' in name for name in out), 'no kernel found in the library'
    return out


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
