"""Compile libk3moe.so for gfx950 in-tree with hipcc (no torch C++ extension).

The library is plain `extern "C"` HIP code loaded with ctypes, so it does not
depend on torch's headers or ABI. Packed FP32 instructions are disabled for
the device code (-Xclang -target-feature -Xclang -packed-fp32-ops). hipcc hands
that option to both compiler passes and the host (x86) pass prints
"'-packed-fp32-ops' is not a recognized feature for this target"; the device
pass applies it. Every build then disassembles the gfx950 code objects of the
new library and fails if a v_pk_add_f32, v_pk_mul_f32 or v_pk_fma_f32 is in them
(`check_no_packed_fp32`), so the guard does not rest on the option alone.

Floating-point contraction is off (-ffp-contract=off): every product and sum
rounds where the source writes it, as torch's separate operations do (the
combine's w x bf16(y) is rounded before it is added, kimi.py:323); HIP's
default would fuse them into one FMA with a single rounding (its __fmul_rn /
__fadd_rn are plain operators).
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
PKG_ROOT = os.path.dirname(HERE)
CSRC = os.path.join(PKG_ROOT, 'csrc')
REPO = os.path.dirname(PKG_ROOT)
OUT = os.path.join(HERE, 'libk3moe.so')
ARCH = os.environ.get('K3MOE_ARCH', 'gfx950')

# Every kernel starts at a multiple of this many bytes of its code object (the persistent ones at their own): the
# general path's kernels too depend on where they lie. us of a TP8 rank's step at 65 / 129 / 203 tokens and the Kimi
# block at 128 / 777, medians of four runs: at 256 B (the compiler's) 222.2 / 252.0 / 264.3 / 453.9 / 672.2, 512 B
# 222.2 / 252.1 / 264.3 / 453.7 / 670.4, 1 KiB 221.5 / 251.4 / 263.1 / 453.2 / 670.2, 2 KiB 222.2 / 252.0 / 263.2 /
# 453.9 / 672.7, 8 KiB 222.2 / 252.2 / 263.7 / 452.9 / 671.5, 32 KiB 222.4 / 252.7 / 264.6 / 453.3 / 670.7; before the
# persistent kernels left the code object 221.9 / 251.8 / 263.1 / 455.6 / 674.0 (a second run: 1 KiB 223.0 / 251.6 /
# 263.7 / 452.6 / 668.7, before 221.9 / 250.8 / 262.6 / 456.0 / 669.8).
KERNEL_ALIGN = 1024

# Translation units, each a code object of its own (k3moe_persistent.hip: why).
SOURCES = ['k3moe.hip', 'k3moe_persistent.hip']


def hipcc() -> str:
    for cand in (os.environ.get('HIPCC'), shutil.which('hipcc'), '/opt/rocm/bin/hipcc'):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError('hipcc not found')


def command(out: str = OUT, source: str = SOURCES[0], how: str = '-shared') -> list[str]:
    """The hipcc line that makes `out` (how: '-shared' a library, '-c' an object) of one source."""
    return [hipcc(), f'--offload-arch={ARCH}', '-O3', '-std=c++17', '-fPIC', how, '-ffp-contract=off',
            '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops',
            '-Xarch_device', f'-falign-functions={KERNEL_ALIGN}', '-Wno-unused-command-line-argument',
            '-I', os.path.join(REPO, 'include'), os.path.join(CSRC, source), '-o', out]


HOST_PASS_NOTE = "'-packed-fp32-ops' is not a recognized feature for this target"
PACKED_FP32 = ('v_pk_add_f32', 'v_pk_mul_f32', 'v_pk_fma_f32')


def llvm_tool(name: str) -> str:
    for root in (os.environ.get('ROCM_PATH', '/opt/rocm'), '/opt/rocm'):
        path = os.path.join(root, 'llvm', 'bin', name)
        if os.path.exists(path):
            return path
    raise RuntimeError(f'{name} not found under the ROCm llvm tools')


def code_objects(lib: str, tool: str, *args: str) -> list[str]:
    """What an llvm tool prints for each gfx950 code object of `lib` (extracted in a scratch directory)."""
    with tempfile.TemporaryDirectory() as tmp:
        copy = os.path.join(tmp, 'lib.so')
        shutil.copyfile(lib, copy)
        subprocess.run([llvm_tool('llvm-objdump'), '--offloading', copy], cwd=tmp, check=True,
                       capture_output=True, text=True)
        objs = sorted(f for f in os.listdir(tmp) if f.endswith(f'amdgcn-amd-amdhsa--{ARCH}'))
        if not objs:
            raise RuntimeError(f'no {ARCH} code object in {lib}')
        return [subprocess.run([llvm_tool(tool), *args, obj], cwd=tmp, check=True, capture_output=True,
                               text=True).stdout for obj in objs]


def device_disassembly(lib: str) -> str:
    """The gfx950 code objects of `lib`, disassembled."""
    return ''.join(code_objects(lib, 'llvm-objdump', '-d', f'--mcpu={ARCH}'))


def kernel_addresses(lib: str = OUT) -> list[dict[str, int]]:
    """Per code object of `lib`: its kernels' mangled names and their code's addresses in it."""
    tables = []
    for text in code_objects(lib, 'llvm-readelf', '-s', '-W'):
        rows = (ln.split() for ln in text.splitlines())
        tables.append({r[7]: int(r[1], 16) for r in rows if len(r) == 8 and r[3] == 'FUNC'})
    return tables


def check_no_packed_fp32(lib: str = OUT) -> int:
    """Raise if the library's device code holds a packed-FP32 add, multiply or FMA;
    return the number of instructions checked."""
    text = device_disassembly(lib)
    found = sorted({op for op in PACKED_FP32 if op in text})
    if found:
        raise RuntimeError(f'{lib}: packed FP32 instructions in the device code: {found}')
    return sum(1 for ln in text.splitlines() if ln.startswith('\t'))


def build(verbose: bool = False) -> str:
    """Compile every HIP source into libk3moe.so (always rebuilds), check its
    device code for packed FP32 and return its path."""
    tmp = OUT + '.tmp'
    with tempfile.TemporaryDirectory() as objects:
        objs = [os.path.join(objects, s + '.o') for s in SOURCES]
        cmds = [command(obj, src, '-c') for obj, src in zip(objs, SOURCES)]
        if verbose:
            print('\n'.join(' '.join(c) for c in cmds), flush=True)
        runs = [subprocess.Popen(c, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True) for c in cmds]
        said = [r.communicate()[0] for r in runs]   # (both compile at once)
        if any(r.returncode for r in runs):
            raise RuntimeError('hipcc failed:\n' + '\n'.join(said))
        link = subprocess.run([hipcc(), f'--offload-arch={ARCH}', '-shared', '-fPIC', *objs, '-o', tmp],
                              capture_output=True, text=True)
        if link.returncode != 0:
            raise RuntimeError('hipcc failed to link:\n' + link.stderr)
    lines = [ln for text in said for ln in text.splitlines() if ln.strip()]
    host_notes = [ln for ln in lines if HOST_PASS_NOTE in ln]
    other = [ln for ln in lines if HOST_PASS_NOTE not in ln]
    if verbose and host_notes:
        print(f'hipcc host pass: {HOST_PASS_NOTE} (x{len(host_notes)}; the device pass applies it)',
              file=sys.stderr)
    if verbose and other:
        print('\n'.join(other), file=sys.stderr)
    n = check_no_packed_fp32(tmp)
    if verbose:
        print(f'device code: {n} instructions, no packed FP32', flush=True)
    os.replace(tmp, OUT)
    return OUT


if __name__ == '__main__':
    print(build(verbose=True))
