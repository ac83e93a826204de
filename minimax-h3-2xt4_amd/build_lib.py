"""Compile the gfx950 HIP sources into the in-tree C-ABI library libw8a8.so,
and csrc/native.cpp (host C++ on torch's tensors) into the module _native.

    python minimax-h3-2xt4_amd/build_lib.py [--jobs N] [--verbose]

Each csrc/*.hip compiles to an object under _build/ (in parallel), then one
hipcc link produces w8a8/libw8a8.so next to the Python bindings.
csrc/gemm_inst.hip compiles once per (epilogue, output dtype) pair of the
GEMM (INST_VARIANTS), each with its own -D pair. The library needs neither
torch nor Python's headers: it is linked whatever becomes of _native, which is
left out where torch is not installed (only the Python package loads it).
"""
import argparse
import concurrent.futures as cf
import importlib.util
import os
import shutil
import subprocess
import sys
import sysconfig
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / 'csrc'
BUILD = PKG / '_build'
OUT = PKG / 'w8a8' / 'libw8a8.so'
NATIVE_OUT = PKG / 'w8a8' / '_native.so'
ARCH = 'gfx950'

HIPCC_FLAGS = [
    f'--offload-arch={ARCH}', '-O3', '-std=c++17', '-fPIC',
    # Every float expression is evaluated as written: no FMA contraction and
    # no fast-math reassociation or reciprocal division.
    '-ffp-contract=off', '-fno-fast-math',
    # Packed FP32 instructions stay off.
    '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops',
    '-Wno-unused-command-line-argument',
    f'-I{ROOT / "include"}', f'-I{CSRC}',
]


# (epilogue, output dtype) pairs of gemm_inst.hip: epilogue 0 int32, 1 row,
# 2 column; output 1 f16, 2 bf16, 3 f32, 4 i32.
INST_VARIANTS = [(0, 4), (1, 1), (1, 2), (1, 3), (2, 1), (2, 2), (2, 3)]


# Per-file options. attention.hip: MFMA results in VGPRs (its scores feed
# VALU work every block; in AGPRs each block would copy them over).
FILE_FLAGS = {'attention.hip': ['-mllvm', '-amdgpu-mfma-vgpr-form']}


# Kernels whose MFMAs come from inline assembly: mfma_hazards.py checks the
# assembly that the compiler made of them, and the build fails on a hazard.
CHECKED_KERNELS = {'gemm_inst.hip': 'gemm_i8_persistent'}


def hipcc():
    path = shutil.which('hipcc') or '/opt/rocm/bin/hipcc'
    if not Path(path).exists():
        raise RuntimeError('hipcc not found')
    return path


def _units():
    """(source, object name, extra flags) of every object in the library."""
    units = []
    for src in sorted(CSRC.glob('*.hip')):
        if src.name == 'gemm_inst.hip':
            for epi, out in INST_VARIANTS:
                units.append((src, f'{src.stem}_{epi}_{out}.o',
                              [f'-DW8A8_INST_EPI={epi}', f'-DW8A8_INST_OUT={out}']))
        else:
            units.append((src, src.stem + '.o', FILE_FLAGS.get(src.name, [])))
    return units


def _run(cmd, what, verbose):
    if verbose:
        print(' '.join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f'{what} failed:\n{res.stdout}\n{res.stderr}')
    if verbose and res.stderr.strip():
        print(res.stderr, file=sys.stderr)


def _compile(unit, verbose):
    src, name, extra = unit
    obj = BUILD / name
    checked = CHECKED_KERNELS.get(src.name)
    if checked is None:
        _run([hipcc(), *HIPCC_FLAGS, *extra, '-c', str(src), '-o', str(obj)], f'hipcc {src.name}', verbose)
        return obj
    # The assembly is kept (the compiler's temporaries take the output's
    # folder) until the check below has read it.
    tmp = BUILD / f'{obj.stem}.tmp'
    shutil.rmtree(tmp, ignore_errors=True)
    tmp.mkdir()
    _run([hipcc(), *HIPCC_FLAGS, *extra, '-save-temps=obj', '-c', str(src), '-o', str(tmp / name)],
         f'hipcc {src.name}', verbose)
    asm, = tmp.glob(f'*{ARCH}*.s')
    _run([sys.executable, str(PKG / 'mfma_hazards.py'), str(asm), checked], f'wait states of {name}', verbose)
    os.replace(tmp / name, obj)
    shutil.rmtree(tmp)
    return obj


def _compile_native(verbose):
    """Object of csrc/native.cpp: plain host C++ against torch's headers."""
    from torch.utils.cpp_extension import include_paths
    import torch
    obj = BUILD / 'native.o'
    rocm = Path(hipcc()).resolve().parents[1]
    _run(['g++', '-O2', '-std=c++17', '-fPIC', '-fvisibility=hidden', '-D__HIP_PLATFORM_AMD__=1', '-DUSE_ROCM=1',
          f'-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}', f'-I{ROOT / "include"}',
          *(f'-isystem{p}' for p in include_paths()), f'-isystem{rocm / "include"}',
          f'-isystem{sysconfig.get_paths()["include"]}', '-c', str(CSRC / 'native.cpp'), '-o', str(obj)],
         'g++ native.cpp', verbose)
    return obj


def _link_native(obj, verbose):
    from torch.utils.cpp_extension import library_paths
    tmp = NATIVE_OUT.with_suffix('.so.tmp')
    _run(['g++', '-shared', '-fPIC', str(obj), '-o', str(tmp), f'-L{OUT.parent}', '-l:libw8a8.so', '-Wl,-rpath,$ORIGIN',
          *(f'-L{p}' for p in library_paths()), '-ltorch_python', '-ltorch_cpu', '-lc10', '-lc10_hip'],
         'link _native', verbose)
    os.replace(tmp, NATIVE_OUT)


def _link(objs, verbose):
    tmp = OUT.with_suffix('.so.tmp')
    _run([hipcc(), f'--offload-arch={ARCH}', '-shared', '-fPIC', *map(str, objs), '-o', str(tmp)], 'link', verbose)
    os.replace(tmp, OUT)


def build(jobs=None, verbose=False):
    BUILD.mkdir(exist_ok=True)
    units = _units()
    jobs = jobs or min(len(units) + 1, max(1, os.cpu_count() or 4))
    with_native = importlib.util.find_spec('torch') is not None
    with cf.ThreadPoolExecutor(max_workers=jobs) as pool:
        native = pool.submit(_compile_native, verbose) if with_native else None
        objs = list(pool.map(lambda u: _compile(u, verbose), units))
    _link(objs, verbose)
    if with_native:
        _link_native(native.result(), verbose)
    return OUT


if __name__ == '__main__':
    ap = argparse.ArgumentParser()
    ap.add_argument('--jobs', type=int, default=None)
    ap.add_argument('--verbose', action='store_true')
    args = ap.parse_args()
    print(build(args.jobs, args.verbose))
