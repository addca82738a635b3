"""Builds libefgs_hip.so (hipcc, gfx950) and the Python extension efgs/_native.so (its C++ autograd functions) in-tree.

Usage: python build_lib.py [--arch gfx950] [--jobs 8]
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, 'csrc')
BUILD = os.path.join(HERE, '_build')
LIB = os.path.join(HERE, 'efgs', 'libefgs_hip.so')
NATIVE = os.path.join(HERE, 'efgs', '_native.so')

# (source, extra flags). The decision-path files disable FP contraction so instance emission, blend replay and
# Adam follow the exact operation sequence of their definitions.
SOURCES = [
    ('api.cpp', []),
    ('rtc.cpp', []),
    ('scan.hip', []),
    ('raster.hip', ['-ffp-contract=off']),
    ('blend.hip', ['-ffp-contract=off']),
    ('adam.hip', ['-ffp-contract=off']),
    ('densification.hip', ['-ffp-contract=off']),
    ('ngsplat.hip', ['-ffp-contract=off']),
]

COMMON = ['-O3', '-std=c++17', '-fPIC', '-fhip-fp32-correctly-rounded-divide-sqrt',
          '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops', '-Wall', '-Wno-unused-function']


def _compile(src: str, extra: list[str], arch: str) -> str:
    obj = os.path.join(BUILD, src + '.o')
    cmd = ['hipcc', '-x', 'hip', f'--offload-arch={arch}', *COMMON, *extra, '-I', CSRC, '-c', os.path.join(CSRC, src), '-o', obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f'compiling {src} failed:\n{" ".join(cmd)}\n{r.stdout}\n{r.stderr}')
    return obj


def _run(what: str, cmd: list[str]) -> None:
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f'{what} failed:\n{" ".join(cmd)}\n{r.stdout}\n{r.stderr}')


def _compile_binding() -> str:
    """csrc/torch_binding.cpp against the installed torch (host code only)."""
    import torch
    inc = os.path.join(os.path.dirname(torch.__file__), 'include')
    obj = os.path.join(BUILD, 'torch_binding.cpp.o')
    _run('compiling torch_binding.cpp',
         ['g++', '-O2', '-std=c++17', '-fPIC', '-D__HIP_PLATFORM_AMD__=1', '-DUSE_ROCM=1', '-DTORCH_EXTENSION_NAME=_native',
          f'-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}', '-I', inc, '-I', os.path.join(inc, 'torch', 'csrc', 'api', 'include'),
          '-I', os.path.join(os.environ.get('ROCM_PATH', '/opt/rocm'), 'include'), '-I', sysconfig.get_paths()['include'],
          '-c', os.path.join(CSRC, 'torch_binding.cpp'), '-o', obj])
    return obj


def _link_binding(obj: str) -> None:
    import torch
    libs = os.path.join(os.path.dirname(torch.__file__), 'lib')
    tmp = NATIVE + '.tmp'
    _run('linking _native.so', ['g++', '-shared', '-fPIC', '-o', tmp, obj, '-L', libs, '-ltorch_python', '-ltorch', '-ltorch_cpu', '-lc10', '-lc10_hip',
                                '-L', os.path.dirname(LIB), '-l:libefgs_hip.so', '-Wl,-rpath,$ORIGIN'])
    os.replace(tmp, NATIVE)


def build(arch: str = 'gfx950', jobs: int = 8, verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        binding = ex.submit(_compile_binding)
        objs = list(ex.map(lambda s: _compile(s[0], s[1], arch), SOURCES))
        binding_obj = binding.result()
    tmp = LIB + '.tmp'
    _run('linking', ['hipcc', f'--offload-arch={arch}', '-shared', '-fPIC', '-Wl,-soname,libefgs_hip.so', '-o', tmp, *objs, '-lhiprtc'])
    os.replace(tmp, LIB)
    _link_binding(binding_obj)
    if verbose:
        print(f'built {LIB} and {NATIVE}')
    return LIB


if __name__ == '__main__':
    ap = argparse.ArgumentParser()
    ap.add_argument('--arch', default='gfx950')
    ap.add_argument('--jobs', type=int, default=8)
    args = ap.parse_args()
    build(args.arch, args.jobs, verbose=True)
    sys.exit(0)
