"""Builds the gfx950 shared library in-tree with hipcc (no torch C++ ABI involved) and, next to it, the Python extension
with the autograd nodes of the plain path (``_host``: g++ on torch's C++ interface)."""
from __future__ import annotations

import os
import subprocess
import tempfile
from concurrent.futures import ThreadPoolExecutor

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), 'csrc')
INCLUDE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'include')
LIB_PATH = os.path.join(CSRC, 'libtwinkle_amd.so')
SOURCES = ['api.hip', 'kernels_segments.hip', 'kernels_generic.hip', 'kernels_mfma.hip', 'kernels_rank128.hip', 'kernels_shared.hip', 'kernels_optim.hip', 'kernels_grouped.hip', 'kernels_act.hip', 'kernels_yardstick.hip']

# -packed-fp32-ops is switched off on purpose: the compiler must not form packed fp32 VALU ops.
HIPCC_FLAGS = [
    '--offload-arch=gfx950', '-O3', '-std=c++17', '-fPIC', '-Xclang', '-target-feature', '-Xclang',
    '-packed-fp32-ops', '-Wno-unused-command-line-argument',
]


# the autograd nodes of the plain path: a Python extension on torch's C++ interface, linked to the library above
HOST_SOURCE = 'host_torch.cpp'
HOST_PATH = os.path.join(os.path.dirname(CSRC), '_host.so')


def _host_commands(obj: str):
    import sysconfig

    import torch
    root = torch.__path__[0]
    system = [os.path.join(root, 'include'), os.path.join(root, 'include', 'torch', 'csrc', 'api', 'include'),
              '/opt/rocm/include', sysconfig.get_paths()['include']]
    compile_ = ['g++', '-O2', '-std=c++17', '-fPIC', '-D__HIP_PLATFORM_AMD__', '-DUSE_ROCM',
                f'-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}',
                *[a for d in system for a in ('-isystem', d)], '-I', INCLUDE, '-c', os.path.join(CSRC, HOST_SOURCE), '-o', obj]
    link = ['g++', '-shared', obj, '-o', HOST_PATH, '-L', os.path.join(root, 'lib'), '-ltorch_python', '-ltorch',
            '-ltorch_cpu', '-lc10', '-lc10_hip', '-L', CSRC, '-ltwinkle_amd', '-Wl,-rpath,$ORIGIN/csrc']
    return compile_, link


def build_library(verbose: bool = False) -> str:
    """Compile every HIP source (side by side) and link ``csrc/libtwinkle_amd.so``; returns its path."""
    hipcc = os.environ.get('HIPCC', '/opt/rocm/bin/hipcc')

    def run(cmd) -> str:
        proc = subprocess.run(cmd, capture_output=True, text=True)
        if proc.returncode != 0:
            raise RuntimeError('compiling failed:\n' + ' '.join(cmd) + '\n' + proc.stdout + proc.stderr)
        return proc.stderr

    with tempfile.TemporaryDirectory() as tmp:
        objects = [os.path.join(tmp, s.replace('.hip', '.o')) for s in SOURCES]
        compiles = [[hipcc, *HIPCC_FLAGS, '-I', INCLUDE, '-I', CSRC, '-c', os.path.join(CSRC, s), '-o', o]
                    for s, o in zip(SOURCES, objects)]
        with ThreadPoolExecutor(max_workers=min(8, os.cpu_count() or 1)) as pool:
            host_compile, host_link = _host_commands(os.path.join(tmp, 'host_torch.o'))
            notes = list(pool.map(run, [*compiles, host_compile]))
        notes.append(run([hipcc, '--offload-arch=gfx950', '-shared', *objects, '-o', LIB_PATH]))
        notes.append(run(host_link))
    if verbose:
        print('\n'.join(n for n in notes if n))
    return LIB_PATH


if __name__ == '__main__':
    print(build_library(verbose=True))
