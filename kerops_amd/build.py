"""Build step: compile kerops_amd/csrc/*.hip for gfx950 into kerops_amd/_C/libkerops_hip.so, and csrc/host.cpp (the ops'
native call path, host code against the installed torch) into kerops_amd/_C/kerops_host.so.

    python -m kerops_amd.build            # compile every source, link
    python -m kerops_amd.build --verbose

hipcc cross-compiles without a GPU.  Packed-fp32 instructions are disabled for all
device code (-Xclang -target-feature -Xclang -packed-fp32-ops).  The library has
no libtorch / C++-ABI dependency; it needs only the HIP runtime, which the process
that loads it (PyTorch-ROCm) has already mapped.
"""
import argparse
import glob
import os
import subprocess
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, 'csrc')
OUT_DIR = os.path.join(HERE, '_C')
OBJ_DIR = os.path.join(OUT_DIR, 'obj')
LIB_PATH = os.path.join(OUT_DIR, 'libkerops_hip.so')
HOST_PATH = os.path.join(OUT_DIR, 'kerops_host.so')

HOST_SOURCE = os.path.join(CSRC, 'host.cpp')

ARCH = 'gfx950'
HIPCC = os.environ.get('HIPCC', '/opt/rocm/bin/hipcc')
COMMON_FLAGS = [
    '-O3', '-std=c++17', '-fPIC', f'--offload-arch={ARCH}',
    '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops',
    # a*b+c is fused only where the source says fmaf: the quantisers and the backward
    # formulas are defined step by step in IEEE fp32
    '-ffp-contract=off',
    '-Wno-unused-command-line-argument',
]
# Extra flags per source file.  The load/store optimizer pairs 8-byte LDS reads into ds_read2_b64, which gfx950 runs
# at a fraction of the rate of two ds_read_b64: the kernels that read their operands 8 bytes wide are built without it.
PER_FILE_FLAGS = {
    'dwconv_wgrad_dma.hip': ['-Xclang', '-target-feature', '-Xclang', '-load-store-opt'],
    'dwconv_bwd_dma.hip': ['-Xclang', '-target-feature', '-Xclang', '-load-store-opt'],
}


def sources():
    return sorted(glob.glob(os.path.join(CSRC, '*.hip')))


def _compile(src, verbose):
    obj = os.path.join(OBJ_DIR, os.path.basename(src)[:-4] + '.o')
    cmd = [HIPCC] + COMMON_FLAGS + PER_FILE_FLAGS.get(os.path.basename(src), []) + ['-c', src, '-o', obj]
    if verbose:
        print(' '.join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    # the host pass warns that it does not know the packed-fp32 feature: harmless
    err = '\n'.join(l for l in res.stderr.splitlines() if 'packed-fp32-ops' not in l and 'load-store-opt' not in l)
    if res.returncode != 0:
        raise RuntimeError(f'hipcc failed for {src}:\n{err}')
    if verbose and err.strip():
        print(err)
    return obj


def _compile_host(verbose):
    """The Python extension of the ops' native call path: host code only, against the installed torch."""
    import torch
    root = os.path.dirname(torch.__file__)
    cmd = [os.environ.get('CXX', 'g++'), '-O2', '-std=c++17', '-fPIC', '-shared', '-fvisibility=hidden', '-D__HIP_PLATFORM_AMD__=1',
           '-DUSE_ROCM=1', f'-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}',
           f'-DKEROPS_TORCH_VERSION="{torch.__version__}"']
    cmd += ['-isystem', os.path.join(root, 'include'), '-isystem', os.path.join(root, 'include', 'torch', 'csrc', 'api', 'include'),
            '-isystem', os.path.join(os.path.dirname(os.path.dirname(HIPCC)), 'include'),
            '-isystem', sysconfig.get_paths()['include']]
    cmd += ['-Wall', HOST_SOURCE, '-o', HOST_PATH, '-L' + os.path.join(root, 'lib')]
    cmd += ['-lc10', '-lc10_hip', '-ltorch_cpu', '-ltorch_hip', '-ltorch', '-ltorch_python']
    if verbose:
        print(' '.join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f'{cmd[0]} failed for {HOST_SOURCE}:\n{res.stderr}')
    if res.stderr.strip():
        print(res.stderr)


def build(verbose=False, jobs=None):
    os.makedirs(OBJ_DIR, exist_ok=True)
    srcs = sources()
    if not srcs:
        raise RuntimeError(f'no .hip sources under {CSRC}')
    jobs = jobs or min(len(srcs), os.cpu_count() or 1, 8)
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        host = pool.submit(_compile_host, verbose)
        objs = list(pool.map(lambda s: _compile(s, verbose), srcs))
        host.result()
    cmd = [HIPCC, '-shared', '-fPIC', f'--offload-arch={ARCH}', '-o', LIB_PATH] + objs
    if verbose:
        print(' '.join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    return LIB_PATH


if __name__ == '__main__':
    ap = argparse.ArgumentParser()
    ap.add_argument('--verbose', action='store_true')
    ap.add_argument('-j', '--jobs', type=int, default=None)
    args = ap.parse_args()
    print(build(verbose=args.verbose, jobs=args.jobs))
