"""Build libkfac_hip.so (hand-written HIP for gfx950) and _host.so (the host side of its
calls, against torch's headers) in-tree with hipcc.

    python pytorch-sso_amd/build_ext.py

The libraries land next to the Python package (torchsso/) so that they travel with the
source tree; there is no JIT step at import time.
"""
import glob
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, 'csrc')
OUT = os.path.join(HERE, 'torchsso', 'libkfac_hip.so')
HOST_SOURCE = os.path.join(CSRC, 'host_bindings.cpp')
HOST_OUT = os.path.join(HERE, 'torchsso', '_host.so')

HIPCC_FLAGS = [
    '-O3', '-std=c++17', '--offload-arch=gfx950', '-fPIC', '-shared',
    # packed fp32 VALU forms are kept off for every kernel of this library
    '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops',
    '-Wno-unused-command-line-argument',
]


def sources():
    return sorted(glob.glob(os.path.join(CSRC, '*.hip')))


def host_command(hipcc):
    import torch
    root = os.path.dirname(os.path.abspath(torch.__file__))
    rocm = os.path.dirname(os.path.dirname(hipcc))
    abi = int(torch._C._GLIBCXX_USE_CXX11_ABI)
    return ([hipcc, '-x', 'c++', '-O2', '-std=c++17', '-fPIC', '-shared', '-w', '-D__HIP_PLATFORM_AMD__',
             '-D_GLIBCXX_USE_CXX11_ABI=%d' % abi, HOST_SOURCE, '-o', HOST_OUT,
             '-I' + sysconfig.get_paths()['include'], '-I' + os.path.join(root, 'include'),
             '-I' + os.path.join(root, 'include', 'torch', 'csrc', 'api', 'include'),
             '-I' + os.path.join(rocm, 'include'), '-L' + os.path.join(root, 'lib'), '-L' + os.path.join(rocm, 'lib'),
             '-ltorch_python', '-ltorch_cpu', '-lc10', '-lc10_hip', '-lamdhip64'])


def build(verbose=True):
    hipcc = os.environ.get('HIPCC', '/opt/rocm/bin/hipcc')
    objs = []
    cmd = host_command(hipcc)
    if verbose:
        print(' '.join(cmd), flush=True)
    procs = [(HOST_SOURCE, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT))]
    for src in sources():
        obj = src[:-4] + '.o'
        cmd = [hipcc] + [f for f in HIPCC_FLAGS if f != '-shared'] + ['-c', src, '-o', obj]
        if verbose:
            print(' '.join(cmd), flush=True)
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)))
        objs.append(obj)
    for src, p in procs:
        out, _ = p.communicate()
        text = out.decode(errors='replace')
        # hipcc's host pass says it does not know the packed-fp32 feature: harmless
        text = '\n'.join(l for l in text.splitlines() if 'packed-fp32-ops' not in l)
        if p.returncode != 0:
            raise RuntimeError('hipcc failed on %s:\n%s' % (src, text))
        if verbose and text.strip():
            print(text)
    cmd = [hipcc, '--offload-arch=gfx950', '-shared', '-fPIC'] + objs + ['-o', OUT]
    if verbose:
        print(' '.join(cmd), flush=True)
    subprocess.check_call(cmd)
    return OUT


if __name__ == '__main__':
    build()
    sys.exit(0)
