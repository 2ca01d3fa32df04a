"""Builds, in-tree, libocnn_hip.so (gfx950) from csrc/*.hip with hipcc, and ocnn_host.so, the layers'
host path on torch's C++ API (csrc/host.cpp), with the host compiler."""

import hashlib
import os
import subprocess
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
CSRC = os.path.join(HERE, 'csrc')
LIB_DIR = os.path.join(HERE, 'lib')
LIB_PATH = os.path.join(LIB_DIR, 'libocnn_hip.so')
HOST_PATH = os.path.join(LIB_DIR, 'ocnn_host.so')
INCLUDE = os.path.join(ROOT, 'include')

# file -> extra flags.  The key/build kernels must round every fp32 operation
# separately to reproduce the reference's point normalisation bit for bit.
SOURCES = {
    'morton.hip': ['-ffp-contract=off'],
    'build.hip': ['-ffp-contract=off'],
    'neigh.hip': [],
    'conv.hip': [],
    'conv_staged.hip': [],
    'conv_rw.hip': [],
    'conv_tile.hip': [],
    'jobs.hip': [],
    'conv_dense.hip': [],
    'dense_rows.hip': [],
    'conv_sparse.hip': [],
    'wgrad_sparse.hip': [],
    'dense_rw.hip': [],
    'dw_planned.hip': [],
    'dw_siblings.hip': [],
    'wgrad_planned.hip': [],
    'wgrad_f32.hip': [],
    'plan.hip': [],
    'misc.hip': [],
    'select.hip': [],
    'interp.hip': ['-ffp-contract=off'],
    'norm.hip': ['-ffp-contract=off'],
}

COMMON = ['-O3', '--offload-arch=gfx950', '-fPIC', '-std=c++17', '-I', INCLUDE, '-I', CSRC,
          '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops']


def _host_commands():
  """Compiler and linker command of ocnn_host.so: torch's headers and libraries, and the HIP library
  beside it.  (torch's ROCm headers ask for the platform to be named.)"""
  import torch
  base = os.path.dirname(torch.__file__)
  obj = os.path.join(LIB_DIR, 'obj', 'host.o')
  system = [os.path.join(base, 'include'), os.path.join(base, 'include', 'torch', 'csrc', 'api', 'include'),
            os.path.join(os.environ.get('ROCM_PATH', '/opt/rocm'), 'include'), sysconfig.get_paths()['include']]
  compile_ = ['g++', '-O2', '-std=c++17', '-fPIC', '-fvisibility=hidden', '-Wall', '-D__HIP_PLATFORM_AMD__=1',
              '-DUSE_ROCM=1', '-I', INCLUDE, '-I', CSRC] + ['-isystem' + d for d in system] + [
                  '-c', os.path.join(CSRC, 'host.cpp'), '-o', obj]
  link = ['g++', '-shared', '-o', HOST_PATH, obj, '-L', os.path.join(base, 'lib'), '-ltorch_python', '-ltorch',
          '-ltorch_cpu', '-lc10', '-lc10_hip', '-L', LIB_DIR, '-locnn_hip', '-Wl,-rpath,$ORIGIN']
  return compile_, link


STAMP_PATH = os.path.join(LIB_DIR, 'sources.sha256')


def source_hash():
  """Hash of everything the library is built from (sources, headers, flags)."""
  h = hashlib.sha256()
  names = sorted(os.listdir(CSRC))
  for path in [os.path.join(CSRC, n) for n in names] + [os.path.join(INCLUDE, n) for n in sorted(os.listdir(INCLUDE))]:
    if os.path.isfile(path):
      h.update(os.path.basename(path).encode())
      with open(path, 'rb') as f:
        h.update(f.read())
  h.update(repr((COMMON[:4] + COMMON[8:], sorted(SOURCES.items()))).encode())
  import torch
  h.update(torch.__version__.encode())               # (the host part is built against its C++ API)
  return h.hexdigest()


def is_current():
  """True when the library exists and was built from the sources as they are now."""
  try:
    with open(STAMP_PATH) as f:
      stamp = f.read().strip()
  except OSError:
    return False
  return os.path.exists(LIB_PATH) and os.path.exists(HOST_PATH) and stamp == source_hash()


def _hipcc():
  for cand in (os.environ.get('HIPCC'), '/opt/rocm/bin/hipcc', 'hipcc'):
    if cand and (os.path.isabs(cand) and os.path.exists(cand) or not os.path.isabs(cand)):
      return cand
  raise RuntimeError('hipcc not found')


def _run(cmd):
  res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
  if res.returncode != 0:
    raise RuntimeError('command failed: {}\n{}'.format(' '.join(cmd), res.stdout))
  return res.stdout


def build_library(verbose=False):
  """Compiles every HIP source and links the shared library.  Always compiles."""
  os.makedirs(LIB_DIR, exist_ok=True)
  obj_dir = os.path.join(LIB_DIR, 'obj')
  os.makedirs(obj_dir, exist_ok=True)
  hipcc = _hipcc()

  def compile_one(item):
    name, extra = item
    obj = os.path.join(obj_dir, name.replace('.hip', '.o'))
    _run([hipcc] + COMMON + extra + ['-c', os.path.join(CSRC, name), '-o', obj])
    return obj

  host_compile, host_link = _host_commands()
  with ThreadPoolExecutor(max_workers=min(8, len(SOURCES) + 1)) as pool:
    host = pool.submit(_run, host_compile)
    objs = list(pool.map(compile_one, SOURCES.items()))
    host.result()
  _run([hipcc, '--offload-arch=gfx950', '-shared', '-fPIC', '-o', LIB_PATH] + objs)
  _run(host_link)
  with open(STAMP_PATH, 'w') as f:
    f.write(source_hash() + '\n')
  if verbose:
    print('built', LIB_PATH, HOST_PATH)
  return LIB_PATH


if __name__ == '__main__':
  build_library(verbose=True)
