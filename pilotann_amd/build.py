"""Compiles the HIP/C++ sources under ``csrc/`` into ``csrc/libpilotann.so``
for gfx950.  Run as ``python -m pilotann_amd.build``; the library stays in the
source tree, where the ctypes loader looks for it."""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, 'csrc')
LIB = os.path.join(CSRC, 'libpilotann.so')
# tuning build whose traversal kernel tallies cycles per phase of a search
# (``python -m pilotann_amd.build --phase-timers``; ``bench.py --phase-split``
# loads it); not built by default and never the library the package loads
PHASE_LIB = os.path.join(CSRC, 'libpilotann_phase_timers.so')

HIP_SOURCES = ['traverse.hip', 'traverse_wide.hip', 'refine.hip', 'route.hip', 'rotate.hip',
               'knn.hip', 'reverse.hip', 'pipeline.hip']
CXX_SOURCES = ['host_search.cpp']

HIP_FLAGS = [
    '--offload-arch=gfx950', '-O3', '-std=c++17', '-fPIC',
    '-ffp-contract=off',
    # packed fp32 instructions off (device pass; the host pass warns that it
    # does not know the feature, which is harmless)
    '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops',
    '-Wno-unused-command-line-argument', '-Wno-inline-asm',
]
# the reference's host flags (setup.py:39-44) minus -ffast-math: the host
# search must add in the order it is written
CXX_FLAGS = [
    '-O3', '-std=c++17', '-fPIC', '-mavx2', '-mfma', '-fopenmp',
    '-funroll-loops', '-ffp-contract=off', '-fno-fast-math',
]


def _run(cmd, verbose):
    if verbose:
        print(' '.join(cmd), flush=True)
    subprocess.run(cmd, check=True)


def build(verbose: bool = False, output: str = LIB,
          extra_hip_flags=()) -> str:
    """Compile everything and link ``output`` (default: the library the
    loader uses).  ``extra_hip_flags`` are added to the device compiles, e.g.
    ``-DPA_PHASE_TIMERS`` for the tuning build ``PHASE_LIB``."""
    include = os.path.join(ROOT, 'include')
    compiles = []
    for compiler, flags, names in (
            ('hipcc', [*HIP_FLAGS, *extra_hip_flags], HIP_SOURCES),
            ('g++', CXX_FLAGS, CXX_SOURCES)):
        for name in names:
            src = os.path.join(CSRC, name)
            if os.path.exists(src):
                compiles.append([compiler, *flags, '-I', include, '-c', src,
                                 '-o', os.path.join(CSRC, name + '.o')])
    # side by side: the traversal's instances take a minute by themselves
    with ThreadPoolExecutor(max_workers=min(4, os.cpu_count() or 1)) as pool:
        list(pool.map(lambda cmd: _run(cmd, verbose), compiles))
    objects = [cmd[-1] for cmd in compiles]
    _run(['hipcc', '--offload-arch=gfx950', '-shared', '-fPIC', '-o', output,
          *objects, '-lgomp', '-lpthread'], verbose)
    for obj in objects:
        os.remove(obj)
    return output


if __name__ == '__main__':
    if '--phase-timers' in sys.argv:
        print(build(verbose='-q' not in sys.argv, output=PHASE_LIB,
                    extra_hip_flags=['-DPA_PHASE_TIMERS']))
    else:
        print(build(verbose='-q' not in sys.argv))
