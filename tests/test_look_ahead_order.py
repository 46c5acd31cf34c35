"""The order of what a search and its helpers do in LDS.

What a helper of the refine does with a node's neighbours, next to a search that
marks each of them the moment it can see its number: the helper has read every row
that the search takes a distance of.  On the host, with the functions of the kernels'
own header and the search let in between every two of the helper's steps.

And that the compiler is told the order of stores that another wavefront sees: in
the device code of two small kernels a barrier for it stands between them."""
import ctypes
import os
import subprocess

import pytest

from pilotann_amd import build

SOURCE = r"""
#include <hip/hip_runtime.h>
#include "search_lists.h"

// Bit v of `marked`: node v was marked before.  The search runs whenever it is let in:
// it marks the neighbours it can see and remembers which of them are new to it.
// Returns the lanes of the part whose distance the search takes and nobody made.
extern "C" unsigned long long left_out(const int *node, int lanes, int part,
                                       unsigned long long marked) {
    using Ahead = pa::LookAhead<7, 2>;
    unsigned long long wanted = 0, fresh = 0, shown = 0, seen = 0;
    auto search = [&] {
        for (int l = 0; l < lanes; ++l) {
            if (!((shown & ~seen) >> l & 1)) continue;
            seen |= 1ull << l;
            if (node[l] < 0) continue;
            if (!(marked >> node[l] & 1)) fresh |= 1ull << l;
            marked |= 1ull << node[l];
        }
    };
    for (int l = 0; l < lanes; ++l) {
        const bool read = Ahead::look_then_show(
            node[l], (l & 1) == part,
            [&](int v) { search(); return (marked >> v & 1) != 0; }, search,
            [&](int) { shown |= 1ull << l; search(); });
        if (read) wanted |= 1ull << l;
    }
    return fresh & ~wanted;
}
"""


@pytest.fixture(scope='module')
def left_out(tmp_path_factory):
    at = tmp_path_factory.mktemp('order')
    source, lib = at / 'order.hip', at / 'order.so'
    source.write_text(SOURCE)
    subprocess.run(['hipcc', *build.HIP_FLAGS, '-I', build.CSRC,
                    '-I', os.path.join(build.ROOT, 'include'), '-shared', str(source),
                    '-o', str(lib)], check=True)
    fn = ctypes.CDLL(str(lib)).left_out
    fn.restype = ctypes.c_ulonglong
    fn.argtypes = [ctypes.POINTER(ctypes.c_int), ctypes.c_int, ctypes.c_int,
                   ctypes.c_ulonglong]
    return fn


@pytest.mark.parametrize('part', [0, 1])
@pytest.mark.parametrize('marked', [0, 0b1010, 0xffff])
def test_no_distance_is_left_out(part, marked, left_out):
    node = (ctypes.c_int * 16)(*[v if v % 5 else -1 for v in range(16)])
    assert left_out(node, 16, part, marked) == 0


KERNELS = r"""
#include <hip/hip_runtime.h>
#include "search_lists.h"
using Ahead = pa::LookAhead<7, 2>;

extern "C" __global__ void give(Ahead::Slots *slots, int *node) {
    Ahead ahead{*slots, -1, node[1], 1};
    node[0] = ahead.give(node[0], threadIdx.x);
}
extern "C" __global__ void drain(Ahead::Slots *slots, int *query) {
    Ahead ahead{*slots, -1, 0, 0};
    ahead.drain(threadIdx.x);
    *query = 7;
}
"""


@pytest.fixture(scope='module')
def device_code(tmp_path_factory):
    at = tmp_path_factory.mktemp('code')
    source, code = at / 'kernels.hip', at / 'kernels.ll'
    source.write_text(KERNELS)
    subprocess.run(['hipcc', *build.HIP_FLAGS, '-I', build.CSRC,
                    '-I', os.path.join(build.ROOT, 'include'), '--cuda-device-only', '-S',
                    '-emit-llvm', str(source), '-o', str(code)], check=True)
    text = code.read_text()
    return {name: text.split(f'@{name}(', 1)[1].split('\n}', 1)[0].split('\n')
            for name in ('give', 'drain')}


def between(lines, first, second):
    """The lines between the one with ``first`` and the next with ``second``."""
    at = next(i for i, line in enumerate(lines) if first in line)
    return lines[at + 1:next(i for i in range(at + 1, len(lines)) if second in lines[i])]


@pytest.mark.parametrize('kernel,first,second', [
    # the neighbours unset, then the job put; all slots seen idle, then what a
    # helper might read changed
    ('give', 'store atomic i32 -2147483648', 'store atomic i32'),
    ('drain', 'load atomic i32', 'store i32 7'),
])
def test_the_compiler_keeps_the_order(kernel, first, second, device_code):
    assert any('asm sideeffect' in line and '~{memory}' in line
               for line in between(device_code[kernel], first, second))
