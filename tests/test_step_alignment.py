"""Where the caller's tensors may start (CPU): the general path's choice of kernels by their addresses.

place_plan (csrc/k3moe_plan.hpp) compiled for the host: tensors that start inside a 16-byte word (weight scales in
rows that are no whole words: inside a 4-byte one) leave the kernels that read them by direct-to-LDS loads, and what
replaces those fits the areas of the plan's workspace.
"""

import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NAMES = ('x', 'xin', 'router', 'gate_blocks', 'gate_scales', 'up_blocks', 'up_scales', 'down_blocks', 'down_scales')

SOURCE = r'''
#include <stdio.h>
#include <stdlib.h>
#define __host__
#define __device__
#include "k3moe.h"
#include "k3moe_plan.hpp"
using namespace k3moe;
int main(int argc, char **argv) {  // per line: tokens experts topk hidden latent inter path, nine start addresses
  int v[16];
  while (true) {
    for (int j = 0; j < 16; ++j) if (scanf("%d", v + j) != 1) return 0;
    k3moe_dims d{v[0], v[1], v[2], v[3], v[4], v[5], 0, 0, 0, v[6]};
    Plan p;
    make_plan(d, 256, p, 0);
    auto at = [&](int j) { return reinterpret_cast<const void *>((uintptr_t)4096 + v[7 + j]); };
    const size_t y_end = p.o_ids;  // the pair outputs' area ends where the next one starts
    place_plan(p, at(0), at(1), at(2), at(3), at(4), at(5), at(6), at(7), at(8));
    const size_t h = (size_t)p.P * p.I * 2;
    const bool split = p.fgemm, streams = !p.sgemm && !p.xgemm;
    const size_t room = p.path != kPathGeneral ? 0 : (p.o_h == p.o_hq ? p.o_ebf - p.o_hq : p.o_xq - p.o_h);
    printf("%d %d %d %d %d %d %d\n", p.path == kPathGeneral, p.rgemm, p.sgemm != 0, p.xgemm, p.fgemm,
           p.path != kPathGeneral || split || h <= room,
           p.path != kPathGeneral ||
               ((size_t)p.Sr * p.B * p.Epad * 4 <= y_end - p.o_logit && (!streams || p.Sg == 1 || p.o_gcnt > p.o_gpart)));
  }
}
'''

# (tokens, experts, topk, hidden, latent, inter, path): 32, 64 and 96 pairs per unit, the grouped paths, narrow scale
# rows, a router of no whole 64-k steps, few wide experts
STEPS = [(203, 384, 8, 7168, 7168, 256, 0), (1500, 896, 16, 7168, 3584, 384, 0), (2999, 384, 8, 7168, 7168, 256, 0),
         (700, 64, 8, 2048, 2048, 512, 3), (700, 64, 8, 2048, 2048, 512, 6), (300, 16, 2, 1056, 1024, 512, 0),
         (900, 1024, 1, 320, 512, 128, 0)]


@pytest.fixture(scope='module')
def place(tmp_path_factory):
    if shutil.which('g++') is None:
        pytest.skip('no g++')
    tmp = tmp_path_factory.mktemp('place')
    (tmp / 'place.cpp').write_text(SOURCE)
    subprocess.run(['g++', '-std=c++17', '-I', os.path.join(REPO, 'include'), '-I',
                    os.path.join(REPO, 'kimi-k3-goalbox_amd', 'csrc'), str(tmp / 'place.cpp'), '-o', str(tmp / 'place')],
                   check=True)

    def run(rows):
        text = '\n'.join(' '.join(map(str, r)) for r in rows)
        out = subprocess.run([str(tmp / 'place')], input=text, capture_output=True, text=True, check=True).stdout
        return [tuple(map(int, ln.split())) for ln in out.splitlines()]
    return run


@pytest.mark.parametrize('step', STEPS, ids=str)
def test_kernels_by_where_the_tensors_start(place, step):
    K, I = step[4:6]
    (whole,) = place([(*step, *[0]*9)])
    assert whole[0] == 1 and (whole[2] or whole[3])
    for j, name in enumerate(NAMES):
        offsets = (1, 2, 4, 8, 16)
        for off, got in zip(offsets, place([(*step, *[off*(i == j) for i in range(9)]) for off in offsets])):
            general, rgemm, sgemm, xgemm, fgemm, h_fits, rest_fits = got
            row = K//32 if name in ('gate_scales', 'up_scales') else I//32
            need = 4 if name.endswith('scales') and row % 16 else 16
            router = name in ('x', 'router') and off % 16
            streams = name not in ('x', 'router') and off % need
            assert rgemm == (0 if router else whole[1]), (name, off)
            assert (sgemm, xgemm, fgemm) == ((0, 0, 0) if streams else whole[2:5]), (name, off)
            assert h_fits and rest_fits, (name, off)


def test_persistent_plans_stay(place):
    assert place([(8, 384, 8, 7168, 7168, 256, 0, *[1]*9)])[0][0] == 0
