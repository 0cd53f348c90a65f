"""The room for the pieces of cut reductions in a preconditioning's scratch (csrc/precond_plan.h, which the engine
plans its calls with): it holds what a call writes, whatever the call says its operands are.  The query knows which
factors of A the caller keeps in halves, not which operands are factors."""
import ctypes
import itertools
import os
import random
import subprocess

import pytest

from torchsso import _hip

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), 'pytorch-sso_amd', 'csrc')
ROCM = os.environ.get('ROCM_PATH', '/opt/rocm')

# a line per call: the number of layers, then dG dA g_factored a_factored a_halves of each; printed: (room, need) of
# each layer, in tiles.  Need: the largest tile number times the pieces a tile has room for, as the kernels count.
PROGRAM = r'''
#include <cstdio>
#include "precond_plan.h"
using namespace kfac;
int main() {
  int layers;
  while (scanf("%d", &layers) == 1) {
    std::vector<int> v[5];
    for (int l = 0; l < layers; ++l)
      for (auto& x : v) {
        int value;
        if (scanf("%d", &value) != 1) return 1;
        x.push_back(value);
      }
    const int *const dG = v[0].data(), *const dA = v[1].data();
    const std::vector<int> room = halves_room(layers, dA, v[4].data());
    const std::vector<int> flags = operand_flags(layers, v[2].data(), v[3].data(), room.data());
    PieceSizes planned, pbs;
    plan_pieces(layers, dG, dA, room.data(), planned);
    call_pieces(layers, dG, dA, flags.data(), planned, pbs, false);
    for (int l = 0; l < layers; ++l) {
      long need = 0;
      for (int product = 0; product < PRODUCTS; ++product)
        for (int step = 0; step < STEPS; ++step) {
          const StepShape sh = step_shape(product, step, dG[l], dA[l], flags[l], false);
          const long pieces = piece_count(sh.longest, pbs[product][step]);
          if (pieces > 1) need = std::max(need, sh.tiles * pieces);
        }
      printf("%ld %ld ", (long)(piece_floats(dG[l], dA[l], room[l], planned) / (PLAN_TILE * PLAN_TILE)), need);
    }
    printf("\n");
  }
}
'''


@pytest.fixture(scope='module')
def rooms(tmp_path_factory):
    d = tmp_path_factory.mktemp('plan')
    (d / 'main.cpp').write_text(PROGRAM)
    subprocess.run(['g++', '-std=c++17', '-D__HIP_PLATFORM_AMD__', '-w', '-I', CSRC, '-isystem',
                    os.path.join(ROCM, 'include'), str(d / 'main.cpp'), '-o', str(d / 'main')], check=True)

    def run(calls):
        text = '\n'.join('%d %s' % (len(c), ' '.join(str(v) for layer in c for v in layer)) for c in calls)
        out = subprocess.run([str(d / 'main')], input=text, check=True, capture_output=True, text=True).stdout
        values = [[int(v) for v in line.split()] for line in out.splitlines()]
        assert len(values) == len(calls)
        return [list(zip(v[::2], v[1::2])) for v in values]
    return run


FLAGS = list(itertools.product((0, 1), repeat=3))
SIZES = [(64, 9216), (64, 2305), (300, 1025), (1000, 4608), (64, 1024), (64, 1280), (256, 2305), (512, 4609),
         (4096, 9217), (1, 2), (128, 128), (129, 129), (10, 513)]


def test_one_layer(rooms):
    calls = [[size + flags] for size in SIZES for flags in FLAGS]
    for call, ((room, need),) in zip(calls, rooms(calls)):
        assert need <= room, call


def test_lists_of_layers(rooms):
    rng = random.Random(0)
    size = lambda: int(round(2 ** rng.uniform(0, 13.3)))
    calls = [[(size(), size()) + rng.choice(FLAGS) for _ in range(rng.randint(1, 12))] for _ in range(4000)]
    for call, layers in zip(calls, rooms(calls)):
        assert all(need <= room for room, need in layers), call


def test_the_query_of_the_library_has_this_room(rooms):
    lib = _hip.load()
    calls = [[size + (1, a_factored, 1)] for size in SIZES for a_factored in (0, 1)]
    for call, ((_, need),) in zip(calls, rooms(calls)):
        dG, dA = call[0][:2]
        one = lambda v: (ctypes.c_int * 1)(v)
        scratch = 4 * (2 * dG * dA + need * 128 * 128)
        assert lib.kfac_precondition_halves_workspace_bytes(1, one(dG), one(dA), one(1)) >= scratch, call
