"""Host choices of tile shape, K split and attention kernel (CPU only): the
library's own inline functions, compiled from its headers, at the sizes whose
kernels the GPU tests mean to reach on 256 CUs."""
import subprocess
from pathlib import Path

import pytest

import build_lib
from test_gpu_attention import BOTH_KERNELS, LONG_PLAIN
from test_gpu_kernels import NARROW_TILE_SHAPES, RING_CASES, TILE_SHAPES

TESTS = Path(__file__).resolve().parent
CUS = 256
T256, T256x192, T128x256, T128x192 = 4, 3, 2, 1   # GemmPlan.nb


@pytest.fixture(scope='module')
def ask(tmp_path_factory):
    exe = tmp_path_factory.mktemp('plans') / 'driver'
    rocm = Path(build_lib.hipcc()).resolve().parents[1]
    subprocess.run(['g++', '-std=c++17', '-O1', '-D__HIP_PLATFORM_AMD__=1', f'-isystem{rocm / "include"}',
                    f'-I{build_lib.CSRC}', f'-I{build_lib.ROOT / "include"}', str(TESTS / 'plan_driver.cpp'), '-o',
                    str(exe)], check=True)

    def run(what, *sizes):
        res = subprocess.run([str(exe)], input=' '.join(map(str, (what, *sizes, CUS))), text=True, check=True,
                             capture_output=True)
        return tuple(map(int, res.stdout.split()))
    return run


@pytest.mark.parametrize('m,n,k,nb', [(510, 512, 640, T128x256), (1376, 512, 1152, T128x256),
                                      (73, 9387, 1024, T128x256), (342, 1024, 896, T128x256)])
def test_narrow_tiles_do_not_add_a_finishing_launch(ask, m, n, k, nb):
    assert ask('gemm', m, n, k)[:2] == (nb, 1)


@pytest.mark.parametrize('m,n,k', [(160, 512, 2304), (146, 512, 2432), (1060, 256, 3840), (126, 1280, 3584)])
def test_narrow_tiles_split_eight_ways_only_where_that_was_the_plan(ask, m, n, k):
    assert ask('gemm', m, n, k)[:2] == (T128x256, 4)


@pytest.mark.parametrize('shape,plan', RING_CASES + TILE_SHAPES + NARROW_TILE_SHAPES)
def test_plans_of_the_gpu_tests(ask, shape, plan):
    assert ask('gemm', *shape) == plan


def test_ring_cases_cross_tile_boundaries_at_other_phases():
    slots = {T256: (2, 5), T256x192: (2, 5), T128x256: (1, 3), T128x192: (1, 4)}
    for nb, (units, ring) in slots.items():
        phases = {units * (k // 128) % ring for (_, _, k), plan in RING_CASES if plan[0] == nb and plan[2] > CUS}
        assert phases - {0}, nb
    assert {k // 128 % 4 for (_, _, k), plan in RING_CASES if plan[0] == T128x192} == {1, 2, 3}


@pytest.mark.parametrize('nq,heads,nk,split', BOTH_KERNELS + [LONG_PLAIN])
def test_attention_kernels_of_the_gpu_tests(ask, nq, heads, nk, split):
    assert ask('attention', nq, heads, nk) == (int(split),)
    assert ask('attention', nq, 1, nk) == (int(nk > 128),) or (nq, heads, nk, split) == LONG_PLAIN


@pytest.mark.parametrize('nq,heads,nk,split', [(2752, 6, 357, 0), (5435, 4, 364, 0), (6139, 4, 748, 0), (6139, 4, 492, 1),
                                               (6139, 4, 1004, 1), (353, 16, 1000, 1), (700, 24, 3000, 1)])
def test_three_rounds_split_only_full_steps(ask, nq, heads, nk, split):
    assert ask('attention', nq, heads, nk) == (split,)
