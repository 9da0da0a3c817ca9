"""Products in the kernel form and tile that each case names, against float64.

Which form a product takes follows from its sizes alone (gemm_plan), so every
case states what it is there for and the plan is checked against that, without
a GPU too: a rule that moves a case to another form fails here instead of
leaving a form without a test.
"""
import ctypes as C

import pytest

from mesh_amd import _lib
from tests import test_gpu_kernels as kernels

STORE, SWIGLU = 0, 1


class GemmPlan(C.Structure):
    """zr::GemmPlan (zr_internal.h)."""
    _fields_ = [(n, C.c_int) for n in ("wm", "wn", "waves_m", "waves_n", "stages")] + [("few_rows", C.c_bool)] + \
               [(n, C.c_int) for n in ("KT", "NT", "row_blocks", "col_blocks", "splits", "kt_per_split")] + \
               [("direct", C.c_bool), ("ws_floats", C.c_size_t)]


def gemm_plan(m, n, k, epilogue):
    fn = C.CDLL(_lib.LIB_PATH)._ZN2zr9gemm_planEiiii
    fn.restype, fn.argtypes = GemmPlan, [C.c_int] * 4
    return fn(m, n, k, epilogue)


# (m, k, f, k-steps per wave of 4)
KSPLIT = [(9, 128, 64, 1), (15, 256, 96, 2), (31, 512, 1024, 4), (32, 2048, 5632, 16),  # one tile of 32 rows
          (33, 128, 64, 1), (45, 256, 96, 2), (63, 896, 512, 7)]                          # two


@pytest.mark.parametrize("m,k,f,steps", KSPLIT)
def test_ksplit_cases_take_the_launch_they_name(m, k, f, steps):
    p = gemm_plan(m, 2 * f, k, SWIGLU)
    assert (p.few_rows, p.waves_m, p.direct, p.splits, p.KT) == (False, 0, True, 1, 4 * steps)


@pytest.mark.gpu
@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("m,k,f,steps", KSPLIT)
def test_swiglu_with_k_over_four_waves(split, m, k, f, steps):
    """gemm_swiglu_ksplit_kernel: fewer steps per wave than its ring has
    stages, and rows that end inside a 32-row tile."""
    kernels.test_gemm_swiglu_matches_fp64(split, m, k, f)


# K steps that are no multiple of 4: (m, k, f, row tile, splits)
REDUCED = [(9, 64, 32, 32, 1), (11, 96, 96, 32, 1), (23, 320, 320, 32, 2), (32, 1120, 96, 32, 7),
           (33, 96, 96, 64, 1), (50, 320, 512, 64, 2)]


@pytest.mark.parametrize("m,k,f,bm,splits", REDUCED)
def test_reduced_cases_take_the_tiles_they_name(m, k, f, bm, splits):
    p = gemm_plan(m, 2 * f, k, SWIGLU)
    assert (p.few_rows, p.wm * p.waves_m * 32, p.wn * p.waves_n * 32, p.splits, p.direct) == (False, bm, 128, splits, False)


@pytest.mark.gpu
@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("m,k,f,bm,splits", REDUCED)
def test_swiglu_in_the_slab_reduce(split, m, k, f, bm, splits):
    kernels.test_gemm_swiglu_matches_fp64(split, m, k, f)
