"""The forms in which 2 to 16 rows are dealt, asked of the plan itself (a header without anything of the device)."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

from helpers import DEALT_ROWS
from karume_amd import build

SHIM = """
#include "gemv_i4_rows_plan.h"
// {SPAN, R, deal}, 0 where the product is not dealt
extern "C" void forms(const uint32_t* shapes, uint32_t count, uint32_t* out) {
  for (uint32_t i = 0; i < count; ++i, shapes += 6, out += 3) {
    const uint32_t x = shapes[0], m = shapes[2], n = shapes[3], k = shapes[4], group = shapes[5];
    out[0] = out[1] = out[2] = 0;
    // (fp16 rows in groups of 128 and more, K a multiple of 256, are the matrix cores')
    if (!krm::rows_dealt(x == 4, m, n, k, group) || (x == 2 && group >= 128 && k % 256 == 0)) continue;
    uint32_t shift = 0;
    while ((1u << shift) < group) ++shift;
    const krm::RowsPlan p = krm::plan_rows(x, shapes[1], 256, m, n, k, shift);
    out[0] = p.span; out[1] = p.rows; out[2] = p.deal;
  }
}
"""


@pytest.fixture(scope="module")
def forms(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no compiler")
    at = tmp_path_factory.mktemp("plan")
    (at / "shim.cpp").write_text(SHIM)
    library = os.path.join(at, "shim.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", build.CSRC, str(at / "shim.cpp"), "-o", library],
                   check=True)
    call = C.CDLL(library).forms

    def of(shapes):
        shapes = np.ascontiguousarray(shapes, dtype=np.uint32)
        out = np.empty((len(shapes), 3), dtype=np.uint32)
        call(shapes.ctypes.data_as(C.c_void_p), len(shapes), out.ctypes.data_as(C.c_void_p))
        return [(int(s[0]), *map(int, f)) for s, f in zip(shapes, out)]
    return of


def test_every_form_has_a_product_that_the_gpu_tests_run(forms):
    rng = np.random.default_rng(0)
    count = 300000
    group = rng.choice([32, 64, 128], size=count)
    shapes = np.stack([rng.choice([2, 4], size=count), rng.choice([2, 4], size=count), rng.integers(2, 17, size=count),
                       np.exp(rng.uniform(0, np.log(32000), size=count)).astype(np.int64),
                       np.maximum(1, np.exp(rng.uniform(0, np.log(11008), size=count)).astype(np.int64) // group) * group,
                       group], axis=1)
    reached = {f for f in forms(shapes) if f[1]}
    tested = forms(DEALT_ROWS)
    assert all(f[1] for f in tested)
    assert len(reached) == 45 and set(tested) == reached
