"""The dispatch rules and launch plans of the dims reductions, on the CPU: the
host half of kf_reduce_dims.h is compiled by itself and asked for its plans."""
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include "kf_reduce_dims.h"
int kf_set_error(int code, const char*, ...) { return code; }
using namespace kf;
static long long arg(char** v, int i) { return atoll(v[i]); }

int main(int n, char** v) {
  if (!strcmp(v[1], "lanes"))  // offset rows cols col_stride has_x
    printf("%d\n", (int)u8_lanes((const void*)(uintptr_t)(4096 + arg(v, 2)), arg(v, 3), arg(v, 4), arg(v, 5), arg(v, 6)));
  if (!strcmp(v[1], "slabs"))  // es rows cols batch
    printf("%d\n", (int)use_mid_flat(arg(v, 3), arg(v, 4), arg(v, 3), arg(v, 2), arg(v, 5), arg(v, 3) * arg(v, 4), 1,
                                     arg(v, 3)));
  return 0;
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not installed")
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.hip").write_text(SOURCE)
    subprocess.run([HIPCC, "-O1", "-std=c++17", "--offload-arch=gfx950", "--offload-host-only",
                    "-I", os.path.join(REPO, "kernelforge.jl_amd", "csrc"), "-I", os.path.join(REPO, "include"),
                    str(d / "plan.hip"), "-o", str(d / "plan")], check=True, capture_output=True)

    def ask(*args):
        r = subprocess.run([str(d / "plan"), *map(str, args)], capture_output=True, text=True)
        assert r.returncode == 0, r.stdout
        return r.stdout.split()

    return ask


@pytest.mark.parametrize("offset,rows,cols,stride,x,lanes", [
    (0, 16, 10**6, 32, 0, 0), (0, 32, 10**6, 48, 1, 0), (0, 17, 10**6, 22, 0, 0), (1, 20, 10**6, 32, 0, 0),
    (0, 20, 10**6, 32, 0, 1), (0, 33, 10**6, 38, 0, 1), (0, 48, 10**6, 64, 1, 1), (0, 2048, 100, 2064, 0, 1),
    (0, 2049, 100, 2064, 0, 0), (0, 95, 10**6, 95, 1, 0), (0, 96, 1000, 96, 0, 1), (0, 112, 535_714, 112, 0, 0),
    (0, 301, 199_335, 301, 0, 0), (0, 301, 199_335, 301, 1, 1), (0, 301, 3000, 301, 0, 1), (0, 200, 300_000, 200, 0, 1),
    (0, 1001, 59_940, 1001, 0, 1), (3, 301, 199_335, 301, 0, 1)])
def test_u8_columns_that_take_lane_groups(plan, offset, rows, cols, stride, x, lanes):
    assert int(plan("lanes", offset, rows, cols, stride, x)[0]) == lanes


@pytest.mark.parametrize("es,rows,cols,batch,flat", [
    (4, 128, 4, 64, 0), (4, 128, 4, 1535, 0), (4, 128, 4, 1536, 1), (8, 128, 4, 1536, 1), (4, 3, 5, 10**6, 1),
    (4, 128, 9, 10**6, 0), (1, 500, 2, 2048, 0), (1, 33, 40, 6143, 0), (1, 33, 40, 6144, 1), (1, 16, 16, 1536, 1),
    (1, 256, 2, 2048, 0)])
def test_slabs_that_are_staged_whole(plan, es, rows, cols, batch, flat):
    assert int(plan("slabs", es, rows, cols, batch)[0]) == flat
