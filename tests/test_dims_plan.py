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

// every launch's partials against the scratch query, over shapes and alignments
static int bounds() {
  const int64_t rows_l[] = {2, 3, 5, 8, 15, 16, 17, 31, 33, 65, 127, 200, 255, 256, 257, 300, 511, 513, 777, 1000, 1001,
                            1024, 1027, 2047, 2049, 4001, 4096, 4099, 8197, 10007, 65535, 131071, 262143, 1050001};
  const int64_t cols_l[] = {2, 3, 7, 8, 16, 17, 33, 64, 80, 128, 200, 400, 1000, 3001, 20000, 100003, 1000003};
  long long seen = 0, cut = 0;
  for (size_t es : {1, 4, 8})
    for (int64_t r : rows_l)
      for (int64_t c : cols_l)
        for (int64_t b : {1, 2, 7, 64, 130, 1000, 70000}) {
          if ((double)r * c * b * es > 4e10) continue;
          const int64_t room = (int64_t)dim_query(es, r, c, 2, b) - (int64_t)kRedReserved;
          const int64_t nb = b < kMaxBatchPerLaunch ? b : kMaxBatchPerLaunch;
          for (int al = 0; al < 3; ++al) {  // odd column strides, aligned ones, aligned ones at an odd base
            const int64_t cs = al ? (r + 16) / 16 * 16 : r | 1;
            const void* A = (const void*)(uintptr_t)(al == 2 ? 4096 + es : 4096);
            const DimVec v = dim_vec(A, r, cs, es, 2, b, cs * c, false, nullptr, 0);
            const bool needs = dim_need(es, r, c, 2, b, v) > 0;
            const DimPlan p = plan_launch(es, r, c, 2, v.vec, b, true), q = plan_launch(es, r, c, 2, v.vec, b, false);
            const int64_t ev = 16 / (int64_t)es, units = p.unit_vec ? (r + ev - 1) / ev : r;
            const bool whole = v.vec && r % ev == 0;
            ++seen;
            cut += plan_dim(es, r, c, 2, v.vec, b, p.ragged).split > p.split;
            if ((p.split > 1 && (int64_t)p.split * r * (int64_t)es * nb > room) || (q.split > 1 && !needs) ||
                p.split > 65535 || (p.narrow && units > kDimBlock) || (!p.narrow && !p.ragged && !p.elems) || (p.ragged && r < ev) ||
                (p.elems && (p.narrow || p.ragged || r <= kDimBlock || r > kDimBlock * ev)) ||
                (p.narrow && p.ragged && !whole && p.split > kNarrowRaggedSplits && b == 1 &&
                 p.split > plan_dim(es, r, c, 2, v.vec, b, true).split)) {
              printf("es %zu %lld x %lld batch %lld alignment %d: split %d, %d without scratch, room %lld\n", es,
                     (long long)r, (long long)c, (long long)b, al, p.split, q.split, (long long)room);
              return 1;
            }
          }
        }
  printf("ok %lld %lld\n", seen, cut);
  return 0;
}

int main(int n, char** v) {
  if (!strcmp(v[1], "bounds")) return bounds();
  if (!strcmp(v[1], "split"))  // es rows cols: contiguous columns
    printf("%d\n", plan_launch(arg(v, 2), arg(v, 3), arg(v, 4), 2,
                               dim_vec((const void*)4096, arg(v, 3), arg(v, 3), arg(v, 2), 2, 1, 0, false, nullptr, 0).vec,
                               1, true).split);
  if (!strcmp(v[1], "elems"))  // es rows cols batch: contiguous columns
    printf("%d\n", (int)plan_launch(arg(v, 2), arg(v, 3), arg(v, 4), 2,
                                    dim_vec((const void*)4096, arg(v, 3), arg(v, 3), arg(v, 2), 2, arg(v, 5),
                                            arg(v, 3) * arg(v, 4), false, nullptr, 0).vec,
                                    arg(v, 5), true).elems);
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


def test_partials_stay_within_the_scratch_query(plan):
    # whatever the alignment: the launch splits no further than the query has
    # room for, and not at all without scratch unless the query plans a split
    ok, seen, cut = plan("bounds")
    assert ok == "ok" and int(seen) > 10_000 and int(cut) > 100


@pytest.mark.parametrize("es,rows,cols,low,high", [
    (4, 1001, 30_001, 256, 512), (8, 401, 30_001, 256, 512), (1, 4001, 30_001, 256, 512),   # not 1875 partial columns
    (4, 1001, 2001, 256, 512), (1, 301, 3001, 64, 128), (4, 1001, 200, 16, 64),             # not a few workgroups
    (4, 257, 40, 1, 3), (4, 1000, 30_001, 1024, 2048)])                                     # too short; aligned: as planned
def test_splits_of_narrow_rows_off_the_vector_grid(plan, es, rows, cols, low, high):
    assert low <= int(plan("split", es, rows, cols)[0]) <= high


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


@pytest.mark.parametrize("es,rows,cols,batch,elems", [
    (1, 301, 2, 1, 1), (1, 4001, 2048, 1, 1), (1, 4001, 2049, 1, 0), (1, 256, 20, 1, 0), (1, 304, 400, 1, 0),
    (1, 4097, 20, 1, 0), (1, 500, 8, 2000, 1), (1, 500, 8, 2200, 0), (4, 1001, 20, 1, 1), (4, 1001, 31, 1, 1),
    (4, 1001, 32, 1, 0), (4, 1001, 255, 1, 0), (4, 1001, 256, 1, 1), (8, 511, 1024, 1, 1), (8, 511, 1025, 1, 0),
    (4, 1000, 20, 1, 0), (4, 1025, 20, 1, 0)])
def test_small_matrices_off_the_vector_grid(plan, es, rows, cols, batch, elems):
    assert int(plan("elems", es, rows, cols, batch)[0]) == elems
