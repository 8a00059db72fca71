"""Which tiles the bf16 products take: the rules of pd_gemm_dtl.hpp, compiled for the host
and asked. Pins both sides that were measured, and the sizes by which the GPU tests mean to
reach one kernel or the other."""

import os
import shutil
import subprocess

import pytest

from param_decomp_amd import builder

SRC = """#include "%s"
#include <cstdio>
#include <cstdlib>
int main(int n, char** v) {
  long a[4] = {0, 0, 0, 1};
  for (int i = 2; i < n; ++i) a[i - 2] = atol(v[i]);
  const char* r = "small";
  if (v[1][0] == 'd') r = pd::big_tiles(a[0], a[1], a[2]) ? "big" : pd::deep_ring(a[0], a[1], a[2]) ? "deep"
                                                     : pd::dense_fills(a[0], a[1]) ? "small" : "small, 8 waves";
  else if (pd::big_tiles_grouped(a[0], a[1], a[2], a[3])) r = "big";
  puts(r);
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    if not (shutil.which(builder.HIPCC) or os.path.exists(builder.HIPCC)):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.hip").write_text(SRC % os.path.join(builder.CSRC, "pd_gemm_dtl.hpp"))
    subprocess.run([builder.HIPCC, "-std=c++17", "--cuda-host-only", str(d / "rule.hip"), "-o", str(d / "rule")],
                   check=True, capture_output=True)
    return lambda *a: subprocess.run([str(d / "rule"), *map(str, a)], check=True, capture_output=True,
                                     text=True).stdout.strip()


@pytest.mark.parametrize("J,E,N,problems,tile", [
    (65536, 42, 512, 2, "big"), (50664, 32, 1968, 1, "big"),
    # few rows per group: a tile per group whatever its size
    (1352, 128, 528, 1, "small"), (560, 128, 1528, 1, "small"), (248, 64, 1312, 1, "small"), (40, 128, 4096, 1, "small"),
    # the group sizes of the GPU tests
    (20578, 5, 520, 1, "big"), (20196, 5, 520, 1, "big"), (8192, 42, 512, 2, "big"), (343, 8, 264, 1, "small")])
def test_grouped_tiles(rule, J, E, N, problems, tile):
    assert rule("grouped", J, E, N, problems) == tile


@pytest.mark.parametrize("M,N,K,tile", [
    (4096, 3072, 4096, "big"), (8192, 1024, 768, "small"), (768, 4096, 4096, "deep"), (8192, 3072, 4864, "big"), (3001, 768, 4096, "deep"),
    (3000, 4104, 8, "big"), (3000, 4104, 320, "big"), (4000, 3072, 200, "big"), (2048, 2048, 768, "deep"), (2048, 2048, 760, "small, 8 waves"),
    (8192, 768, 7168, "small, 8 waves"), (8192, 1024, 3072, "small"), (7912, 968, 1464, "small"),
    (4096, 3072, 768, "big"), (4096, 4096, 776, "big"), (4000, 4104, 200, "small"),
    # the CI MLP's: hidden layer, head and pullback; the pullback and the input gradient
    (3000, 4104, 72, "big"), (3000, 4104, 4104, "big"), (3000, 72, 4104, "deep"), (300, 776, 840, "deep"),
    (300, 72, 776, "deep")])
def test_dense_tiles(rule, M, N, K, tile):
    assert rule("dense", M, N, K) == tile
