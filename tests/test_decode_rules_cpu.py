"""The decode kernel's rules of wq_gemm_plan.cpp, compiled as host code and asked on both sides of their lines."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "relax_amd", "csrc")

WRAPPER = """
#include "%s/wq_gemm_plan.cpp"
namespace wq {
int cu_count() { return 256; }
bool gemm_pipe_applicable(const Problem& p) { return p.k %% 64 == 0; }
}
static wq::Problem problem(int bits, int group, int64_t m, int64_t n, int64_t k, int tiled) {
  wq::Problem p{nullptr, nullptr, nullptr, nullptr, m, n, k, bits, group, 0, nullptr};
  p.tiled = tiled != 0;
  return p;
}
extern "C" int reads(int bits, int64_t m, int64_t n, int64_t k, int tiled, int tile_rows, int rounds) {
  return wq::weight_reads(problem(bits, bits == 4 ? 32 : 128, m, n, k, tiled), tile_rows, rounds != 0);
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(WRAPPER % CSRC)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + CSRC, "-o", str(d / "rules.so"), str(d / "rules.cpp")], check=True)
    so = C.CDLL(str(d / "rules.so"))
    so.reads.argtypes = [C.c_int, C.c_int64, C.c_int64, C.c_int64, C.c_int, C.c_int, C.c_int]
    return so


OWN, PAIRS, ONCE = 0, 1, 2


@pytest.mark.parametrize("bits,m,n,k,tiled,tile_rows,rounds,want", [
    # canonical int4 above 85 MB: non-temporally at 1 and 2 rows only (at 16 rows 33792 x 5120 takes 28.9 us so, 27.7 by own chunks)
    (4, 1, 33792, 5120, 0, 16, 0, ONCE), (4, 2, 33792, 5120, 0, 16, 0, ONCE), (4, 3, 33792, 5120, 0, 16, 0, OWN), (4, 8, 43008, 4096, 0, 16, 0, OWN),
    (4, 16, 33792, 5120, 0, 16, 0, OWN), (4, 1, 27648, 5120, 0, 16, 0, OWN), (4, 3, 152064, 4096, 0, 16, 1, OWN), (4, 2, 152064, 4096, 0, 16, 1, OWN),
    (4, 16, 33792, 5120, 1, 16, 0, ONCE), (4, 3, 152064, 4096, 1, 16, 1, ONCE),
    (8, 1, 12496, 5120, 0, 16, 0, PAIRS), (8, 16, 12512, 5120, 0, 16, 0, ONCE), (8, 8, 15360, 5120, 1, 16, 0, ONCE), (8, 8, 12288, 4096, 1, 16, 0, OWN),
    (8, 8, 2432, 4096, 0, 16, 0, OWN), (8, 8, 2448, 4096, 0, 16, 0, PAIRS), (8, 8, 8192, 1920, 0, 16, 0, OWN), (8, 4, 5120, 13824, 0, 10, 0, OWN),
    (8, 4, 10240, 8192, 0, 14, 0, ONCE), (8, 3, 152064, 5120, 0, 16, 1, ONCE), (8, 3, 70000, 896, 0, 16, 1, OWN)])
def test_how_the_decode_kernel_reads_its_weights(rules, bits, m, n, k, tiled, tile_rows, rounds, want):
    assert rules.reads(bits, m, n, k, tiled, tile_rows, rounds) == want
