"""Which calls of more than 256 rows split K on the library's memory (split_clearly_ahead in wq_gemm_plan.cpp), asked on problems that were timed
both ways on an MI355X (the times differ by 4 % and more): what the split makes slower is not split, what gains most by it is.  In between some run
whole that would gain (8, 615 x 1687 x 4608: 24.6 us whole, 22.3 split)."""
import ctypes as C
import os
import subprocess

import pytest

from tests.test_gemm_plan_cpu import CSRC, WRAPPER

ASK = """
extern "C" int clearly(int bits, int group, int64_t m, int64_t n, int64_t k, int tiled) {
  wq::Problem p{nullptr, nullptr, nullptr, nullptr, m, n, k, bits, group, 0, nullptr};
  p.tiled = tiled != 0;
  const wq::GemmPlan split = wq::plan_stream(p, true);
  return split.split == 1 ? -1 : wq::split_clearly_ahead(split, wq::plan_stream(p, false));
}
"""


@pytest.fixture(scope="module")
def clearly(tmp_path_factory):
    d = tmp_path_factory.mktemp("margin")
    (d / "margin.cpp").write_text(WRAPPER % CSRC + ASK)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + CSRC, "-o", str(d / "margin.so"), str(d / "margin.cpp")], check=True)
    f = C.CDLL(str(d / "margin.so")).clearly
    f.argtypes = [C.c_int, C.c_int, C.c_int64, C.c_int64, C.c_int64, C.c_int]
    return lambda bits, m, n, k, tiled: f(bits, 32 if bits == 4 else 128, m, n, k, tiled)


# (bits, M, N, K, us whole, us split)
SLOWER_SPLIT = [(8, 266, 896, 2560, 8.4, 9.4), (8, 297, 672, 2560, 8.0, 8.8), (8, 512, 512, 3072, 8.8, 9.5), (8, 349, 768, 3584, 9.5, 10.4), (8, 320, 896, 3840, 9.9, 10.8),
                (8, 299, 1280, 4864, 11.5, 12.5), (8, 269, 1161, 5120, 12.1, 12.8), (8, 300, 1786, 4608, 13.9, 15.4), (8, 742, 768, 5120, 15.4, 16.3), (8, 1204, 512, 5120, 15.6, 16.7),
                (4, 638, 1024, 5376, 17.4, 18.4), (8, 973, 768, 7680, 21.7, 22.7), (8, 1073, 768, 7936, 22.4, 24.1), (8, 351, 2048, 8448, 23.2, 24.4), (4, 831, 1406, 6400, 25.1, 26.4)]
FASTER_SPLIT = [(4, 350, 512, 6400, 15.0, 11.6), (8, 308, 512, 5888, 13.2, 10.3), (4, 261, 512, 10240, 21.6, 13.0), (8, 263, 592, 13824, 25.5, 15.0), (8, 259, 1096, 11520, 22.5, 18.8),
                (4, 549, 1152, 11264, 30.2, 25.8), (8, 300, 5120, 5120, 29.7, 28.2), (4, 551, 2037, 9728, 38.5, 34.7), (4, 512, 4096, 11008, 58.1, 53.9),
                (4, 425, 3150, 12288, 50.6, 47.6), (8, 300, 5120, 13824, 70.7, 61.7), (8, 1440, 1280, 13824, 74.0, 61.2)]


@pytest.mark.parametrize("bits,m,n,k,whole_us,split_us", SLOWER_SPLIT + FASTER_SPLIT)
def test_a_split_on_the_librarys_memory_is_the_faster_call(clearly, bits, m, n, k, whole_us, split_us):
    faster = split_us < whole_us
    assert [clearly(bits, m, n, k, tiled) for tiled in (0, 1)] == [faster, faster], "the same on either layout, for the same sums"
