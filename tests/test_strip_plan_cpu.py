"""Where the strip kernel is taken from 17 rows on (wq_gemm_plan.cpp), compiled as host code and asked on problems that were timed on an
MI355X without and with it; and what has to hold whatever the times: both layouts choose alike, and a build exists for the choice."""
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
extern "C" int ask(int bits, int group, int64_t m, int64_t n, int64_t k, int tiled) {
  wq::Problem p{nullptr, nullptr, nullptr, nullptr, m, n, k, bits, group, 0, nullptr};
  p.tiled = tiled != 0;
  const wq::GemmPlan strip = wq::plan_strip(p);
  const bool ahead = wq::strip_ahead(p, strip, wq::plan_stream(p, true));
  if (ahead && (strip.variant < 1 || strip.variant > 4 || !wq::strip_fits(wq::strip_row_blocks(m), strip.variant))) return -1;
  return ahead ? strip.variant : 0;
}
extern "C" int chosen(int bits, int group, int64_t m, int64_t n, int64_t k, int tiled, float other_us, float* us) {
  wq::Problem p{nullptr, nullptr, nullptr, nullptr, m, n, k, bits, group, 0, nullptr};
  p.tiled = tiled != 0;
  const wq::GemmPlan strip = wq::plan_strip(p), stream = wq::plan_stream(p, true);
  us[0] = other_us > 0.f ? other_us : wq::skinny_cost(p), us[1] = stream.us, us[2] = strip.us;
  return wq::choose_streamed(p, strip, stream, us[0]);
}
extern "C" int captured(int bits, int group, int64_t m, int64_t n, int64_t k, int tiled) {
  wq::Problem p{nullptr, nullptr, nullptr, nullptr, m, n, k, bits, group, 0, nullptr};
  p.tiled = tiled != 0;
  return wq::choose_streamed(p, wq::plan_strip(p), wq::plan_stream(p, false), wq::skinny_cost(p));
}
"""


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    d = tmp_path_factory.mktemp("strip")
    (d / "plan.cpp").write_text(WRAPPER % CSRC)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + CSRC, "-o", str(d / "plan.so"), str(d / "plan.cpp")], check=True)
    so = C.CDLL(str(d / "plan.so"))
    f = so.ask
    f.argtypes = [C.c_int, C.c_int, C.c_int64, C.c_int64, C.c_int64, C.c_int]
    so.chosen.argtypes = f.argtypes + [C.c_float, C.POINTER(C.c_float)]
    so.captured.argtypes = f.argtypes
    f.chosen, f.captured = so.chosen, so.captured
    return f


# (bits, M, N, K, column tiles, us of the strip kernel, us of the call without it); 0: not taken
TIMED = [(4, 37, 4096, 4096, 1, 9.3, 11.4), (4, 20, 4096, 4096, 1, 7.3, 8.1), (4, 37, 12288, 4096, 3, 13.9, 15.5), (4, 20, 12288, 4096, 3, 11.3, 12.4),
         (4, 37, 4096, 11008, 0, 21.5, 15.8), (4, 64, 22016, 4096, 0, 58.7, 22.6), (8, 37, 5120, 13824, 0, 37.6, 23.1), (8, 37, 27648, 5120, 0, 42.2, 39.4),
         # (K of a step more than the SIMDs share evenly; two slices on four column tiles)
         (4, 57, 3840, 1280, 0, 6.3, 5.8), (4, 34, 13312, 2304, 0, 11.5, 10.7), (8, 70, 7424, 3072, 0, 14.0, 12.6)]


@pytest.mark.parametrize("bits,m,n,k,tiles,strip_us,other_us", TIMED)
def test_the_faster_one_is_taken(ask, bits, m, n, k, tiles, strip_us, other_us):
    assert (strip_us < other_us) == (tiles > 0)
    for tiled in (0, 1):
        assert ask(bits, 32 if bits == 4 else 128, m, n, k, tiled) == tiles


def test_both_layouts_choose_alike_and_the_build_is_there(ask):
    taken = 0
    for bits in (4, 8):
        for m in (17, 24, 25, 33, 40, 41, 49, 56, 57, 64, 65, 72, 100, 129, 191, 256):
            for n in (128, 130, 1024, 2304, 4096, 5121, 8192, 12288, 16384, 22528):
                for k in (1024, 1024 + 256, 2816, 4096, 8192, 13824):
                    got = [ask(bits, 32 if bits == 4 else 128, m, n, k, tiled) for tiled in (0, 1)]
                    assert got[0] == got[1] >= 0, (bits, m, n, k)
                    taken += got[0] > 0
    assert taken > 300


@pytest.mark.parametrize("bits,group,m,n,k", [(4, 32, 16, 4096, 4096), (4, 32, 257, 1024, 1024), (4, 32, 37, 127, 4096), (4, 32, 37, 4096, 4096 + 128),
                                              (4, 64, 37, 4096, 4096), (8, 128, 37, 2048, 2048 + 128), (8, 32, 37, 2048, 2048)])
def test_not_where_it_does_not_apply(ask, bits, group, m, n, k):
    assert ask(bits, group, m, n, k, 0) == 0


@pytest.mark.parametrize("bits,m,n,k,other_us", [(4, 29, 3840, 5120, 0.0), (4, 26, 3840, 5120, 0.0), (4, 37, 4096, 4096, 8.0), (4, 37, 4096, 4096, 8.6), (8, 128, 1024, 2048, 0.0)])
def test_the_other_kernel_is_compared_with_what_would_run(ask, bits, m, n, k, other_us):
    """No kernel runs that is called slower than the other one, also where the strips are ahead of the streamed tiles on both
    layouts together and behind them on this one."""
    for tiled in (0, 1):
        us = (C.c_float * 3)()
        choice = ask.chosen(bits, 32 if bits == 4 else 128, m, n, k, tiled, other_us, us)
        assert choice == 0 or us[choice] <= us[0], (choice, list(us))
        assert (choice == 2) == (ask(bits, 32 if bits == 4 else 128, m, n, k, tiled) > 0 and us[2] <= us[0])


@pytest.mark.parametrize("bits,m,n,k", [(4, 25, 8544, 5632), (4, 31, 8656, 5632), (4, 17, 10896, 9728), (4, 37, 4096, 4096)])
def test_strips_stay_strips_under_capture(ask, bits, m, n, k):
    """Where a split that a captured call has no memory for is called little faster than none, too."""
    for tiled in (0, 1):
        assert ask.chosen(bits, 32, m, n, k, tiled, 0.0, (C.c_float * 3)()) == 2
        assert ask.captured(bits, 32, m, n, k, tiled) == 2


def test_requests_into_lds_take_m0_as_an_operand():
    import re

    asm = re.findall(r"asm volatile\((.*?)\);", open(os.path.join(CSRC, "wq_gemm_strip.hip")).read(), re.S)
    requests = [a for a in asm if "offen lds" in a]
    assert len(requests) == 2 and all('::"{m0}"(lds)' in a for a in requests)
    assert not any(re.search(r"\bm0\b", a.split("::")[0]) for a in asm)
