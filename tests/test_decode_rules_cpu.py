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
extern "C" int64_t streams(int bits, int group, int64_t m, int64_t n, int64_t k) {
  const wq::GemmPlan plan = wq::plan_decode_stream(problem(bits, group, m, n, k, 0));
  return plan.split > 1 ? plan.bytes : 0;
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
    so.streams.argtypes, so.streams.restype = [C.c_int, C.c_int, C.c_int64, C.c_int64, C.c_int64], C.c_int64
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


# (bits, group, M, N, K, streamed): on both sides of each line of decode_streams
STREAMED = [
    (8, 128, 8, 4096, 11008, 1), (8, 128, 8, 4096, 10880, 0), (8, 128, 16, 4096, 9728, 1), (8, 128, 16, 4096, 9600, 0), (8, 64, 10, 400, 9728, 1),
    (4, 32, 10, 4096, 11008, 1), (4, 32, 9, 4096, 11008, 0), (4, 128, 16, 4096, 10752, 1), (4, 32, 16, 4096, 10496, 0),
    (8, 128, 10, 5120, 8192, 1), (8, 128, 9, 5120, 8192, 0), (8, 128, 16, 5120, 8064, 0), (8, 128, 16, 4097, 8192, 1), (8, 32, 16, 5440, 8192, 1),
    (8, 128, 16, 5441, 8192, 0), (8, 128, 16, 5441, 13824, 1), (8, 128, 9, 5441, 13824, 0), (8, 128, 16, 6144, 13056, 1), (8, 128, 16, 6145, 13824, 0),
    (4, 64, 12, 5440, 8192, 1), (4, 32, 11, 5440, 8192, 0), (4, 32, 16, 5441, 8192, 0), (4, 32, 16, 8192, 10752, 1), (4, 32, 16, 8193, 10752, 0),
    (8, 16, 16, 5120, 13824, 0), (8, 128, 17, 5120, 13824, 0), (8, 128, 1, 4096, 60032, 0), (8, 128, 2, 4096, 60032, 1)]


@pytest.mark.parametrize("bits,group,m,n,k,streamed", STREAMED)
def test_long_k_on_the_streamed_kernel(rules, bits, group, m, n, k, streamed):
    got = rules.streams(bits, group, m, n, k)
    assert (got > 0) == bool(streamed) and got <= 16384 + (4 << 20), got


# The calls of wq_capi.cpp with every launch replaced by a note of what it was asked for.
CALLS = """
#include <string>
#include "%(csrc)s/wq_internal.h"
#include "%(csrc)s/../../include/mi355x_wq.h"
namespace wq {
static std::string route;
static int64_t need;
static char array[16];
static int note(const char* what, int rc) { route += what; return rc; }
int launch_gemm_stream_decode(const Problem&, void* space, int64_t) {
  return note(space == nullptr ? "slot " : space == array ? "stream:array " : "stream:workspace ", space == nullptr);
}
int launch_gemv_split(const Problem&, void* space, int64_t) { return note(space == array ? "split:array " : "split:workspace ", 0); }
int64_t decode_workspace_bytes(const Problem&) { return need; }
void* static_scratch_address() { return array; }
int64_t gemv_static_scratch_bytes() { return kDecodeSplitBytes; }
int64_t gemm_workspace_bytes(const Problem&, bool) { return 0; }
bool gemv_applicable(const Problem& p) { return p.m <= 16; }
int launch_gemv(const Problem&, int) { return note("decode ", 0); }
int launch_skinny(const Problem&, int, void*, int64_t) { return note("skinny ", 0); }
int launch_gemm(const Problem&, int, void*, int64_t) { return note("gemm ", 0); }
int launch_dequant(const Problem&, void*) { return 0; }
int launch_tile_weights(const Problem&, void*, void*, bool) { return 0; }
bool tiled_layout_defined(int, int, int64_t) { return true; }
}
extern "C" const char* route(int form, int64_t m, int64_t need) {
  static char x[64] __attribute__((aligned(16)));
  const mi355x_wq_desc d{8, 128, 0, 0, 5120, 13824};
  wq::route.clear();
  wq::need = need;
  const int rc = form == 0   ? mi355x_wq_matmul(&d, x, x, x, x, m, nullptr)
                 : form == 1 ? mi355x_wq_matmul_ws(&d, x, x, x, nullptr, x, m, nullptr, 0, x, need)
                             : mi355x_wq_matmul_static_ws(&d, x, x, x, nullptr, x, m, nullptr, 0);
  if (rc != 0) wq::route += "refused";
  return wq::route.c_str();
}
"""


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    d = tmp_path_factory.mktemp("calls")
    (d / "calls.cpp").write_text(CALLS % dict(csrc=CSRC))
    flags = ["-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + CSRC]
    subprocess.run(["g++", "-shared", "-fPIC", *flags, "-o", str(d / "calls.so"), str(d / "calls.cpp"), os.path.join(CSRC, "wq_capi.cpp"),
                    "-L/opt/rocm/lib", "-Wl,-rpath,/opt/rocm/lib", "-lamdhip64"], check=True)
    so = C.CDLL(str(d / "calls.so"))
    so.route.argtypes, so.route.restype = [C.c_int, C.c_int64, C.c_int64], C.c_char_p
    return lambda form, m, need: so.route(("plain", "workspace", "array").index(form), m, need).decode().split()


def test_the_scratch_array_call_never_asks_for_a_slot(route):
    """A slot's first use allocates, which that entry point does not."""
    assert route("plain", 16, 0) == ["slot"]
    assert route("workspace", 16, 1 << 20) == ["split:workspace", "stream:workspace", "slot"]
    assert route("array", 16, 1 << 20) == ["split:array", "stream:array", "decode"]
    assert route("array", 16, 0) == ["decode"]
    assert route("array", 16, (4 << 20) + 16385) == ["refused"]
    assert route("array", 40, 0) == route("plain", 40, 0) == ["skinny"]
