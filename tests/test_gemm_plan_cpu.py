"""The choice of kernel from 17 rows on (wq_gemm_plan.cpp), compiled as host code and asked on problems whose kernels were
timed on an MI355X: it has to name the kernel that was the faster one (the pairs differ by 8 % at least)."""
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
extern "C" int64_t plan_bytes(int bits, int group, int64_t m, int64_t n, int64_t k) {
  return wq::plan_stream(wq::Problem{nullptr, nullptr, nullptr, nullptr, m, n, k, bits, group, 0, nullptr}, true).bytes;
}
extern "C" int pieces(int bits, int group, int64_t m, int64_t n, int64_t k, int rows, int columns, int macro_step) {
  return wq::stream_scale_pieces(wq::Problem{nullptr, nullptr, nullptr, nullptr, m, n, k, bits, group, 0, nullptr}, rows, columns, macro_step);
}
extern "C" int ask(int bits, int group, int64_t m, int64_t n, int64_t k, int tiled, int may_split, float* us) {
  wq::Problem p{nullptr, nullptr, nullptr, nullptr, m, n, k, bits, group, 0, nullptr};
  p.tiled = tiled != 0;
  const wq::GemmPlan plan = wq::plan_stream(p, may_split != 0);
  us[0] = plan.us, us[1] = wq::other_gemm_cost(p), us[2] = wq::skinny_cost(p);
  return plan.variant | plan.split << 8;
}
"""


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(WRAPPER % CSRC)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + CSRC, "-o", str(d / "plan.so"), str(d / "plan.cpp")], check=True)
    so = C.CDLL(str(d / "plan.so"))
    so.plan_bytes.argtypes, so.plan_bytes.restype = [C.c_int, C.c_int, C.c_int64, C.c_int64, C.c_int64], C.c_int64
    f = so.ask
    f.argtypes = [C.c_int, C.c_int, C.c_int64, C.c_int64, C.c_int64, C.c_int, C.c_int, C.POINTER(C.c_float)]

    def call(bits, m, n, k, tiled, may_split=True, group=None):
        us = (C.c_float * 3)()
        r = f(bits, group or (32 if bits == 4 else 128), m, n, k, tiled, may_split, us)
        return r & 0xFF, r >> 8, dict(zip(("stream", "other", "skinny"), us))
    so.pieces.argtypes = [C.c_int, C.c_int] + [C.c_int64] * 3 + [C.c_int] * 3
    call.plan_bytes, call.pieces = so.plan_bytes, so.pieces
    return call


# (bits, M, N, K, tile-major, the faster one, us of the direct-weight kernel, us of the streamed one)
ABOVE_256_ROWS = [
    (8, 512, 15360, 5120, 1, "direct", 80.2, 104.0), (8, 1024, 5120, 13824, 1, "direct", 163.3, 210.3),
    (8, 1536, 15360, 5120, 1, "direct", 229.7, 282.2), (8, 768, 27648, 5120, 1, "direct", 224.5, 277.3),
    (8, 1049, 5425, 3072, 1, "direct", 51.9, 61.6), (8, 407, 13173, 2048, 1, "direct", 40.6, 46.3),
    (4, 1536, 12288, 4096, 1, "direct", 162.9, 177.7), (4, 768, 22016, 4096, 1, "direct", 160.4, 175.0),
    (8, 512, 5120, 13824, 0, "stream", 129.8, 103.3), (8, 2048, 15360, 5120, 0, "stream", 342.0, 291.9),
    (4, 277, 13519, 9728, 1, "direct", 111.0, 124.2), (4, 768, 4096, 11008, 0, "stream", 104.1, 83.3), (4, 1906, 2640, 1280, 0, "stream", 28.5, 21.2),
    (8, 300, 2048, 1280, 0, "stream", 17.1, 8.3), (4, 300, 2048, 1280, 1, "stream", 15.3, 8.4),
    (8, 341, 29056, 1792, 1, "stream", 63.8, 57.5), (4, 467, 19584, 1792, 1, "stream", 58.0, 52.4),
    (8, 512, 5120, 13824, 1, "stream", 134.7, 113.3), (4, 1024, 4096, 11008, 1, "stream", 105.8, 97.0),
    (4, 1273, 18827, 1280, 0, "stream", 105.3, 89.1), (4, 747, 7825, 1280, 0, "stream", 33.3, 29.4), (4, 1728, 8711, 3840, 0, "stream", 139.9, 126.6),
    (4, 1158, 6239, 1280, 0, "stream", 35.9, 31.5), (8, 1124, 19983, 1280, 0, "stream", 108.9, 95.8)]


@pytest.mark.parametrize("bits,m,n,k,tiled,faster,direct_us,stream_us", ABOVE_256_ROWS)
def test_direct_or_streamed_above_256_rows(ask, bits, m, n, k, tiled, faster, direct_us, stream_us):
    assert (direct_us < stream_us) == (faster == "direct")
    us = ask(bits, m, n, k, tiled, may_split=False)[2]
    assert (us["other"] < us["stream"]) == (faster == "direct"), us


def test_pipeline_or_streamed_on_odd_columns(ask):
    """Group sizes the direct-weight kernel does not take: 25.0 us on the pipeline, 30.1 streamed; 407 rows and more K
    the other way round (60.6 / 43.3), tile-major weights only streamed."""
    assert (lambda us: us["other"] < us["stream"])(ask(8, 1123, 5165, 1024, 0, False, group=32)[2])
    assert (lambda us: us["other"] > us["stream"])(ask(8, 407, 13173, 2048, 0, False, group=32)[2])
    assert ask(8, 407, 13173, 1920, 1, False)[2]["other"] > 1e20


def test_tiles_of_odd_columns_and_of_long_k(ask):
    # 4096 x 11008 at 2048 rows in 128 x 256 tiles: 164.8 us, in the 256 x 256 tiles of one table for all sizes 180.9
    assert ask(4, 2048, 4096, 11008, 0, False)[0] == 1
    # rows of an odd N begin between two 4-byte boundaries: 8.6 us a round more on 128 x 256 tiles
    even, odd = ask(4, 407, 13174, 1024, 0, False), ask(4, 407, 13173, 1024, 0, False)
    assert odd[2]["stream"] > even[2]["stream"]
    # a K split is planned only where it may be had
    assert ask(8, 256, 5120, 13824, 0, True)[1] > 1 and ask(8, 256, 5120, 13824, 0, False)[1] == 1


def test_both_layouts_get_the_same_tile_and_windows(ask):
    for bits in (4, 8):
        for m in (17, 33, 52, 99, 200, 256, 407, 1024):
            for n, k in ((1000, 8192), (4090, 8192), (4096, 11008), (5120, 5120), (6528, 1024), (22016, 4096)):
                assert ask(bits, m, n, k, 0)[:2] == ask(bits, m, n, k, 1)[:2], (bits, m, n, k)


# (bits, group, M, N, K, tile-major, the faster one, us of the register-activation kernel, of the best streamed tile and split)
UP_TO_256_ROWS = [
    (8, 128, 63, 2816, 1792, 1, "skinny", 7.1, 8.7), (8, 128, 39, 4096, 2048, 1, "skinny", 6.5, 8.9),
    (8, 128, 44, 3328, 1792, 1, "skinny", 6.2, 8.5), (8, 128, 19, 6912, 2304, 1, "skinny", 7.5, 9.7),
    (8, 128, 145, 768, 1792, 1, "skinny", 6.5, 7.8), (8, 128, 25, 3584, 2048, 0, "skinny", 5.5, 7.7),
    (4, 32, 17, 3811, 2048, 0, "skinny", 5.5, 7.4), (4, 32, 27, 3865, 2048, 1, "skinny", 5.4, 7.7),
    (8, 64, 21, 2795, 1792, 0, "skinny", 6.0, 7.5), (4, 32, 64, 8192, 1024, 0, "stream", 9.6, 5.9),
    (4, 32, 192, 2048, 2304, 0, "stream", 12.3, 8.1), (4, 32, 52, 6144, 2304, 1, "stream", 12.1, 9.0),
    (8, 128, 18, 7111, 2560, 1, "skinny", 8.1, 10.0), (4, 32, 48, 9366, 1024, 0, "stream", 10.3, 7.3),
    (4, 32, 39, 953, 1024, 1, "stream", 6.6, 5.7), (4, 128, 73, 1024, 2304, 0, "stream", 10.1, 7.4),
    (8, 32, 61, 1995, 2304, 0, "stream", 12.6, 8.1), (8, 128, 17, 1024, 13824, 1, "stream", 15.9, 11.3), (8, 128, 99, 5120, 13824, 0, "stream", 60.0, 33.0)]


@pytest.mark.parametrize("bits,group,m,n,k,tiled,faster,skinny_us,stream_us", UP_TO_256_ROWS)
def test_register_activation_kernel_or_streamed(ask, bits, group, m, n, k, tiled, faster, skinny_us, stream_us):
    assert (skinny_us < stream_us) == (faster == "skinny")
    us = ask(bits, m, n, k, tiled, group=group)[2]
    assert (us["skinny"] < us["stream"]) == (faster == "skinny"), us


def test_the_workspace_query_is_the_size_of_the_split_that_runs(ask):
    """From 17 rows on mi355x_wq_workspace_bytes answers with the plan's size where some tail's call splits K (the kernels that
    could run instead are slower for it), 0 elsewhere; a call is never short of a workspace sized by it."""
    from relax_amd import lib

    q = lib.load().mi355x_wq_workspace_bytes
    split = 0
    for bits, group in ((4, 32), (8, 128), (4, 64), (8, 32)):
        for m in (17, 33, 48, 64, 99, 128, 200, 256, 384, 512):
            for n in (1024, 2304, 5120, 5121, 9216, 22528):
                for k in (1024, 2816, 5120, 8192, 13824):
                    for tiled in (0, 1) if group in (32, 128) and (bits, group) in ((4, 32), (8, 128)) else (0,):
                        _, windows, us = ask(bits, m, n, k, tiled, group=group)
                        got, need = q(lib.make_desc(bits, group, n, k), m, tiled), ask.plan_bytes(bits, group, m, n, k)
                        assert got in (0, need) and (windows > 1 or got == 0), (bits, group, m, n, k, tiled)
                        if windows > 1 and us["stream"] < min(us["other"], us["skinny"]):
                            assert got == need > 16384, (bits, group, m, n, k, tiled)
                            split += 1
    assert split > 300


# (bits, group, M, N, K, tile, macro step of it, us with two bytes a scale request, us in pieces of eight groups)
SCALE_PIECES = [(4, 64, 20, 2304, 5632, 32, 64, 256, 8.8, 9.2), (4, 128, 95, 1545, 9728, 32, 64, 256, 11.9, 12.5), (8, 128, 87, 4608, 1536, 32, 64, 256, 6.17, 6.38),
                (8, 128, 20, 14592, 5632, 32, 64, 256, 21.4, 20.3),
                (8, 128, 256, 15360, 5120, 128, 128, 128, 47.0, 46.1), (8, 128, 99, 27648, 5120, 128, 128, 128, 47.6, 45.9),
                (4, 32, 333, 3712, 4608, 128, 256, 256, 22.2, 24.0), (4, 32, 2048, 22016, 4096, 128, 256, 256, 364.0, 358.0)]


@pytest.mark.parametrize("bits,group,m,n,k,rows,columns,macro_step,plain_us,pieces_us", SCALE_PIECES)
def test_scale_pieces_where_they_were_the_faster(ask, bits, group, m, n, k, rows, columns, macro_step, plain_us, pieces_us):
    assert bool(ask.pieces(bits, group, m, n, k, rows, columns, macro_step)) == (pieces_us < plain_us)


@pytest.mark.parametrize("bits,group,k", [(8, 128, 1152), (4, 64, 4160), (8, 256, 256)])
def test_no_scale_pieces_past_a_rows_end_or_off_the_word_grid(ask, bits, group, k):
    assert not ask.pieces(bits, group, 4096, 4096, k, 128, 128, 128)
