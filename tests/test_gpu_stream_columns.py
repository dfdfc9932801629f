"""The streamed GEMM's tiles of 96 columns at their edges, as the other tiles are tested, and a matrix whose default call takes one."""
import pytest

from oracle import c_oracle, wq_oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tests import test_gpu_stream as stream  # noqa: E402
from tests import test_gpu_stream_tail as stream_tail  # noqa: E402
from tests.test_gpu_parity import _dev, assert_close  # noqa: E402


@pytest.mark.parametrize("variant", [38, 39])  # 64 x 96, 32 x 96
@pytest.mark.parametrize("bits,m,n,k,group", [
    (4, 1, 1, 32, 32), (4, 33, 95, 1056, 32), (4, 64, 96, 1024, 32), (4, 65, 97, 256, 32), (4, 17, 290, 2304, 64), (4, 32, 191, 1152, 128),
    (8, 2, 3, 128, 128), (8, 64, 193, 384, 128), (8, 31, 96, 704, 64), (8, 100, 130, 160, 32), (8, 40, 575, 1280, 128)])
def test_at_the_edges(variant, bits, m, n, k, group):
    stream.test_every_tile_shape_at_its_edges(variant, bits, m, n, k, group)


@pytest.mark.parametrize("variant", [38, 39])
@pytest.mark.parametrize("m,n,shift", [(37, 1, (1, 0, 0)), (33, 95, (1, 1, 0)), (64, 97, (0, 1, 1)), (70, 193, (1, 1, 0)), (31, 96, (1, 0, 0))])
def test_rows_off_the_4_byte_grid_and_in_place(variant, m, n, shift):
    stream_tail.test_rows_off_the_4_byte_grid(variant, m, n, shift)


@pytest.mark.parametrize("m,variant", [(37, 38), (20, 39)])
def test_a_default_call_that_takes_one(m, variant):
    import relax_amd

    x, wq, s, g = O.make_case(m, m, 22016, 2048, 4)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    y = relax_amd.wq_matmul(dx, dw, ds, 4, g).cpu().numpy()
    assert (y == stream.run(dx, dw, ds, 4, g, variant)).all()
    rows = [0, m - 1]
    assert_close(y[rows], c_oracle.wq_matmul(x[rows], wq, s, 4, g, nthreads=8), (m, variant), ulp_fraction=0.005)
