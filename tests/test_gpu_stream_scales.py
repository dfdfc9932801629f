"""The streamed GEMM's scales in pieces of eight groups: rows of few groups, pieces that end past a row or the buffer, macro steps and K
windows that begin within a piece, against the oracle and against the tile-major layout, which has none; and beside them the rows that keep
two bytes a request (an odd number of groups, K that is no multiple of 256)."""
import numpy as np
import pytest

from oracle import c_oracle, wq_oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tests import test_gpu_stream as stream  # noqa: E402
from tests.test_gpu_parity import _dev, assert_close  # noqa: E402


@pytest.mark.parametrize("variant", [31, 32, 33, 34, 35, 36, 37, 38, 39])
@pytest.mark.parametrize("bits,m,n,k,group", [(8, 20, 67, 256, 128), (8, 65, 130, 2304, 128), (8, 33, 97, 1280, 32), (8, 33, 97, 1536, 256), (8, 20, 40, 1280, 256),
                                              (4, 40, 129, 2816, 128), (4, 20, 70, 1536, 64), (4, 33, 65, 1280, 128), (4, 17, 60, 768, 256)])
def test_pieces_at_their_edges(variant, bits, m, n, k, group):
    stream.test_every_tile_shape_at_its_edges(variant, bits, m, n, k, group)


@pytest.mark.parametrize("variant,k", [(31, 512), (31, 1280), (31, 2816), (33, 512), (33, 2816)])
def test_pieces_of_one_macro_step(variant, k):
    """Enough tiles of 256 columns to fill the chip: the bits of the tile-major layout, which has no pieces, and of a smaller call, which has
    none on 128 x 256 tiles (31).  There a piece is one macro step, and from 1280 of K on its place in the ring of two has been used before; on 256 x 256 tiles (33) it is two."""
    import relax_amd

    m, n = 1030, 6146
    x, wq, s, g = O.make_case(5, m, n, k, 4)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    plain = stream.run(dx, dw, ds, 4, g, variant)
    wt, st = relax_amd.wq_tile_weights(dw, ds, 4, g)
    assert np.array_equal(stream.run(dx, wt, st, 4, g, variant, tiled_n=n).view(np.uint16), plain.view(np.uint16))
    assert np.array_equal(stream.run(dx[:64].contiguous(), dw, ds, 4, g, variant).view(np.uint16), plain[:64].view(np.uint16))
    rows = [0, 63, 64, m - 1]
    assert_close(plain[rows], c_oracle.wq_matmul(x[rows], wq, s, 4, g, nthreads=8), variant, ulp_fraction=0.005)


@pytest.mark.parametrize("bits,m,n,k,group,variant", [(8, 40, 130, 1280, 128, 35), (8, 130, 130, 2304, 128, 32), (4, 40, 130, 1280, 128, 34)])
def test_what_is_not_finite_stays_in_its_column(bits, m, n, k, group, variant):
    x, wq, s, g = O.make_case(9, m, n, k, bits, group)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    plain = stream.run(dx, dw, ds, bits, g, variant).view(np.uint16)
    cols, bad = [0, 64, n - 1], ds.clone()
    bad[0, 0], bad[64, -1], bad[n - 1, 1] = float("nan"), float("inf"), float("nan")
    keep = np.setdiff1d(np.arange(n), cols)
    assert np.array_equal(stream.run(dx, dw, bad, bits, g, variant).view(np.uint16)[:, keep], plain[:, keep])


@pytest.mark.parametrize("bits,m,n,k,group", [(8, 99, 1022, 13824, 128), (8, 200, 1000, 8192, 64), (4, 200, 1000, 11008, 128), (8, 40, 1000, 6912, 32)])
def test_windows_that_begin_within_a_piece(bits, m, n, k, group):
    import relax_amd

    x, wq, s, g = O.make_case(m, m, n, k, bits, group)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    torch.cuda.synchronize()
    need = relax_amd.wq_workspace_bytes(bits, g, n, k, m)
    assert need > 16384, "the case is meant to split"
    ws = relax_amd.wq_workspace(need)
    on_ws = relax_amd.wq_matmul(dx, dw, ds, bits, g, workspace=ws)
    assert int(ws.count_nonzero()) > 0, "the split ran on the workspace"
    rows = [0, m // 2, m - 1]
    assert_close(on_ws.cpu().numpy()[rows], c_oracle.wq_matmul(x[rows], wq, s, bits, g, nthreads=8), (bits, m, n, k), ulp_fraction=0.005)
    assert torch.equal(relax_amd.wq_matmul(dx, dw, ds, bits, g).view(torch.int16), on_ws.view(torch.int16))
    # hipStreamPerThread has no workspace of the library's: the windows run one after the other
    class PerThread:
        cuda_stream = 2

    serial = relax_amd.wq_matmul(dx, dw, ds, bits, g, stream=PerThread)
    torch.cuda.synchronize()
    assert torch.equal(serial.view(torch.int16), on_ws.view(torch.int16))
