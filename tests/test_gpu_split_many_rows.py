"""Calls of more than 256 rows without a workspace: which of them split K on the library's memory, and what they do where that is taken."""
import threading

import pytest

from oracle import c_oracle, wq_oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tests.test_gpu_parity import _dev, assert_close  # noqa: E402
from tests.test_gpu_stream import PerThread  # noqa: E402


def same_bits(a, b):
    return torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("bits,m,n,k", [(8, 266, 896, 2560), (8, 299, 1280, 4864), (8, 351, 2048, 8448), (4, 831, 1406, 6400)])
def test_a_call_that_the_split_would_slow_down_runs_whole(bits, m, n, k, tiled):
    """As on hipStreamPerThread and under capture; with a workspace it is split as before."""
    import relax_amd

    x, wq, s, g = O.make_case(m + n, m, n, k, bits)
    dx, dw, ds, kw = _dev(x), _dev(wq), _dev(s), {}
    if tiled:
        dw, ds = relax_amd.wq_tile_weights(dw, ds, bits, g)
        kw["tiled_n"] = n
    whole = relax_amd.wq_matmul(dx, dw, ds, bits, g, stream=PerThread, **kw)
    torch.cuda.synchronize()
    assert same_bits(relax_amd.wq_matmul(dx, dw, ds, bits, g, **kw), whole)
    need = relax_amd.wq_workspace_bytes(bits, g, n, k, m)
    assert need > 16384
    split = relax_amd.wq_matmul(dx, dw, ds, bits, g, workspace=relax_amd.wq_workspace(need), **kw)
    assert not same_bits(split, whole)
    rows = [0, m // 2, m - 1]
    want = c_oracle.wq_matmul(x[rows], wq, s, bits, g, nthreads=8)
    for y in (whole, split):
        assert_close(y.cpu().numpy()[rows], want, (bits, m, n, k), ulp_fraction=0.005)


# 128 x 128 tiles, 64 x 128 and 64 x 64
SPLIT = [(8, 621, 1654, 9216), (4, 342, 1536, 13568), (4, 350, 512, 6400)]


@pytest.mark.parametrize("bits,m,n,k", SPLIT)
def test_a_ninth_busy_stream_has_the_bits_of_the_others(bits, m, n, k):
    """Eight streams own the eight workspaces and are busy with products ahead of their calls; the ninth's calls walk the windows in turn."""
    import relax_amd

    x, wq, s, g = O.make_case(m + n, m, n, k, bits)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    alone = relax_amd.wq_matmul(dx, dw, ds, bits, g)
    big = torch.randn(8192, 8192, device="cuda", dtype=torch.float16)
    big @ big
    streams = [torch.cuda.Stream() for _ in range(10)]
    outs = [torch.empty_like(alone) for _ in range(30)]
    products = [torch.empty_like(big) for _ in range(8)]
    torch.cuda.synchronize()
    for i, stream in enumerate(streams[:8]):
        with torch.cuda.stream(stream):
            for _ in range(4):
                torch.mm(big, big, out=products[i])
            relax_amd.wq_matmul(dx, dw, ds, bits, g, out=outs[i])
    for i in range(8, 30):
        relax_amd.wq_matmul(dx, dw, ds, bits, g, stream=streams[8 + i % 2], out=outs[i])
    torch.cuda.synchronize()
    assert all(same_bits(y, alone) for y in outs)


@pytest.mark.parametrize("bits,m,n,k", SPLIT)
def test_more_threads_and_streams_than_workspaces(bits, m, n, k):
    import relax_amd

    x, wq, s, g = O.make_case(m + n, m, n, k, bits)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    alone = relax_amd.wq_matmul(dx, dw, ds, bits, g)
    torch.cuda.synchronize()
    outs = [[] for _ in range(12)]

    def worker(mine):
        stream = torch.cuda.Stream()
        for _ in range(5):
            for _ in range(3):
                mine.append(relax_amd.wq_matmul(dx, dw, ds, bits, g, stream=stream, out=torch.empty_like(alone)))
            stream.synchronize()

    threads = [threading.Thread(target=worker, args=(o,)) for o in outs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert all(same_bits(y, alone) for mine in outs for y in mine)
