"""The streamed GEMM (wq_gemm_stream.hip): every tile shape at the edges of its tiles, stages and macro steps, every group size it
takes, both layouts, the tails, and the split of K on a workspace and on the library's own slots, against the oracle."""
import numpy as np
import pytest

from oracle import c_oracle, wq_oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tests.test_gpu_parity import _dev, _fused_operands, assert_close, assert_fused  # noqa: E402

VARIANTS = [31, 32, 33, 34, 35, 36, 37]  # 128 x 256, 128 x 128, 256 x 256, 64 x 128, 64 x 64, 32 x 64, 32 x 128


def run(x, wq, s, bits, g, variant, **kw):
    import relax_amd
    from relax_amd import lib

    y = relax_amd.wq_matmul(x, wq, s, bits, g, kernel=lib.KERNEL_GEMM, variant=variant, **kw)
    torch.cuda.synchronize()
    return y.cpu().numpy()


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("bits,m,n,k,group", [
    (4, 1, 1, 32, 32), (4, 33, 65, 96, 32), (4, 65, 130, 256, 32), (4, 257, 257, 1056, 32), (4, 200, 136, 1024, 32), (4, 129, 64, 2304, 64),
    (4, 70, 301, 1152, 128), (4, 40, 128, 1536, 256), (8, 2, 3, 128, 128), (8, 64, 127, 384, 128), (8, 130, 258, 1280, 128),
    (8, 100, 40, 160, 32), (8, 31, 515, 704, 64), (8, 256, 256, 512, 256)])
def test_every_tile_shape_at_its_edges(variant, bits, m, n, k, group):
    import relax_amd

    x, wq, s, g = O.make_case(1000 + m + n + k, m, n, k, bits, group)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    want = c_oracle.wq_matmul(x, wq, s, bits, g, nthreads=8)
    plain = run(dx, dw, ds, bits, g, variant)
    assert_close(plain, want, (variant, bits, m, n, k, group))
    bias, res = _fused_operands(m + n, m, n)
    fused = run(dx, dw, ds, bits, g, variant, bias=_dev(bias), activation="relu", residual=_dev(res))
    assert_fused(fused, plain, want, bias, "relu", res, (variant, bits, m, n, k, group))
    if n % 2 == 0:
        gated = run(dx, dw, ds, bits, g, variant, activation="silu_mul")
        tail = c_oracle.epilogue(plain, activation="silu_mul")
        assert (gated.view(np.uint16) != tail.view(np.uint16)).sum() <= max(1, gated.size // 1000)
    if group == (32 if bits == 4 else 128) and k % (256 if bits == 4 else 128) == 0:
        wt, st = relax_amd.wq_tile_weights(dw, ds, bits, g)
        assert np.array_equal(run(dx, wt, st, bits, g, variant, tiled_n=n).view(np.uint16), plain.view(np.uint16)), "tile-major"


@pytest.mark.parametrize("bits,m,n,k", [(4, 40, 1000, 11008), (4, 200, 2048, 4352), (8, 99, 1022, 13824), (8, 256, 513, 5120)])
def test_k_split_on_the_librarys_slots_on_a_workspace_and_under_capture(bits, m, n, k):
    """Calls that bring no workspace split on a slot of the library's: same bits as on a caller's workspace, on two
    streams at once as on one; under capture (no slot) the unsplit call's result, equal in every replay."""
    import relax_amd

    x, wq, s, g = O.make_case(m + n, m, n, k, bits)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    y = relax_amd.wq_matmul(dx, dw, ds, bits, g)
    ws = relax_amd.wq_workspace(1 << 25)
    on_ws = relax_amd.wq_matmul(dx, dw, ds, bits, g, workspace=ws)
    torch.cuda.synchronize()
    assert int(ws[:16384].view(torch.int32).abs().sum()) == 0
    assert torch.equal(y.view(torch.int16), on_ws.view(torch.int16))
    rows = [0, m // 2, m - 1]
    want = c_oracle.wq_matmul(x[rows], wq, s, bits, g, nthreads=8)
    assert_close(y.cpu().numpy()[rows], want, (bits, m, n, k), ulp_fraction=0.005)
    streams, outs = [torch.cuda.Stream() for _ in range(2)], []
    for _ in range(20):
        for st in streams:
            with torch.cuda.stream(st):
                outs.append(relax_amd.wq_matmul(dx, dw, ds, bits, g))
    torch.cuda.synchronize()
    assert all(torch.equal(o.view(torch.int16), y.view(torch.int16)) for o in outs)
    graph, out = torch.cuda.CUDAGraph(), torch.empty_like(y)
    with torch.cuda.graph(graph):
        relax_amd.wq_matmul(dx, dw, ds, bits, g, out=out)
    first = None
    for _ in range(3):
        out.zero_()
        graph.replay()
        relax_amd.wq_matmul(dx, dw, ds, bits, g)
        torch.cuda.synchronize()
        first = out.clone() if first is None else first
        assert torch.equal(out, first)
    assert_close(first.cpu().numpy()[rows], want, ("captured", bits, m, n, k), ulp_fraction=0.005)


def test_more_threads_and_streams_than_slots():
    """Twelve streams, a thread each, for eight slots that pass from idle streams to others: every result is the split call's
    or, without a slot, the unsplit one's."""
    import threading

    import relax_amd

    x, wq, s, g = O.make_case(3, 40, 1000, 11008, 4)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    split = relax_amd.wq_matmul(dx, dw, ds, 4, g)
    graph, unsplit = torch.cuda.CUDAGraph(), torch.empty_like(split)
    with torch.cuda.graph(graph):
        relax_amd.wq_matmul(dx, dw, ds, 4, g, out=unsplit)
    graph.replay()
    torch.cuda.synchronize()
    outs = [[] for _ in range(12)]

    def worker(mine):
        stream = torch.cuda.Stream()
        for burst in range(10):
            for _ in range(3):
                mine.append(relax_amd.wq_matmul(dx, dw, ds, 4, g, stream=stream, out=torch.empty_like(split)))
            stream.synchronize()

    threads = [threading.Thread(target=worker, args=(o,)) for o in outs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert all(torch.equal(y, split) or torch.equal(y, unsplit) for mine in outs for y in mine)
