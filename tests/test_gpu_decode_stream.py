"""Up to 16 rows on the streamed GEMM (long K on canonical weights): against the oracle on both sides of the rule's lines, with every
tail, and where the call has to stay with the decode kernel -- under capture, on hipStreamPerThread, gelu in place."""
import os
import subprocess
import sys

import numpy as np
import pytest

from oracle import c_oracle, wq_oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tests.test_gpu_parity import _dev, _fused_operands, assert_close  # noqa: E402

# N at the edges of one tile of 16 per CU, of one and a quarter, of two; K and rows at the edges of the lines
CASES = [(8, 6, 4097, 13824), (8, 5, 4112, 13824), (8, 10, 5120, 8192), (8, 16, 5121, 13824), (8, 10, 5440, 8192), (8, 12, 5441, 8192), (8, 16, 6145, 13824), (8, 9, 1000, 9856),
         (8, 8, 4096, 11008), (4, 16, 4090, 11008), (4, 10, 4096, 11008), (4, 11, 8192, 10752), (4, 12, 8193, 10752), (4, 9, 4100, 11008)]


@pytest.mark.parametrize("bits,m,n,k", CASES)
def test_long_k_against_the_oracle(bits, m, n, k):
    import relax_amd

    x, wq, s, g = O.make_case(m + n, m, n, k, bits)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    bias, res = _fused_operands(m + n, m, n)
    plain = relax_amd.wq_matmul(dx, dw, ds, bits, g).cpu().numpy()
    rows = [0, m // 2, m - 1]
    assert_close(plain[rows], c_oracle.wq_matmul(x[rows], wq, s, bits, g, nthreads=8), (bits, m, n, k), ulp_fraction=0.005)
    again = relax_amd.wq_matmul(dx, dw, ds, bits, g).cpu().numpy()
    assert np.array_equal(again.view(np.uint16), plain.view(np.uint16))
    for tail in (dict(bias=bias, activation="relu", residual=res), dict(bias=bias, activation="gelu"), dict(residual=res)):
        got = relax_amd.wq_matmul(dx, dw, ds, bits, g, **{a: _dev(b) if isinstance(b, np.ndarray) else b for a, b in tail.items()})
        want = O.epilogue(plain, **tail)
        assert np.array_equal(got.cpu().numpy().view(np.uint16), want.view(np.uint16)), list(tail)


def test_calls_that_stay_with_the_decode_kernel():
    """They agree with the kernel family they name; a captured call replays to the same result."""
    import relax_amd
    from relax_amd import lib

    bits, m, n, k = 8, 16, 5120, 13824
    x, wq, s, g = O.make_case(5, m, n, k, bits)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    decode = relax_amd.wq_matmul(dx, dw, ds, bits, g, kernel=lib.KERNEL_GEMV)

    class PerThread:
        cuda_stream = 2

    torch.cuda.synchronize()
    per_thread = relax_amd.wq_matmul(dx, dw, ds, bits, g, stream=PerThread)
    torch.cuda.synchronize()
    assert torch.equal(per_thread.view(torch.int16), decode.view(torch.int16))
    out, graph = torch.empty_like(decode), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        relax_amd.wq_matmul(dx, dw, ds, bits, g, out=out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        relax_amd.wq_matmul(dx, dw, ds, bits, g)
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), decode.view(torch.int16))
    res = _dev(_fused_operands(1, m, n)[1])
    y = res.clone()
    relax_amd.wq_matmul(dx, dw, ds, bits, g, activation="gelu", residual=y, out=y)
    want = relax_amd.wq_matmul(dx, dw, ds, bits, g, activation="gelu", residual=res, kernel=lib.KERNEL_GEMV)
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("streams", [9, 24, 30])
def test_as_many_streams_as_slots_and_more(streams):
    """Calls in flight on every stream at once: the bits of a call that is alone, which are the streamed kernel's, on all of them."""
    import relax_amd
    from relax_amd import lib

    x, wq, s, g = O.make_case(6, 16, 1000, 9856, 8)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    alone = relax_amd.wq_matmul(dx, dw, ds, 8, g)
    decode = relax_amd.wq_matmul(dx, dw, ds, 8, g, kernel=lib.KERNEL_GEMV)
    assert not torch.equal(alone.view(torch.int16), decode.view(torch.int16)), "the case is meant to be one of the streamed kernel's"
    handles = [torch.cuda.Stream() for _ in range(streams)]
    torch.cuda.synchronize()
    outs = [relax_amd.wq_matmul(dx, dw, ds, 8, g, stream=h, out=torch.empty_like(alone)) for _ in range(4) for h in handles]
    torch.cuda.synchronize()
    assert all(torch.equal(o.view(torch.int16), alone.view(torch.int16)) for o in outs)


@pytest.mark.parametrize("bits,m,n,k,streamed", [(4, 16, 8191, 11008, True), (4, 10, 5120, 11008, True), (8, 16, 5760, 13824, True),
                                                 (8, 16, 5120, 13824, False), (4, 12, 4096, 11008, False)])
def test_on_a_workspace_and_on_the_scratch_array(bits, m, n, k, streamed):
    """A workspace holds the decode kernel's split, and where that does not split the streamed one's: the results there have the eager
    call's bits, captured and on hipStreamPerThread as well.  The library's scratch array is as good as a workspace."""
    import relax_amd
    from relax_amd import lib

    x, wq, s, g = O.make_case(m + k, m, n, k, bits)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    res = _dev(_fused_operands(m, m, n)[1])
    need = relax_amd.wq_workspace_bytes(bits, g, n, k, m)
    assert 16384 < need <= lib.load().mi355x_wq_static_ws_bytes()
    ws = relax_amd.wq_workspace(need)
    rows = [0, m // 2, m - 1]
    for tail in ({}, dict(residual=res)):
        plain = relax_amd.wq_matmul(dx, dw, ds, bits, g, **tail)
        on_ws = relax_amd.wq_matmul(dx, dw, ds, bits, g, workspace=ws, **tail)
        torch.cuda.synchronize()
        assert torch.equal(on_ws.view(torch.int16), plain.view(torch.int16)) == streamed
        assert int(ws[:16384].view(torch.int32).abs().sum()) == 0

        class PerThread:
            cuda_stream = 2

        outs = [relax_amd.wq_matmul(dx, dw, ds, bits, g, workspace=ws, stream=PerThread, **tail)]
        torch.cuda.synchronize()
        y = torch.empty_like(plain)
        ep = lib.WqEpilogue(None, tail["residual"].data_ptr() if tail else None, lib.ACT_NONE, 0)
        lib.check(lib.load().mi355x_wq_matmul_static_ws(lib.make_desc(bits, g, n, k), dx.data_ptr(), dw.data_ptr(), ds.data_ptr(), ep, y.data_ptr(),
                                                        m, int(torch.cuda.current_stream().cuda_stream), 0))
        torch.cuda.synchronize()
        outs.append(y)
        graph, out = torch.cuda.CUDAGraph(), torch.empty_like(plain)
        with torch.cuda.graph(graph):
            relax_amd.wq_matmul(dx, dw, ds, bits, g, workspace=ws, out=out, **tail)
        for _ in range(3):
            out.zero_()
            graph.replay()
            relax_amd.wq_matmul(dx, dw, ds, bits, g, **tail)
            torch.cuda.synchronize()
            outs.append(out.clone())
        assert all(torch.equal(o.view(torch.int16), on_ws.view(torch.int16)) for o in outs)
        if not tail:
            assert_close(on_ws.cpu().numpy()[rows], c_oracle.wq_matmul(x[rows], wq, s, bits, g, nthreads=8), (bits, m, n, k), ulp_fraction=0.005)
    # one that is too small: as without
    small = relax_amd.wq_matmul(dx, dw, ds, bits, g, workspace=ws[:need - 16])
    assert torch.equal(small.view(torch.int16), relax_amd.wq_matmul(dx, dw, ds, bits, g).view(torch.int16))


FIRST_LAUNCH_UNDER_CAPTURE = """
import torch, relax_amd
from relax_amd import lib
from oracle import wq_oracle as O
import numpy as np
x, wq, s, g = O.make_case(5, 16, 5120, 13824, 8)
dx, dw, ds = (torch.from_numpy(a.view(np.int32) if a.dtype == np.uint32 else a).cuda() for a in (x, wq, s))
relax_amd.wq_matmul(dx, dw, ds, 8, g)
torch.cuda.synchronize()
out, graph = torch.empty((16, 5120), dtype=torch.float16, device="cuda"), torch.cuda.CUDAGraph()
with torch.cuda.graph(graph):
    relax_amd.wq_matmul(dx, dw, ds, 8, g, out=out)
for _ in range(3):
    out.zero_()
    graph.replay()
    torch.cuda.synchronize()
    got = out.clone()
    want = relax_amd.wq_matmul(dx, dw, ds, 8, g, kernel=lib.KERNEL_GEMV)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
"""


def test_one_eager_call_is_enough_before_a_capture():
    """The eager call launches the streamed kernel, the captured one the decode kernel: its first launch in the process is the captured
    one, so this needs a process of its own."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", FIRST_LAUNCH_UNDER_CAPTURE], cwd=root, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
