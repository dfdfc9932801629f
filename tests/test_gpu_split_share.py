"""The streamed GEMM's split on tiles of 128 columns, whose windows share the finishing of a tile: rows that end within a tile and within a
row quad, two to eight windows, the tails, and workgroups whose fellows come late because other streams have the chip."""
import pytest

from oracle import c_oracle, wq_oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tests.test_gpu_parity import _dev, _fused_operands, assert_close  # noqa: E402
from tests.test_gpu_stream import PerThread  # noqa: E402


@pytest.mark.parametrize("bits,m,n,k", [(8, 99, 5120, 13824), (8, 72, 5121, 13824), (8, 130, 4100, 13824), (8, 249, 5120, 5120), (8, 200, 2050, 12288),
                                        (8, 101, 7000, 9984), (4, 121, 3000, 13824), (4, 180, 3378, 12288), (4, 238, 4186, 12288), (4, 200, 5758, 11008)])
def test_split_on_memory_and_one_window_after_the_other(bits, m, n, k):
    import relax_amd

    x, wq, s, g = O.make_case(m + n, m, n, k, bits)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    bias, res = (_dev(t) for t in _fused_operands(m + n, m, n))
    need = relax_amd.wq_workspace_bytes(bits, g, n, k, m)
    assert need > 16384, "the case is meant to split"
    space = relax_amd.wq_workspace(need)
    rows = [0, m // 2, m - 1]
    tails = [{}, dict(bias=bias, activation="gelu"), dict(residual=res)] + ([dict(activation="silu_mul")] if n % 2 == 0 else [])
    for tail in tails:
        serial = relax_amd.wq_matmul(dx, dw, ds, bits, g, stream=PerThread, **tail)
        torch.cuda.synchronize()
        for _ in range(3):
            assert torch.equal(relax_amd.wq_matmul(dx, dw, ds, bits, g, **tail).view(torch.int16), serial.view(torch.int16)), list(tail)
            assert torch.equal(relax_amd.wq_matmul(dx, dw, ds, bits, g, workspace=space, **tail).view(torch.int16), serial.view(torch.int16)), list(tail)
        assert int(space[:16384].view(torch.int32).abs().sum()) == 0, "counters are back at zero"
        if not tail:
            assert_close(serial.cpu().numpy()[rows], c_oracle.wq_matmul(x[rows], wq, s, bits, g, nthreads=8), (bits, m, n, k), ulp_fraction=0.005)


def test_workgroups_that_come_late():
    """Six streams whose calls together have several times as many workgroups as the chip has room for, beside products that take it for
    longer than a workgroup waits: whoever finishes a part, the bits are those of a call that is alone."""
    import relax_amd

    cases = [(8, 99, 5120, 13824), (8, 250, 5120, 5120), (4, 128, 2816, 7680)]
    operands, alone = [], []
    for bits, m, n, k in cases:
        x, wq, s, g = O.make_case(m, m, n, k, bits)
        operands.append((_dev(x), _dev(wq), _dev(s), bits, g))
        alone.append(relax_amd.wq_matmul(*operands[-1]))
    big = torch.randn(4096, 4096, device="cuda", dtype=torch.float16)
    torch.cuda.synchronize()
    streams, outs = [torch.cuda.Stream() for _ in range(6)], []
    side = torch.cuda.Stream()
    for _ in range(8):
        with torch.cuda.stream(side):
            big @ big
        for i, stream in enumerate(streams):
            outs.append((i % 3, relax_amd.wq_matmul(*operands[i % 3], stream=stream, out=torch.empty_like(alone[i % 3]))))
    torch.cuda.synchronize()
    assert all(torch.equal(y.view(torch.int16), alone[i].view(torch.int16)) for i, y in outs)


@pytest.mark.parametrize("bits,m,n,k", [(4, 512, 4096, 11008), (8, 300, 5120, 13824), (8, 257, 1001, 9216), (4, 1024, 2048, 8192), (4, 385, 640, 12800)])
def test_more_than_256_rows_split_on_the_librarys_memory(bits, m, n, k):
    """Without a workspace the bits of the split on one; captured, and on hipStreamPerThread, the unsplit call's."""
    import relax_amd

    x, wq, s, g = O.make_case(m + n, m, n, k, bits)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    res = _dev(_fused_operands(m + n, m, n)[1])
    need = relax_amd.wq_workspace_bytes(bits, g, n, k, m)
    assert need > 16384, "the case is meant to split"
    space = relax_amd.wq_workspace(need)
    rows = [0, m // 2, m - 1]
    want = c_oracle.wq_matmul(x[rows], wq, s, bits, g, nthreads=8)
    for tail in ({}, dict(residual=res)):
        split = relax_amd.wq_matmul(dx, dw, ds, bits, g, workspace=space, **tail)
        for stream in (None, torch.cuda.Stream()):
            torch.cuda.synchronize()
            y = relax_amd.wq_matmul(dx, dw, ds, bits, g, stream=stream, **tail)
            torch.cuda.synchronize()
            assert torch.equal(y.view(torch.int16), split.view(torch.int16)), list(tail)
        whole = relax_amd.wq_matmul(dx, dw, ds, bits, g, stream=PerThread, **tail)
        torch.cuda.synchronize()
        captured, graph = torch.empty_like(whole), torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            relax_amd.wq_matmul(dx, dw, ds, bits, g, out=captured, **tail)
        for _ in range(3):
            captured.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(captured.view(torch.int16), whole.view(torch.int16)), list(tail)
        if not tail:
            assert_close(split.cpu().numpy()[rows], want, (bits, m, n, k), ulp_fraction=0.005)
            assert_close(whole.cpu().numpy()[rows], want, (bits, m, n, k), ulp_fraction=0.005)
