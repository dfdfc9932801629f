"""The strip kernel (wq_gemm_strip.hip): every build at the edges of its row blocks, slices, column tiles and steps of K, both layouts and
the tails, against the oracle; and what must not reach a neighbour."""
import numpy as np
import pytest

from oracle import c_oracle, wq_oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tests.test_gpu_parity import _dev, _fused_operands, assert_close, assert_fused  # noqa: E402
from tests.test_gpu_stream import run  # noqa: E402

VARIANTS = [41, 42, 43, 44]  # one to four column tiles of 16 a workgroup


def fits(bits, m, variant):
    slices = -(-m // 64)
    blocks = max(3, -(-(-(-m // slices)) // 8))
    blocks = 8 if blocks == 7 else blocks
    return 8 * (blocks * 2048 + (variant - 40) * 2048 + 1024) <= 160 * 1024


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("bits,m,n,k", [
    (4, 1, 128, 256), (4, 17, 129, 2048), (4, 24, 257, 2304), (4, 25, 130, 1024), (4, 33, 191, 4096), (4, 40, 2001, 1280), (4, 41, 144, 2560),
    (4, 49, 300, 512), (4, 64, 128, 4352), (4, 65, 258, 2304), (4, 129, 200, 1024), (4, 256, 136, 1280),
    (8, 2, 131, 256), (8, 17, 128, 1280), (8, 32, 515, 2304), (8, 37, 190, 2048), (8, 48, 1001, 768), (8, 57, 128, 3328), (8, 72, 250, 1024),
    (8, 200, 128, 1280)])
def test_every_build_at_its_edges(variant, bits, m, n, k):
    import relax_amd

    x, wq, s, g = O.make_case(2000 + m + n + k, m, n, k, bits)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    if not fits(bits, m, variant):
        with pytest.raises(Exception, match="does not apply"):
            run(dx, dw, ds, bits, g, variant)
        return
    want = c_oracle.wq_matmul(x, wq, s, bits, g, nthreads=8)
    plain = run(dx, dw, ds, bits, g, variant)
    assert_close(plain, want, (variant, bits, m, n, k))
    bias, res = _fused_operands(m + n, m, n)
    assert_fused(run(dx, dw, ds, bits, g, variant, bias=_dev(bias), activation="relu", residual=_dev(res)), plain, want, bias, "relu", res, (variant, bits, m, n, k))
    gelu, tail = run(dx, dw, ds, bits, g, variant, bias=_dev(bias), activation="gelu"), c_oracle.epilogue(plain, bias, "gelu")
    assert (gelu.view(np.uint16) != tail.view(np.uint16)).sum() <= max(1, gelu.size // 1000)
    if n % 2 == 0:
        gated = run(dx, dw, ds, bits, g, variant, activation="silu_mul")
        tail = c_oracle.epilogue(plain, activation="silu_mul")
        assert (gated.view(np.uint16) != tail.view(np.uint16)).sum() <= max(1, gated.size // 1000)
    if k % (256 if bits == 4 else 128) == 0:
        wt, st = relax_amd.wq_tile_weights(dw, ds, bits, g)
        assert np.array_equal(run(dx, wt, st, bits, g, variant, tiled_n=n).view(np.uint16), plain.view(np.uint16)), "tile-major"


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("k", [8448, 8704, 16640])
def test_int8_scales_past_a_wavefronts_first_piece(variant, k):
    """A wavefront's share of K is more than the eight steps of a piece of scales: the bits of the tile-major build, which asks for them
    step by step (and the oracle, at the bound of the other calls of long K)."""
    import relax_amd

    x, wq, s, g = O.make_case(k, 33, 160, k, 8)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    plain = run(dx, dw, ds, 8, g, variant)
    wt, st = relax_amd.wq_tile_weights(dw, ds, 8, g)
    assert np.array_equal(run(dx, wt, st, 8, g, variant, tiled_n=160).view(np.uint16), plain.view(np.uint16))
    assert_close(plain, c_oracle.wq_matmul(x, wq, s, 8, g, nthreads=8), (variant, k), ulp_fraction=0.005)


@pytest.mark.parametrize("bits,m,n,k,variant", [(4, 37, 200, 2304, 43), (4, 70, 144, 1024, 41), (8, 20, 130, 1280, 44)])
def test_what_is_not_finite_stays_in_its_row_and_column(bits, m, n, k, variant):
    """Rows and columns meet in LDS rows, fragments and slices: an infinite or NaN activation changes its row only, an infinite or NaN
    scale its column only, and the outputs past the end keep what they held."""
    x, wq, s, g = O.make_case(7, m, n, k, bits)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    plain = run(dx, dw, ds, bits, g, variant).view(np.uint16)
    rows, cols = [0, m // 2, m - 1], [0, 17, n - 1]
    bx, bs = dx.clone(), ds.clone()
    bx[rows[0], 5], bx[rows[1], k - 1], bx[rows[2], k // 2] = float("inf"), float("nan"), float("-inf")
    bs[cols[0], 0], bs[cols[1], -1], bs[cols[2], -1] = float("nan"), float("inf"), float("nan")
    keep_r, keep_c = np.setdiff1d(np.arange(m), rows), np.setdiff1d(np.arange(n), cols)
    assert np.array_equal(run(bx, dw, ds, bits, g, variant).view(np.uint16)[keep_r], plain[keep_r])
    assert np.array_equal(run(dx, dw, bs, bits, g, variant).view(np.uint16)[:, keep_c], plain[:, keep_c])
    guarded = torch.full((m * n + 64,), 3.0, dtype=torch.float16, device="cuda")
    run(dx, dw, ds, bits, g, variant, out=guarded[32:32 + m * n].view(m, n))
    assert (guarded[:32] == 3).all() and (guarded[32 + m * n:] == 3).all()
    assert np.array_equal(guarded[32:32 + m * n].view(m, n).cpu().numpy().view(np.uint16), plain)


@pytest.mark.parametrize("variant,bits,m,n,k", [(v, *c) for c in ((4, 20, 145, 1280), (4, 70, 262, 512), (8, 33, 131, 1024), (8, 130, 128, 768))
                                                for v in VARIANTS if fits(c[0], c[1], v)])
def test_the_residual_in_the_output_buffer(variant, bits, m, n, k):
    """The residual is read before the K loop, by the lane that writes the element."""
    import relax_amd

    x, wq, s, g = O.make_case(3000 + m + n, m, n, k, bits)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    bias, res = _fused_operands(m + n, m, n)
    layouts = [(dw, ds, {}), (*relax_amd.wq_tile_weights(dw, ds, bits, g), dict(tiled_n=n))]
    for w_, s_, kw in layouts:
        plain = run(dx, w_, s_, bits, g, variant, **kw)
        for tail, want in (({}, {}), (dict(bias=_dev(bias), activation="relu"), dict(bias=bias, activation="relu"))):
            y = _dev(res)
            run(dx, w_, s_, bits, g, variant, out=y, residual=y, **tail, **kw)
            assert np.array_equal(y.cpu().numpy().view(np.uint16), O.epilogue(plain, residual=res, **want).view(np.uint16)), (variant, list(kw), list(tail))


@pytest.mark.parametrize("bits,m,n,k", [(4, 37, 4096, 4096), (4, 20, 8064, 2048), (8, 128, 1024, 2048), (4, 25, 8544, 5632)])
def test_default_calls_that_take_it(bits, m, n, k):
    """The same bits with a workspace, on other streams, and from every replay of a graph."""
    import relax_amd

    x, wq, s, g = O.make_case(m + n, m, n, k, bits)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    y = relax_amd.wq_matmul(dx, dw, ds, bits, g)
    assert any(torch.equal(y, torch.from_numpy(run(dx, dw, ds, bits, g, v)).cuda()) for v in VARIANTS if fits(bits, m, v))
    rows = [0, m // 2, m - 1]
    assert_close(y.cpu().numpy()[rows], c_oracle.wq_matmul(x[rows], wq, s, bits, g, nthreads=8), (bits, m, n, k), ulp_fraction=0.005)
    assert torch.equal(relax_amd.wq_matmul(dx, dw, ds, bits, g, workspace=relax_amd.wq_workspace(1 << 25)), y)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        other = relax_amd.wq_matmul(dx, dw, ds, bits, g)
    torch.cuda.synchronize()
    assert torch.equal(other, y)
    graph, out = torch.cuda.CUDAGraph(), torch.empty_like(y)
    with torch.cuda.graph(graph):
        relax_amd.wq_matmul(dx, dw, ds, bits, g, out=out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        assert torch.equal(out, y)
