"""The decode kernel's ways of reading weights (weight_reads in wq_gemm_plan.cpp): pairs of lanes that share whole lines and swap
what they hold of each other's rows, and the same without keeping the lines.  A build reads so only on tiles of 14 and more rows, so the
10-row tiles of the same build, whose lanes read their own chunks, have to give the same bits."""
import numpy as np
import pytest

from oracle import c_oracle, wq_oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

OWN = 1015  # 10-row tiles, one workgroup of eight wavefronts per CU, two-chunk super steps


def _problem(bits, n, k, group, m, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if bits == 4:
        wq = torch.randint(-(1 << 31), (1 << 31) - 1, (n, k // 8), dtype=torch.int32, device="cuda", generator=gen)
    else:
        wq = torch.randint(-127, 128, (n, k), dtype=torch.int8, device="cuda", generator=gen).view(torch.int32)
    mean = 1.0 / ((4.63 if bits == 4 else 73.6) * k ** 0.5)
    s = torch.rand((n, k // group), device="cuda", generator=gen).add_(0.5).mul_(mean).half()
    return torch.randn((m, k), dtype=torch.float16, device="cuda", generator=gen), wq, s


def _same(a, b):
    return torch.equal(a.view(torch.int16), b.view(torch.int16))


def _against_the_oracle(y, x, wq, s, bits, group):
    """The columns at the edges of the first and the last tiles."""
    n = wq.shape[0]
    cols = sorted({c for c in (0, 1, 13, 14, 15, 16, 17, n // 2, n - 17, n - 16, n - 15, n - 2, n - 1) if 0 <= c < n})
    want = c_oracle.wq_matmul(x.cpu().numpy(), wq[cols].cpu().numpy().view(np.uint32), s[cols].cpu().numpy(), bits, group, nthreads=8)
    got = y[:, cols].cpu().numpy().astype(np.float64)
    assert np.all(np.abs(got - want.astype(np.float64)) <= 1e-2 + 1e-2 * np.abs(want.astype(np.float64)))


# (bits, N, K, group, rows): above 10 MB in pairs of lanes, above 64 MB (int4: 85 MB, 1 and 2 rows) non-temporally; N that leaves a last tile
# of one row, of an odd and of an even number of rows; K in one piece and in phases, whose length, and with it the order of the sums, goes by the
# tiles per workgroup: there N gives each one tile of either height
CASES = [(8, 2561, 4096, 128, 1), (8, 2573, 4096, 64, 3), (8, 2574, 4096, 32, 8), (8, 5003, 2048, 16, 16), (8, 1309, 8192, 128, 16),
         (8, 1303, 8192, 64, 9), (8, 2447, 4224, 32, 2), (8, 8193, 8192, 128, 1), (8, 8190, 8192, 64, 5), (8, 8201, 8192, 32, 6),
         (8, 2559, 26112, 32, 16), (8, 2546, 26112, 128, 9),
         (4, 20755, 8192, 32, 1), (4, 20756, 8192, 64, 2), (4, 20769, 8192, 128, 2), (4, 20755, 8192, 32, 3)]


@pytest.mark.parametrize("bits,n,k,group,m", CASES)
def test_whole_lines_and_own_chunks_have_the_same_bits(bits, n, k, group, m):
    import relax_amd
    from relax_amd import lib

    x, wq, s = _problem(bits, n, k, group, m, n + m)
    own = relax_amd.wq_matmul(x, wq, s, bits, group, kernel=lib.KERNEL_GEMV, variant=OWN)
    for tile_rows in (14, 15, 16):
        y = relax_amd.wq_matmul(x, wq, s, bits, group, kernel=lib.KERNEL_GEMV, variant=tile_rows * 100 + 15)
        assert _same(y, own), (tile_rows, int((y != own).sum()))
    _against_the_oracle(own, x, wq, s, bits, group)


@pytest.mark.parametrize("bits,n,k,group,m", [(8, 2562, 4096, 128, 1), (8, 2590, 4096, 32, 8), (8, 1306, 8192, 64, 16), (8, 8194, 8192, 128, 3),
                                              (4, 20758, 8192, 32, 2), (4, 20790, 8192, 128, 1)])
def test_a_gate_row_and_its_up_row_as_a_pair(bits, n, k, group, m):
    """The gated tail's tiles interleave the two halves of the weight rows: a pair of lanes reads from both."""
    import relax_amd
    from relax_amd import lib

    x, wq, s = _problem(bits, n, k, group, m, n + m)
    kw = dict(kernel=lib.KERNEL_GEMV, variant=1615)
    h = relax_amd.wq_matmul(x, wq, s, bits, group, kernel=lib.KERNEL_GEMV, variant=OWN)
    y = relax_amd.wq_matmul(x, wq, s, bits, group, activation="silu_mul", **kw)
    want = O.epilogue(h.cpu().numpy(), activation="silu_mul")
    assert np.array_equal(y.cpu().numpy().view(np.uint16), want.view(np.uint16))


@pytest.mark.parametrize("bits,n,k,m", [(8, 8193, 8192, 2), (8, 8200, 8192, 5), (8, 2550, 26112, 16), (4, 20755, 8192, 1), (4, 20766, 8192, 3)])
def test_tile_major_weights_that_are_not_kept(bits, n, k, m):
    import relax_amd
    from relax_amd import lib

    group = 32 if bits == 4 else 128
    x, wq, s = _problem(bits, n, k, group, m, n + m)
    own = relax_amd.wq_matmul(x, wq, s, bits, group, kernel=lib.KERNEL_GEMV, variant=OWN)
    wt, st = relax_amd.wq_tile_weights(wq, s, bits, group)
    y = relax_amd.wq_matmul(x, wt, st, bits, group, tiled_n=n, kernel=lib.KERNEL_GEMV, variant=1615)
    assert _same(y, own)
