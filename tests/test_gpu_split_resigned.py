"""The streamed GEMM's shared finishing where no workgroup sees its fellows come (GEMM variant 50: it does not look): all but a tile's last to
arrive write their own parts as well, resign and leave, and the last to arrive finishes what is left."""
import pytest

from oracle import wq_oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tests.test_gpu_parity import _dev, _fused_operands  # noqa: E402


# two to seven windows on 128 x 128 tiles, two to five on 64 x 128; rows that end within a tile and within a row quad
@pytest.mark.parametrize("bits,m,n,k", [(4, 200, 5758, 11008), (8, 249, 5120, 5120), (8, 101, 7000, 9984), (8, 72, 4720, 10240), (8, 99, 5120, 13824), (8, 74, 4164, 12544),
                                        (8, 300, 5120, 13824), (8, 146, 4208, 9728), (8, 72, 5121, 13824), (8, 142, 2182, 13312), (4, 121, 3000, 13824)])
def test_every_workgroup_resigns(bits, m, n, k):
    import relax_amd
    from relax_amd import lib

    x, wq, s, g = O.make_case(m + n, m, n, k, bits)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    bias, res = (_dev(t) for t in _fused_operands(m + n, m, n))
    for tail in [{}, dict(bias=bias, activation="gelu"), dict(residual=res)] + ([dict(activation="silu_mul")] if n % 2 == 0 else []):
        seen = relax_amd.wq_matmul(dx, dw, ds, bits, g, **tail)
        for _ in range(4):  # (the counters have to be back at zero for either kind)
            resigned = relax_amd.wq_matmul(dx, dw, ds, bits, g, kernel=lib.KERNEL_GEMM, variant=50, **tail)
            again = relax_amd.wq_matmul(dx, dw, ds, bits, g, **tail)
            assert torch.equal(resigned.view(torch.int16), seen.view(torch.int16)), list(tail)
            assert torch.equal(again.view(torch.int16), seen.view(torch.int16)), list(tail)


def test_tile_major_weights():
    import relax_amd
    from relax_amd import lib

    x, wq, s, g = O.make_case(5, 99, 5120, 13824, 8)
    wt, st = relax_amd.wq_tile_weights(_dev(wq), _dev(s), 8, g)
    seen = relax_amd.wq_matmul(_dev(x), wt, st, 8, g, tiled_n=5120)
    resigned = relax_amd.wq_matmul(_dev(x), wt, st, 8, g, tiled_n=5120, kernel=lib.KERNEL_GEMM, variant=50)
    assert torch.equal(resigned.view(torch.int16), seen.view(torch.int16))


# 64 x 64 tiles, more tiles than half of the CUs, up to 16 rows, and strips
@pytest.mark.parametrize("bits,m,n,k", [(4, 37, 4096, 11008), (8, 99, 27648, 5120), (4, 12, 4096, 11008), (4, 73, 5556, 10752)])
def test_where_the_call_shares_nothing_it_does_not_apply(bits, m, n, k):
    import relax_amd
    from relax_amd import lib

    x, wq, s, g = O.make_case(6, m, n, k, bits)
    with pytest.raises(lib.WqError, match="does not apply"):
        relax_amd.wq_matmul(_dev(x), _dev(wq), _dev(s), bits, g, kernel=lib.KERNEL_GEMM, variant=50)
