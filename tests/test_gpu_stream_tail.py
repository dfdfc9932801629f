"""Outputs of the streamed GEMM whose rows do not begin on 4-byte boundaries: odd N at the edges of a wavefront's 64 columns,
and outputs, residuals and biases at odd multiples of two bytes.  The tail is float16 arithmetic on the plain output, so it is
compared bit for bit; the plain output against the oracle."""
import numpy as np
import pytest

from oracle import c_oracle, wq_oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tests.test_gpu_parity import _dev, _fused_operands, assert_close  # noqa: E402


def at(a, halves):
    """The array on the device, `halves` float16 behind a 16-byte boundary, between guards."""
    flat = torch.full((a.size + 64,), 7.0, dtype=torch.float16, device="cuda")
    view = flat[16 + halves:16 + halves + a.size].view(a.shape)
    view.copy_(torch.from_numpy(a))
    return view, flat


@pytest.mark.parametrize("variant", [31, 32, 33, 34, 35, 36, 37])
@pytest.mark.parametrize("m,n", [(37, 1), (5, 2), (33, 3), (70, 63), (64, 65), (129, 66), (31, 127), (100, 257), (260, 131)])
@pytest.mark.parametrize("shift", [(0, 0, 0), (1, 0, 0), (0, 1, 1), (1, 1, 0)])
def test_rows_off_the_4_byte_grid(variant, m, n, shift):
    import relax_amd
    from relax_amd import lib

    bits = 4 if (m + n) % 2 else 8
    x, wq, s, g = O.make_case(77 + m + n, m, n, 256, bits)
    dx, dw, ds = _dev(x), _dev(wq), _dev(s)
    bias, res = _fused_operands(m + n, m, n)
    oy, ob, orr = shift
    kw = dict(kernel=lib.KERNEL_GEMM, variant=variant)
    plain = relax_amd.wq_matmul(dx, dw, ds, bits, g, **kw).cpu().numpy()
    assert_close(plain, c_oracle.wq_matmul(x, wq, s, bits, g, nthreads=8), (variant, m, n))
    db, dr = at(bias, ob)[0], at(res, orr)[0]
    tails = [({}, {}), (dict(bias=db), dict(bias=bias)), (dict(residual=dr), dict(residual=res)),
             (dict(bias=db, activation="relu", residual=dr), dict(bias=bias, activation="relu", residual=res)),
             (dict(bias=db, activation="gelu"), dict(bias=bias, activation="gelu")),
             (dict(activation="gelu", residual=dr), dict(activation="gelu", residual=res))]
    for given, want in tails:
        y, flat = at(np.zeros((m, n), np.float16), oy)
        relax_amd.wq_matmul(dx, dw, ds, bits, g, out=y, **given, **kw)
        got = y.cpu().numpy()
        assert np.array_equal(got.view(np.uint16), O.epilogue(plain, **want).view(np.uint16)), (variant, m, n, shift, list(given))
        guards = torch.cat([flat[:16 + oy], flat[16 + oy + m * n:]])
        assert bool((guards == 7.0).all()), "written outside the output"
    # in place: the residual is the output
    y, _ = at(res, oy)
    relax_amd.wq_matmul(dx, dw, ds, bits, g, out=y, residual=y, **kw)
    assert np.array_equal(y.cpu().numpy().view(np.uint16), O.epilogue(plain, residual=res).view(np.uint16)), "in place"
