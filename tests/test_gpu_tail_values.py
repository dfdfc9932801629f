"""The tails' functions on every float16 value: erf, exp and the reciprocal are evaluated by short forms in float32 (wq_device.h)
that have to give the float16 values of the exact functions for all inputs, so results are compared bit for bit."""
import numpy as np
import pytest

from oracle import wq_oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

ALL = np.arange(65536, dtype=np.uint16).view(np.float16)
K, GROUP = 256, 128


def _same(got, want):
    got, want = got.reshape(-1), want.reshape(-1)
    both_nan = np.isnan(got) & np.isnan(want)
    off = (got.view(np.uint16) != want.view(np.uint16)) & ~both_nan
    assert not off.any(), (int(off.sum()), got[off][:4], want[off][:4])


@pytest.mark.parametrize("m", [1, 20, 80])
def test_gelu_of_every_value(m):
    """Activations of zero, so that the bias is what gelu sees: a column for each of the 65536 values."""
    import relax_amd

    n = ALL.size
    x = torch.zeros((m, K), dtype=torch.float16, device="cuda")
    wq = torch.zeros((n, K // 4), dtype=torch.int32, device="cuda")
    s = torch.ones((n, K // GROUP), dtype=torch.float16, device="cuda")
    y = relax_amd.wq_matmul(x, wq, s, 8, GROUP, bias=torch.from_numpy(ALL.copy()).cuda(), activation="gelu")
    with np.errstate(all="ignore"):
        want = O.epilogue(np.zeros((1, n), np.float16), ALL, "gelu", None)
    y = y.cpu().numpy()
    for row in (0, m - 1):
        _same(y[row], want)


@pytest.mark.parametrize("rows", [16, 1000, None])
def test_silu_of_every_finite_value(rows):
    """A row of activations for each finite value: the gate reads it with weight one, the up column a constant."""
    import relax_amd

    values = ALL[np.isfinite(ALL) & (ALL.view(np.uint16) != 0x8000)]  # (a sum of products is never -0 here)
    x = np.zeros((values.size, K), np.float16)
    x[:, 0], x[:, 1] = values, 1.0
    w = np.zeros((2, K), np.int8)
    w[0, 0] = w[1, 1] = 1
    xd = torch.from_numpy(x).cuda()
    wq, s = torch.from_numpy(w.view(np.int32)).cuda(), torch.ones((2, K // GROUP), dtype=torch.float16, device="cuda")
    with np.errstate(all="ignore"):
        want = O.epilogue(np.stack([values, np.ones_like(values)], axis=1), activation="silu_mul")
    step = rows or values.size
    starts = range(0, values.size, step) if step >= 1000 else range(0, values.size - step, step * 97)
    for at in starts:
        got = relax_amd.wq_matmul(xd[at:at + step], wq, s, 8, GROUP, activation="silu_mul").cpu().numpy()
        _same(got, want[at:at + step])
