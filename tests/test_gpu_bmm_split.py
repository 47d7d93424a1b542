"""dc_bmm's split products: depths around the 16-deep step, tiles' edges, and elements that are not
finite (whose split has NaN remainders) against float32 arithmetic."""
import numpy as np
import pytest

from tests._data import assert_f32

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (2, 127, 63, 15), (1, 129, 65, 17), (2, 128, 128, 16), (1, 64, 200, 33),
                                   (3, 260, 64, 4), (1, 132, 132, 36)])
@pytest.mark.parametrize("la,lb", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_depths_and_edges(oracle_lib, shape, la, lb):
    from densecore_amd import _native
    print(f"[case] bmm split {shape} A transposed {la} B transposed {lb}", flush=True)
    batch, m, n, k = shape
    rng = np.random.default_rng(m + n + k + la + 2 * lb)
    a, b = rng.standard_normal((batch, m, k), dtype=np.float32), rng.standard_normal((batch, k, n), dtype=np.float32)

    def operand(x, transposed):
        if not transposed:
            return torch.from_numpy(x).to(DEV)
        return torch.from_numpy(np.ascontiguousarray(x.transpose(0, 2, 1))).to(DEV).transpose(1, 2)

    got = _native._bmm(operand(a, la), operand(b, lb)).cpu().numpy()
    assert_f32(got, oracle_lib.bmm(a, b, b_k_contiguous=bool(lb)), f"bmm {shape}")


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan, 3.4e38])
def test_elements_beyond_the_split(bad):
    """One element of A: its row of C is what float32 gives, the other rows are as without it."""
    from densecore_amd import _native
    rng = np.random.default_rng(4)
    a, b = rng.standard_normal((2, 150, 40), dtype=np.float32), rng.standard_normal((2, 40, 140), dtype=np.float32)
    b[1, 7] = np.where(np.abs(b[1, 7]) < 0.1, np.float32(0.1), b[1, 7]) * 0.5
    plain = _native._bmm(torch.from_numpy(a).to(DEV), torch.from_numpy(b).to(DEV)).cpu().numpy()
    a[1, 33, 7] = bad
    got = _native._bmm(torch.from_numpy(a).to(DEV), torch.from_numpy(b).to(DEV)).cpu().numpy()
    with np.errstate(invalid="ignore", over="ignore"):
        want = (a[1, 33].astype(np.float64) @ b[1].astype(np.float64)).astype(np.float32)
    assert np.allclose(got[1, 33], want, rtol=1e-5, equal_nan=True)
    got[1, 33] = plain[1, 33]
    assert_f32(got, plain, "other rows")
