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


def _us(f):
    f()
    start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    times = []
    for _ in range(5):
        start.record()
        for _ in range(10):
            f()
        end.record()
        end.synchronize()
        times.append(start.elapsed_time(end) * 100)
    return min(times)


def test_nan_rows_are_final():
    """Rows of NaN (the softmax of a fully masked query) make their own rows of C NaN and no others,
    beside elements the split cannot hold too, and are not computed twice: 1.6 times the plain product
    where every tile has one (16 when its tile was computed again in float32)."""
    from densecore_amd import _native
    rng = np.random.default_rng(11)
    a, b = rng.standard_normal((256, 512, 512), dtype=np.float32), rng.standard_normal((256, 512, 64), dtype=np.float32)
    ta, tb = torch.from_numpy(a).to(DEV), torch.from_numpy(b).to(DEV)
    plain = _native._bmm(ta, tb)
    before = _us(lambda: _native._bmm(ta, tb))
    ta[:, 5::128] = float("nan")
    got = _native._bmm(ta, tb)
    assert torch.isnan(got[:, 5::128]).all()
    got[:, 5::128] = plain[:, 5::128]
    assert torch.equal(got, plain)
    after = _us(lambda: _native._bmm(ta, tb))
    print(f"  {before:.0f} us, with NaN rows {after:.0f} us", flush=True)
    assert after < 5 * before
    # A large element in the tile of a NaN row: its row is what float32 gives.
    ta[3, 40, 7] = 3.4e38
    b[3, 7] *= 0.25
    tb[3] = torch.from_numpy(b[3]).to(DEV)
    got = _native._bmm(ta, tb)[3].cpu().numpy()
    a[3, 40, 7] = 3.4e38
    want = (a[3, 40].astype(np.float64) @ b[3].astype(np.float64)).astype(np.float32)
    assert np.allclose(got[40], want, rtol=1e-5) and np.isnan(got[5::128]).all() and np.isfinite(np.delete(got, np.s_[5::128], 0)).all()


@pytest.mark.parametrize("k", [1, 2, 3, 5, 15, 17, 34])
@pytest.mark.parametrize("la,lb", [(0, 0), (1, 0), (0, 1), (1, 1), (2, 0), (1, 2)])
@pytest.mark.parametrize("m,n,shift", [(1, 1, 0), (67, 130, 1), (129, 63, 3), (66, 65, 2)])
def test_ragged_operands(oracle_lib, m, n, k, la, lb, shift):
    """Rows that are no whole 16-byte parts, at every offset from them, along k (0), along m or n (1) and
    with no unit stride (2): elements past a row's end, which hold NaN here, are not read into it."""
    from densecore_amd import _native
    print(f"[case] bmm ragged {m}x{n}x{k} A {la} B {lb} shift {shift}", flush=True)
    rng = np.random.default_rng(m + n + k + shift)
    batch = 3
    a, b = rng.standard_normal((batch, m, k), dtype=np.float32), rng.standard_normal((batch, k, n), dtype=np.float32)

    def operand(x, along):  # x is (batch, rows, k)
        if along == 1:
            x = x.transpose(0, 2, 1)
        step = 2 if along == 2 else 1
        pad = torch.full((batch, x.shape[1], shift + step * x.shape[2] + 5), float("nan"), device=DEV)
        view = pad[:, :, shift:shift + step * x.shape[2]:step]
        view.copy_(torch.from_numpy(np.ascontiguousarray(x)))
        return view.transpose(1, 2) if along == 1 else view

    got = _native._bmm(operand(a, la), operand(b.transpose(0, 2, 1), lb).transpose(1, 2)).cpu().numpy()
    assert_f32(got, oracle_lib.bmm(a, b, b_k_contiguous=lb != 1), f"bmm {m}x{n}x{k}")
