"""Gradients of keys that a padding mask hides from every query, under operands that are not finite.

The reference visits such keys: their probability is exp(-inf - lse) = 0, so they get zeros, and NaN
where 0 meets a NaN or infinite element of dO, Q or lse, whichever tile they lie in.  The float32
backward skips groups of 32 masked keys and tiles of 128 only where that is exact.
"""
import ctypes

import numpy as np
import pytest

from tests._data import assert_f32_nan

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _t(x):
    return torch.from_numpy(np.ascontiguousarray(x)).to(DEV)


def _backward(q, k, v, g, out, lse, causal, m, workspace):
    """dq, dk, dv through the C ABI with the full workspace, or what dsum alone needs, or one that
    holds a part of the batches at a time."""
    from densecore_amd import _lib, _native
    B, H, L, E = q.shape
    Hkv, S = k.shape[1], k.shape[2]
    d = _lib.Desc(B, H, Hkv, L, S, E, int(causal), 0, 0.0, _lib.DC_F32, 0, m.stride(0), m.stride(1), m.stride(2))
    Lb = _lib.lib()
    full, least = int(Lb.dc_sdpa_bwd_workspace_size(ctypes.byref(d))), (B * H * L * 4 + 255) // 256 * 256
    size = {"full": full, "least": least, "pieces": least + (full - least) * 2 // 3}[workspace]
    ws = torch.empty(size, dtype=torch.uint8, device=DEV)
    dq, dk, dv = (torch.full_like(x, 3.0) for x in (q, k, v))
    p = lambda x: x.data_ptr()
    _lib.check(Lb.dc_sdpa_bwd(ctypes.byref(d), p(g), p(q), p(k), p(v), p(out), p(lse), p(m), p(dq), p(dk), p(dv), p(ws),
                              size, torch.cuda.current_stream().cuda_stream))
    return dq, dk, dv


# Where the bad element goes: a query row, seen by every key of its head, hidden ones among them; or a
# hidden key.  Lengths 40 and 300 of 420: closed groups in an open tile, and closed tiles.
BAD = [(None, 0.0), ("g", np.nan), ("g", np.inf), ("q", np.nan), ("lse", np.nan), ("q", 1e30), ("k", np.nan), ("v", np.inf), ("k", 1e30)]


@pytest.mark.parametrize("workspace", ["full", "pieces", "least"])
@pytest.mark.parametrize("where,bad", BAD)
@pytest.mark.parametrize("E,causal,H,Hkv", [(64, False, 2, 2), (40, True, 4, 2)])
def test_hidden_keys(oracle_lib, E, causal, H, Hkv, where, bad, workspace):
    print(f"[case] hidden keys E{E} causal={causal} H{H} Hkv{Hkv} {where}={bad} workspace={workspace}", flush=True)
    rng = np.random.default_rng(E)
    B, L, S = 3, 420 if causal else 70, 420
    row = L - 1 if causal else 37  # causal: a query past every key
    q, g = (rng.standard_normal((B, H, L, E), dtype=np.float32) for _ in range(2))
    k, v = (rng.standard_normal((B, Hkv, S, E), dtype=np.float32) for _ in range(2))
    m = np.zeros((B, 1, 1, S), np.float32)
    for b, n in enumerate((40, 300, 0)):  # the last text has no key at all
        m[b, ..., n:] = -np.inf
    full = np.ascontiguousarray(np.broadcast_to(m, (B, H, L, S)))
    out, lse = oracle_lib.forward(q, k, v, causal, None, full)
    lse = lse.copy()
    if where in ("g", "q"):
        {"g": g, "q": q}[where][1, 1, row, 3] = bad
    elif where == "lse":
        lse[0, 1, row] = bad
    elif where is not None:
        {"k": k, "v": v}[where][0, Hkv - 1, 400, 3] = bad
    with np.errstate(all="ignore"):
        ref = oracle_lib.backward(g, q, k, v, out, lse, causal, None, full)
    tm = _t(m).expand(B, H, L, S)
    got = _backward(*(_t(x) for x in (q, k, v, g, out, lse)), causal, tm, workspace)
    for name, a, b in zip(("dq", "dk", "dv"), got, ref):
        a = a.cpu().numpy()
        if causal and where in ("k", "v"):
            continue  # a hidden key past the diagonal: which tiles meet it is each implementation's
        assert (a[np.isinf(b)] == b[np.isinf(b)]).all(), name
        a, b = (np.where(np.isinf(b), 0, x) for x in (a, b))
        big = np.abs(b) > 1e6  # 1e30 in q or k: relative to its own size
        assert np.allclose(a[big], b[big], rtol=1e-4), name
        assert_f32_nan(np.where(big, 0, a), np.where(big, 0, b), name)
