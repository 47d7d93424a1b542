"""Float32 operands that bf16 rounds to infinity or that are not finite: the split products have NaN
there and the kernels redo what they reach in float32, on every schedule and under every mask.

One element of a row is 3.4e38 and the dimension it meets in the other operand is zero, so float32
arithmetic stays finite: every result is compared with the oracle's, the one dimension the element
reaches relative to its size.
"""
import ctypes

import numpy as np
import pytest

from tests._data import assert_f32, assert_f32_nan

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"
BIG = np.float32(3.4e38)

CASES = [  # B, H, Hkv, L, S, E, causal, mask, stream-K ranges
    (1, 2, 2, 70, 200, 64, False, None, True), (2, 4, 2, 150, 150, 64, True, None, True), (2, 2, 1, 130, 100, 32, True, None, True),
    (1, 2, 2, 33, 300, 40, False, "full", True), (2, 2, 2, 140, 140, 64, True, "full", True), (3, 4, 2, 70, 300, 64, False, "pad", True),
    (3, 2, 2, 45, 200, 36, False, "pad", True), (20, 16, 16, 40, 257, 64, False, None, False), (18, 16, 16, 130, 257, 32, True, None, False),
    (15, 16, 16, 40, 257, 64, False, "pad", False), (1, 2, 2, 65, 100, 63, False, None, True), (1, 4, 2, 150, 150, 80, True, None, True),
]


def _t(x):
    return torch.from_numpy(np.ascontiguousarray(x)).to(DEV)


def _inputs(B, H, Hkv, L, S, E, mask, seed):
    rng = np.random.default_rng(seed)
    x = {n: rng.standard_normal((B, h, m, E), dtype=np.float32) for n, h, m in (("q", H, L), ("k", Hkv, S), ("v", Hkv, S), ("g", H, L))}
    m = None
    if mask == "full":
        m = rng.standard_normal((B, H, L, S), dtype=np.float32)
        m[rng.random((B, H, L, S)) < 0.3] = -np.inf
    elif mask == "pad":
        m = np.zeros((B, 1, 1, S), np.float32)
        for b in range(B):
            m[b, ..., S * (b + 1) // B:] = -np.inf
    return x, m


def _backward(x, out, lse, causal, m, least):
    from densecore_amd import _lib
    q, k, v, g = (x[n] for n in "qkvg")
    B, H, L, E = q.shape
    ms = (0, 0, 0) if m is None else m.stride()[:3]
    d = _lib.Desc(B, H, k.shape[1], L, k.shape[2], E, int(causal), 0, 0.0, _lib.DC_F32, 0, *ms)
    Lb = _lib.lib()
    size = (B * H * L * 4 + 255) // 256 * 256 if least else int(Lb.dc_sdpa_bwd_workspace_size(ctypes.byref(d)))
    ws = torch.empty(size, dtype=torch.uint8, device=DEV)
    got = [torch.full_like(t, 3.0) for t in (q, k, v)]
    p = lambda t: None if t is None else t.data_ptr()
    _lib.check(Lb.dc_sdpa_bwd(ctypes.byref(d), p(g), p(q), p(k), p(v), p(out), p(lse), p(m), *(p(t) for t in got), p(ws), size,
                              torch.cuda.current_stream().cuda_stream))
    return got


# The operand with the large element, the one whose same dim is zero, and the gradient that takes it.
WHERE = [("q", "k", 1), ("k", "q", 0), ("v", "g", None), ("g", "v", 2)]


@pytest.mark.parametrize("least", [False, True])
@pytest.mark.parametrize("bad,zero,reached", WHERE)
@pytest.mark.parametrize("B,H,Hkv,L,S,E,causal,mask,streamk", CASES)
def test_backward_beyond_the_split(oracle_lib, B, H, Hkv, L, S, E, causal, mask, streamk, bad, zero, reached, least):
    from densecore_amd import _native
    print(f"[case] not finite B{B} H{H} Hkv{Hkv} L{L} S{S} E{E} causal={causal} mask={mask} {bad} least={least}", flush=True)
    x, m = _inputs(B, H, Hkv, L, S, E, mask, L + S + E)
    dim = E - 3
    x[zero][..., dim] = 0
    for b in {0, B - 1}:
        x[bad][b, -1, x[bad].shape[2] // 3, dim] = BIG
    full = None if m is None else np.ascontiguousarray(np.broadcast_to(m, (B, H, L, S)))
    out, lse = oracle_lib.forward(x["q"], x["k"], x["v"], causal, None, full)
    ref = oracle_lib.backward(x["g"], x["q"], x["k"], x["v"], out, lse, causal, None, full)
    tx = {n: _t(a) for n, a in x.items()}
    tm = None if m is None else _t(m).expand(B, H, L, S)
    if not least and E <= 64:
        ranges = _native._schedule(True, tx["q"], tx["k"], tx["v"], causal, None, tm)["streamk_ranges"]
        assert (ranges > 0) == streamk
    got = _backward(tx, _t(out), _t(lse), causal, tm, least)
    for i, (name, a, r) in enumerate(zip(("dq", "dk", "dv"), got, ref)):
        a = a.cpu().numpy()
        if i == reached:
            # one term of 1e30 and more, or none: its probability times a difference of dot products
            # of unit normals, each held to 2e-5
            assert np.allclose(a[..., dim] / BIG, r[..., dim] / BIG, rtol=1e-4, atol=2e-5), name
            a, r = np.delete(a, dim, -1), np.delete(r, dim, -1)
        assert_f32(a, r, name)


@pytest.mark.parametrize("least", [False, True])
@pytest.mark.parametrize("where,bad", [("g", np.inf), ("g", np.nan), ("q", np.nan), ("k", np.inf), ("v", np.nan)])
@pytest.mark.parametrize("B,H,Hkv,L,S,E", [(1, 2, 2, 70, 200, 64), (2, 4, 2, 64, 300, 40), (20, 16, 16, 40, 257, 64)])
def test_backward_not_finite(oracle_lib, B, H, Hkv, L, S, E, where, bad, least):
    """NaN and infinities where the oracle has them (no mask, not causal: every tile sees every pair)."""
    print(f"[case] not finite B{B} H{H} Hkv{Hkv} L{L} S{S} E{E} {where}={bad} least={least}", flush=True)
    x, _ = _inputs(B, H, Hkv, L, S, E, None, L + S + E)
    x[where][B - 1, 1, 30, 5] = bad
    with np.errstate(all="ignore"):
        out, lse = oracle_lib.forward(x["q"], x["k"], x["v"], False)
        ref = oracle_lib.backward(x["g"], x["q"], x["k"], x["v"], out, lse, False)
    got = _backward({n: _t(a) for n, a in x.items()}, _t(out), _t(lse), False, None, least)
    for name, a, r in zip(("dq", "dk", "dv"), got, ref):
        a = a.cpu().numpy()
        assert (a[np.isinf(r)] == r[np.isinf(r)]).all(), name
        assert_f32_nan(np.where(np.isinf(r), 0, a), np.where(np.isinf(r), 0, r), name)
