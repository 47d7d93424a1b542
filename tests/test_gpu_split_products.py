"""Float32 attention whose products run on the bf16 matrix cores (each operand split in three).

Edges of the 32-key and 128-key tiles, of the 32-query steps, of the head dims (zero-padded, rows that
are not whole 16-byte parts, 65 to 127 forward), of key-padding masks (dead tiles inside and at the
end, a batch without any key, masks that differ between heads) and of the schedules, against the
oracle at the float32 bar; and operands that are not finite, whose split has NaN remainders, against
plain float32 arithmetic.
"""
import numpy as np
import pytest

from tests._data import assert_f32, assert_f32_nan

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"

CASES = [  # B, H, Hkv, L, S, E, causal, mask
    (1, 1, 1, 1, 1, 64, False, None), (1, 2, 1, 31, 33, 16, False, None), (2, 2, 2, 129, 127, 64, True, None),
    (1, 2, 2, 160, 160, 63, True, None), (1, 2, 2, 97, 256, 72, False, None), (1, 2, 1, 200, 130, 100, True, None),
    (1, 2, 2, 65, 65, 127, True, None), (40, 16, 16, 128, 160, 64, True, None), (24, 16, 8, 96, 288, 32, False, None),
    (3, 4, 2, 70, 320, 64, False, "pad"), (3, 4, 4, 257, 300, 36, False, "holes"), (2, 4, 4, 130, 140, 64, False, "heads"),
    (2, 2, 2, 64, 1056, 64, False, "holes"), (2, 3, 3, 90, 150, 64, False, "full"), (2, 3, 3, 150, 150, 44, True, "full"),
    (2, 2, 2, 100, 260, 90, False, "pad"),
]


def _t(x):
    return torch.from_numpy(np.ascontiguousarray(x)).to(DEV)


def _mask(kind, rng, B, H, L, S):
    if kind is None:
        return None
    if kind == "full":
        m = rng.standard_normal((B, H, L, S), dtype=np.float32)
        m[rng.random((B, H, L, S)) < 0.3] = -np.inf
        m[0, 0, L // 2] = -np.inf
        return m
    m = np.zeros((B, H if kind == "heads" else 1, 1, S), np.float32)
    if kind == "pad":
        for b in range(B):
            m[b, ..., S * b // B:] = -np.inf  # batch 0 has no key at all
    elif kind == "holes":
        m[..., S // 4:S // 4 + 70] = -np.inf
        m[-1, ..., 5:] = rng.standard_normal(S - 5)
    else:
        for h in range(H):
            m[:, h, :, 10 + 30 * h:] = -np.inf
    return m


@pytest.mark.parametrize("B,H,Hkv,L,S,E,causal,mask", CASES)
def test_split_products(oracle_lib, B, H, Hkv, L, S, E, causal, mask):
    from densecore_amd import _native
    print(f"[case] split products B{B} H{H} Hkv{Hkv} L{L} S{S} E{E} causal={causal} mask={mask}", flush=True)
    rng = np.random.default_rng(B + H + L + S + E)
    q, g = (rng.standard_normal((B, H, L, E), dtype=np.float32) for _ in range(2))
    k, v = (rng.standard_normal((B, Hkv, S, E), dtype=np.float32) for _ in range(2))
    m = _mask(mask, rng, B, H, L, S)
    full = None if m is None else np.ascontiguousarray(np.broadcast_to(m, (B, H, L, S)))
    tm = None if m is None else _t(m).expand(B, H, L, S)
    ref_o, ref_l = oracle_lib.forward(q, k, v, causal, None, full)
    out, lse = _native._flash_attention(_t(q), _t(k), _t(v), causal, None, tm)
    assert_f32(out.cpu().numpy(), ref_o, "out")
    assert_f32(lse.cpu().numpy(), ref_l, "lse")
    ref = oracle_lib.backward(g, q, k, v, ref_o, ref_l, causal, None, full)
    got = _native._flash_attention_backward(_t(g), _t(q), _t(k), _t(v), _t(ref_o), _t(ref_l), causal, None, tm)
    for name, a, b in zip(("dq", "dk", "dv"), got, ref):
        assert_f32(a.cpu().numpy(), b, name)


@pytest.mark.parametrize("E,S", [(64, 200), (40, 33), (96, 130)])
@pytest.mark.parametrize("bad", [np.inf, 3.4e38])
def test_values_beyond_the_split(E, S, bad):
    """An infinite value, or a finite one that bf16 rounds to infinity, reaches its own output dim
    only, as in float32 arithmetic: the others stay what they are without it."""
    from densecore_amd import _native
    rng = np.random.default_rng(E + S)
    q = rng.standard_normal((1, 2, 45, E), dtype=np.float32)
    k, v = (rng.standard_normal((1, 2, S, E), dtype=np.float32) for _ in range(2))
    plain, _ = _native._flash_attention(_t(q), _t(k), _t(v), False)
    p = np.exp(np.einsum("bhld,bhsd->bhls", q.astype(np.float64), k) / np.sqrt(E))
    p /= p.sum(-1, keepdims=True)
    v[0, 1, S - 1, 5] = bad
    out, _ = _native._flash_attention(_t(q), _t(k), _t(v), False)
    out, plain = out.cpu().numpy(), plain.cpu().numpy()
    assert_f32(np.delete(out, 5, -1), np.delete(plain, 5, -1), "other dims")
    assert_f32(out[0, 0], plain[0, 0], "other head")
    want = np.float32(np.inf) if np.isinf(bad) else (p[0, 1, :, S - 1] * np.float64(np.float32(bad))).astype(np.float32)
    assert np.allclose(out[0, 1, :, 5], want, rtol=1e-5)


def test_key_of_infinite_score():
    """A key whose scores are -inf for some queries and +inf for others: the former see the other
    keys, the latter are NaN."""
    from densecore_amd import _native
    rng = np.random.default_rng(8)
    q, k, v = (rng.standard_normal((1, 1, n, 64), dtype=np.float32) for n in (64, 96, 96))
    q[0, 0, :, 3] = np.where(np.arange(64) % 2, 1, -1)
    keep = np.arange(96) != 40
    ref, _ = _native._flash_attention(_t(q), _t(k[:, :, keep]), _t(v[:, :, keep]), False)
    k[0, 0, 40, 3] = np.inf
    out, _ = _native._flash_attention(_t(q), _t(k), _t(v), False)
    out, ref = out.cpu().numpy()[0, 0], ref.cpu().numpy()[0, 0]
    assert_f32(out[::2], ref[::2], "queries of -inf score")
    assert np.isnan(out[1::2]).all()


def test_infinite_output_gradient():
    """dO = inf in one dim of one query: dV's dim is +inf for every key, its other dims as without."""
    from densecore_amd import _native
    rng = np.random.default_rng(9)
    q, k, v, g = (rng.standard_normal((1, 2, 160, 64), dtype=np.float32) for _ in range(4))
    t = [_t(x) for x in (q, k, v)]
    out, lse = _native._flash_attention(*t, False)
    _, _, dv0 = _native._flash_attention_backward(_t(g), *t, out, lse, False)
    g[0, 1, 70, 9] = np.inf
    _, _, dv = _native._flash_attention_backward(_t(g), *t, out, lse, False)
    dv, dv0 = dv.cpu().numpy(), dv0.cpu().numpy()
    assert np.isposinf(dv[0, 1, :, 9]).all()
    assert_f32(np.delete(dv[0, 1], 9, -1), np.delete(dv0[0, 1], 9, -1), "other dims")
    assert_f32(dv[0, 0], dv0[0, 0], "other head")


@pytest.mark.parametrize("E,causal,mask", [(64, True, None), (40, False, "pad"), (33, False, None), (80, True, "full")])
def test_nan_is_final(oracle_lib, E, causal, mask):
    """NaN in one key, one value and one query: NaN where the oracle has it, the bar elsewhere, in a
    multiple of the time (121 times when the rows a NaN reaches were computed again in float32, now 1.3);
    with an element beyond the split beside them too."""
    from densecore_amd import _native
    print(f"[case] NaN operands E{E} causal={causal} mask={mask}", flush=True)
    rng = np.random.default_rng(E)
    B, H, L = 2, 3, 300
    q, k, v = (rng.standard_normal((B, H, L, E), dtype=np.float32) for _ in range(3))
    m = _mask(mask, rng, B, H, L, L)
    if mask == "pad":
        m[:] = 0
        m[1, ..., 200:] = -np.inf
    full = None if m is None else np.ascontiguousarray(np.broadcast_to(m, (B, H, L, L)))
    tm = None if m is None else _t(m).expand(B, H, L, L)
    q[0, 1, 7, 3] = k[0, 2, 150, 1] = v[1, 0, 20, 2] = np.nan
    for beyond in (False, True):
        if beyond:
            v[0, 1, 9, 5] = 3e38
        with np.errstate(all="ignore"):
            ref_o, ref_l = oracle_lib.forward(q, k, v, causal, None, full)
        out, lse = _native._flash_attention(_t(q), _t(k), _t(v), causal, None, tm)
        out, lse = out.cpu().numpy(), lse.cpu().numpy()
        if beyond:  # relative to the element's size
            assert np.allclose(out[0, 1, :, 5] / 3e38, ref_o[0, 1, :, 5] / 3e38, rtol=1e-4, atol=2e-5, equal_nan=True)
            out, ref_o = np.delete(out, 5, -1), np.delete(ref_o, 5, -1)
        assert_f32_nan(out, ref_o, "out")
        assert_f32_nan(lse, ref_l, "lse")


def test_nan_takes_no_longer():
    from densecore_amd import _native
    gen = torch.Generator(device=DEV).manual_seed(2)
    q, k, v = (torch.randn(8, 12, 1024, 64, generator=gen, device=DEV) for _ in range(3))

    def us():
        _native._flash_attention(q, k, v, True)
        times = []
        for _ in range(4):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            _native._flash_attention(q, k, v, True)
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end) * 1e3)
        return min(times)

    plain = us()
    k[:, :, 5] = float("nan")
    after = us()
    print(f"  {plain:.0f} us, with NaN {after:.0f} us", flush=True)
    assert after < 10 * plain


@pytest.mark.parametrize("exponent", [-60, -100])
def test_small_magnitudes(exponent):
    """The parts of a value of 2^-110 and above are bf16 numbers, subnormal ones among them, which the
    matrix cores do not flush: V, dO and a product's operand scaled down by a power of two give the
    scaled results, as far from float64 as unscaled ones.  (Below, what a part loses is under 2^-133; dS
    is smaller than dO by the probabilities, so dQ and dK are held at the larger scale.)"""
    from densecore_amd import _native
    rng = np.random.default_rng(7)
    scale = np.float32(2.0 ** exponent)
    q, k, v, g = (rng.standard_normal((1, 2, 200, 64), dtype=np.float32) for _ in range(4))
    x64 = [x.astype(np.float64) for x in (q, k, v, g)]
    p = np.einsum("bhle,bhse->bhls", x64[0], x64[1]) / 8
    p = np.exp(p - p.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    o64 = p @ x64[2]
    dp = np.einsum("bhle,bhse->bhls", x64[3], x64[2])
    ds = p * (dp - (x64[3] * o64).sum(-1, keepdims=True)) / 8
    want = {"out": o64, "dq": ds @ x64[1], "dk": np.einsum("bhls,bhle->bhse", ds, x64[0]),
            "dv": np.einsum("bhls,bhle->bhse", p, x64[3]), "bmm": np.einsum("bhle,bhse->bhls", x64[2], x64[1])[0]}

    def errors(s):
        out, lse = _native._flash_attention(_t(q), _t(k), _t(v), False)
        got = {"out": _native._flash_attention(_t(q), _t(k), _t(v * s), False)[0]}
        grads = _native._flash_attention_backward(_t(g * s), _t(q), _t(k), _t(v), out, lse, False)
        got.update(zip(("dq", "dk", "dv"), grads))
        got["bmm"] = _native._bmm(_t((v * s)[0]), _t(k[0]).transpose(1, 2))
        return {n: np.linalg.norm(a.cpu().numpy().astype(np.float64) / s - want[n]) / np.linalg.norm(want[n]) for n, a in got.items()}

    plain, small = errors(np.float32(1)), errors(scale)
    print(f"  {plain}\n  {small}", flush=True)
    for n in want:
        if exponent < -90 and n in ("dq", "dk"):
            continue
        assert small[n] <= 1.05 * plain[n], n
