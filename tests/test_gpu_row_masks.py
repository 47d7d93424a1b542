"""bf16 attention under masks that do not depend on the query, and the fp16 copies' one-launch form.

Edges of the row-mask kernels: tiles and halves of tiles with no open key, a batch without any, more
than 64 tiles of 64 keys (the live tiles are found 64 at a time) with a gap of a whole such window,
masks that differ between heads, finite mask values, causal, head counts below and above the dealt
order's 32 and not a multiple of 8, each kernel head dim, rows that are not whole 16-byte parts.  The
copies: slabs at and one vector past what one workgroup holds (65536 elements).
"""
import numpy as np
import pytest

from tests._data import assert_bf16, bf16_round

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"

CASES = [  # B, H, Hkv, L, S, E, causal, mask
    (3, 4, 2, 70, 320, 64, False, "pad"), (3, 11, 11, 130, 200, 64, False, "pad"), (5, 8, 4, 129, 129, 128, True, "pad"),
    (2, 4, 4, 100, 97, 64, False, "heads"), (2, 4, 2, 140, 200, 32, False, "heads"), (1, 2, 2, 33, 8300, 64, False, "window"),
    (2, 2, 2, 65, 300, 40, False, "holes"), (2, 2, 2, 90, 200, 44, True, "holes"), (2, 2, 2, 70, 190, 256, False, "holes"),
    (1, 1, 1, 1, 2, 64, False, "holes"), (1, 2, 1, 1024, 1024, 64, True, None), (1, 2, 2, 1025, 1025, 64, True, None),
]


def _mask(kind, rng, B, H, S):
    if kind is None:
        return None
    m = np.zeros((B, H if kind == "heads" else 1, 1, S), np.float32)
    if kind == "pad":
        for b in range(B):
            m[b, ..., S * b // B:] = -np.inf  # batch 0 has no key at all
    elif kind == "holes":
        m[..., S // 4:S // 4 + 70] = -np.inf
        m[-1, ..., S // 2:] = rng.standard_normal(S - S // 2)
    elif kind == "window":
        m[..., 40:8260] = -np.inf  # tiles 1 to 128: the window of tiles 64 to 127 is all dead
    else:
        for h in range(H):
            m[:, h, :, 10 + 30 * h:] = -np.inf
    return m


@pytest.mark.parametrize("B,H,Hkv,L,S,E,causal,mask", CASES)
def test_row_mask(oracle_lib, B, H, Hkv, L, S, E, causal, mask):
    from densecore_amd import _native
    print(f"[case] row mask B{B} H{H} Hkv{Hkv} L{L} S{S} E{E} causal={causal} mask={mask}", flush=True)
    rng = np.random.default_rng(B + H + L + S + E)
    q, g = (bf16_round(rng.standard_normal((B, H, L, E), dtype=np.float32)) for _ in range(2))
    k, v = (bf16_round(rng.standard_normal((B, Hkv, S, E), dtype=np.float32)) for _ in range(2))
    m = _mask(mask, rng, B, H, S)
    full = None if m is None else np.ascontiguousarray(np.broadcast_to(m, (B, H, L, S)))
    tm = None if m is None else torch.from_numpy(m).to(DEV).expand(B, H, L, S)
    tq, tk, tv, tg = (torch.from_numpy(x).to(DEV, torch.bfloat16) for x in (q, k, v, g))
    ref_o, ref_l = oracle_lib.forward(q, k, v, causal, None, full)
    out, lse = _native._flash_attention(tq, tk, tv, causal, None, tm)
    o, l = out.float().cpu().numpy(), lse.cpu().numpy()
    assert_bf16(o, ref_o, "out")
    assert_bf16(l, ref_l, "lse")
    got = _native._flash_attention_backward(tg, tq, tk, tv, out, lse, causal, None, tm)
    ref = oracle_lib.backward(g, q, k, v, o, l, causal, None, full)
    for name, a, b in zip(("dq", "dk", "dv"), got, ref):
        assert_bf16(a.float().cpu().numpy(), b, name)


def test_masked_tile_garbage():
    """Padding keys of a wholly masked tile may hold NaN: forward and dQ never visit them."""
    from densecore_amd import _native
    print("[case] row mask, NaN in masked tiles", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(5)
    q, k, v, g = (torch.randn(2, 2, 128, 64, generator=gen, device=DEV).bfloat16() for _ in range(4))
    m = torch.zeros(2, 1, 1, 128, device=DEV)
    m[..., 32:] = float("-inf")
    tm = m.expand(2, 2, 128, 128)
    want, lse = _native._flash_attention(q, k, v, False, None, tm)
    k[:, :, 32:], v[:, :, 32:] = float("nan"), float("nan")
    got, lse2 = _native._flash_attention(q, k, v, False, None, tm)
    assert torch.equal(got, want) and torch.equal(lse, lse2)
    dq = _native._flash_attention_backward(g, q, k, v, got, lse, False, None, tm)[0]
    assert not dq.isnan().any()
