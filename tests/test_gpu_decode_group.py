"""Grouped-head decode: one workgroup reads a kv head's keys for up to 8 of its query heads.

Edges of the head groups (2, 4, 8, and more than 8), of a wave's chunk of keys (16 to 64, by head dim
and type), of the split ranges, and of the load forms (whole rows of 16-byte parts, padded head dims,
rows that are not 16-byte aligned), against the oracle at the float32 and bf16 bars.
"""
import ctypes

import numpy as np
import pytest

from tests._data import assert_bf16, assert_f32, bf16_round

torch = pytest.importorskip("torch")
DEV = "cuda:0"

CASES = [  # B, H, Hkv, S, E
    (1, 2, 1, 1, 64), (2, 4, 2, 15, 32), (1, 6, 2, 17, 128), (2, 8, 2, 65, 64), (1, 10, 2, 257, 100),
    (3, 8, 1, 1025, 40), (1, 16, 2, 130, 256), (1, 24, 2, 511, 128), (1, 34, 2, 300, 64),
    (2, 6, 2, 700, 33), (1, 8, 2, 4481, 80), (1, 5, 1, 64, 200),
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("B,H,Hkv,S,E", CASES)
def test_grouped_decode(oracle_lib, B, H, Hkv, S, E, dtype):
    from densecore_amd import _native
    print(f"[case] grouped decode {dtype} B{B} H{H} Hkv{Hkv} S{S} E{E}", flush=True)
    rng = np.random.default_rng(B + H + S + E)
    q, k, v = (rng.standard_normal(s, dtype=np.float32)
               for s in ((B, H, 1, E), (B, Hkv, S, E), (B, Hkv, S, E)))
    if dtype == "bf16":
        q, k, v = bf16_round(q), bf16_round(k), bf16_round(v)
    ref_o, ref_l = oracle_lib.forward(q, k, v, False)
    tdt = torch.float32 if dtype == "f32" else torch.bfloat16
    out, lse = _native._flash_decode(*(torch.from_numpy(x).to(DEV, tdt) for x in (q, k, v)))
    check = assert_f32 if dtype == "f32" else assert_bf16
    check(out.float().cpu().numpy(), ref_o, "out")
    check(lse.cpu().numpy(), ref_l, "lse")


@pytest.mark.gpu
def test_grouped_decode_infinite_value(oracle_lib):
    """An infinity in the last value row of a partly filled chunk reaches only its own dim."""
    from densecore_amd import _native
    rng = np.random.default_rng(3)
    q, k, v = (rng.standard_normal(s, dtype=np.float32) for s in ((1, 4, 1, 64), (1, 1, 70, 64), (1, 1, 70, 64)))
    v[0, 0, 69, 5] = np.inf
    out, _ = _native._flash_decode(*(torch.from_numpy(x).to(DEV) for x in (q, k, v)))
    out = out.cpu().numpy()
    assert np.isposinf(out[..., 5]).all() and np.isfinite(np.delete(out, 5, -1)).all()


def test_grouped_splits_fit_the_scratch():
    """The allocation-free entry point refuses a call only where one split of each head is too much
    for its 16 MiB, or where equal heads of the same shape were refused for their 2048-key ranges."""
    from densecore_amd import _lib
    L = _lib.lib()
    for B in (1, 3, 64):
        for H, Hkv in ((2, 1), (12, 4), (64, 8), (40, 2)):
            for S in (1, 63, 1000, 16384, 1 << 20):
                for E in (32, 80, 256):
                    for dt in (_lib.DC_F32, _lib.DC_BF16):
                        d = _lib.Desc(B, H, Hkv, 1, S, E, 0, 0, 0.0, dt, 0, 0, 0, 0)
                        need = L.dc_sdpa_decode_workspace_size(ctypes.byref(d))
                        st = L.dc_sdpa_decode_noalloc(ctypes.byref(d), *([None] * 6))
                        one = B * H * (E + 2) * 4
                        assert (st == _lib.DC_INVALID_ARGUMENT) == (need <= 1 << 24) == (one <= 1 << 24), (B, H, Hkv, S, E, need)
