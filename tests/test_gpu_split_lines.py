"""The float32 forward's split key ranges below head dim 128: pieces of at least 4 tiles of 32 keys, one
per CU where the plan takes longer ones, rows too short to split, and the results on both sides.
"""
import numpy as np
import pytest

from tests._data import assert_f32

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"

CASES = [  # B, H, L, S, E, causal, pieces: none, short (4 tiles), or one per CU at most
    (1, 1, 200, 256, 32, False, "none"), (1, 1, 200, 257, 32, False, "some"), (1, 1, 200, 172, 64, False, "short"),
    (7, 2, 253, 1260, 32, False, "cu"), (8, 4, 128, 4096, 40, False, "cu"), (1, 1, 128, 16384, 33, False, "cu"),
    (1, 2, 130, 9000, 96, False, "cu"), (1, 16, 1000, 1000, 64, True, "cu"), (2, 6, 512, 512, 64, True, "short"),
]


@pytest.mark.parametrize("B,H,L,S,E,causal,pieces", CASES)
def test_split_lines(oracle_lib, B, H, L, S, E, causal, pieces):
    from densecore_amd import _native
    print(f"[case] split lines B{B} H{H} L{L} S{S} E{E} causal={causal}", flush=True)
    rng = np.random.default_rng(S + E)
    q, k, v = (rng.standard_normal((B, H, n, E), dtype=np.float32) for n in (L, S, S))
    t = [torch.from_numpy(x).to(DEV) for x in (q, k, v)]
    chunk = _native._schedule(False, *t, causal)["split_chunk"]
    if pieces == "none":
        assert chunk == 0
    elif pieces == "short":
        assert chunk == 4
    else:
        assert chunk >= 4
    if pieces == "cu":
        ends = [min(128 * (i + 1), S) if causal else S for i in range(-(-L // 128))]
        total = B * H * sum(-(-(-(-e // 32)) // chunk) for e in ends)
        assert total <= torch.cuda.get_device_properties(0).multi_processor_count
    out, lse = _native._flash_attention(*t, causal)
    ref_o, ref_l = oracle_lib.forward(q, k, v, causal)
    assert_f32(out.cpu().numpy(), ref_o, "out")
    assert_f32(lse.cpu().numpy(), ref_l, "lse")
