"""Float32 forward under key padding with rows of more tiles than a workgroup lists at a time (1024 of
32 keys): tiles on both sides of a list's end, a list without any, and closed tiles that hold NaN, which
are not visited.  The oracle gets the open keys alone.
"""
import numpy as np
import pytest

from tests._data import assert_f32

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"
EDGE = 32 * 1024

CASES = [  # S, E, open ranges of keys (one list per head)
    (EDGE + 1, 64, [[(0, 50), (EDGE - 3, EDGE + 1)]]),
    (EDGE + 232, 80, [[(EDGE - 40, EDGE + 5), (EDGE + 225, EDGE + 232)]]),
    (2 * EDGE + 70, 32, [[(7, 9), (2 * EDGE - 1, 2 * EDGE + 70)], [(EDGE + 5, EDGE + 300)]]),
    (2 * EDGE + 70, 64, [[(2 * EDGE + 3, 2 * EDGE + 4)], [(0, 1)]]),
]


@pytest.mark.parametrize("S,E,opened", CASES)
def test_long_padded_rows(oracle_lib, S, E, opened):
    from densecore_amd import _native
    print(f"[case] long padded rows S{S} E{E} {opened}", flush=True)
    rng = np.random.default_rng(S + E)
    H, L = 2, 140
    q = rng.standard_normal((1, H, L, E), dtype=np.float32)
    k, v = (rng.standard_normal((1, H, S, E), dtype=np.float32) for _ in range(2))
    m = np.full((1, len(opened), 1, S), -np.inf, np.float32)
    for h, ranges in enumerate(opened):
        for a, b in ranges:
            m[0, h, 0, a:b] = 0
    visible = np.broadcast_to(m[0, :, 0] == 0, (H, S))
    pad = -S % 32
    closed = ~np.pad(visible, ((0, 0), (0, pad))).reshape(H, -1, 32).any(-1)
    hidden = np.repeat(closed, 32, -1)[:, :S]
    k[0][hidden], v[0][hidden] = np.nan, np.nan
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)
    out, lse = _native._flash_attention(t(q), t(k), t(v), False, None, t(m).expand(1, H, L, S))
    for h in range(H):
        keys = visible[h]
        ref_o, ref_l = oracle_lib.forward(q[:, h:h + 1], k[:, h:h + 1, keys], v[:, h:h + 1, keys], False)
        assert_f32(out[:, h:h + 1].cpu().numpy(), ref_o, "out")
        assert_f32(lse[:, h:h + 1].cpu().numpy(), ref_l, "lse")


def test_long_padding_is_skipped():
    """Texts of 4096 keys in rows of 65536 take a fraction of the time of full ones (as long when rows
    past a list's end went through all their tiles)."""
    from densecore_amd import _native
    S = 2 * EDGE
    gen = torch.Generator(device=DEV).manual_seed(3)
    q, k, v = (torch.randn(4, h, n, 32, generator=gen, device=DEV) for h, n in ((8, 128), (1, S), (1, S)))

    def us(n):
        m = torch.zeros(4, 1, 1, S, device=DEV)
        m[..., n:] = float("-inf")
        m = m.expand(4, 8, 128, S)
        times = []
        for _ in range(4):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            _native._flash_attention(q, k, v, False, None, m)
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end) * 1e3)
        return min(times)

    full, short = us(S), us(4096)
    print(f"  65536 keys {full:.0f} us, 4096 {short:.0f} us", flush=True)
    assert short < full / 2
