"""The float32 backward's choice between whole key tiles and stream-K ranges at head dims up to 64,
where one workgroup runs per CU: which side of each line the tile counts fall, and the results there.
"""
import numpy as np
import pytest

from tests._data import assert_f32

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"

CASES = [  # key tiles per CU as a ratio, causal, mask, stream-K
    ((1, 1), True, None, True), ((9, 8), True, None, False), ((2, 1), True, None, False),
    ((5, 8), False, None, True), ((3, 4), False, None, False), ((1, 1), False, None, False), ((9, 8), False, None, True),
    ((3, 2), False, None, True), ((13, 8), False, None, False), ((15, 8), False, None, False),
    ((5, 8), False, "pad", True), ((9, 8), False, "pad", False), ((9, 8), False, "full", True), ((9, 8), True, "pad", False),
]


@pytest.mark.parametrize("ratio,causal,mask,streamk", CASES)
def test_lines(oracle_lib, ratio, causal, mask, streamk):
    from densecore_amd import _native
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    B, H = cus * ratio[0] // ratio[1] // 4, 2  # two key tiles per head
    print(f"[case] stream-K lines B{B} H{H} of 2 tiles causal={causal} mask={mask}", flush=True)
    rng = np.random.default_rng(B)
    L, S, E = 140, 150, 32
    q, k, v, g = (rng.standard_normal((B, H, n, E), dtype=np.float32) for n in (L, S, S, L))
    m = None
    if mask:
        m = np.zeros((B, 1, 1 if mask == "pad" else L, S), np.float32)
        m[::2, ..., 100:] = -np.inf
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)
    tm = None if m is None else t(m).expand(B, H, L, S)
    sched = _native._schedule(True, t(q), t(k), t(v), causal, None, tm)
    assert (sched["streamk_ranges"] > 0) == streamk, sched
    full = None if m is None else np.ascontiguousarray(np.broadcast_to(m, (B, H, L, S)))
    out, lse = oracle_lib.forward(q, k, v, causal, None, full)
    ref = oracle_lib.backward(g, q, k, v, out, lse, causal, None, full)
    got = _native._flash_attention_backward(*(t(x) for x in (g, q, k, v, out, lse)), causal, None, tm)
    for name, a, b in zip(("dq", "dk", "dv"), got, ref):
        assert_f32(a.cpu().numpy(), b, name)
