"""The Bernoulli draw at the edges of a chunk's steps (192 words, 96 elements), where the last words, the
last keep word and the engine block that is written back fall in the window, in a step or between
two: bit for bit against the oracle, mask and engine state."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pre", [0, 311, 623])
@pytest.mark.parametrize("n", [64 + 287, 64 + 288, 64 + 289, 64 + 383, 64 + 384, 64 + 385, 64 + 479, 64 + 481, 64 + 577,
                               64 + 65_536 - 97, 64 + 65_536 - 1, 64 + 65_536 + 96, 64 + 2 * 65_536 + 300])
def test_step_edges(n, pre):
    from tests.test_gpu_dropout import _gen, _state_equal, _unpack
    print(f"[case] bernoulli steps n={n} pre={pre}", flush=True)
    g, o = _gen(n + 7 * pre, pre)
    assert np.array_equal(_unpack(g._bernoulli_bits(n, 0.6), n), o.bernoulli(n, 0.6).astype(bool))
    assert _state_equal(g, o)
    assert np.array_equal(_unpack(g._bernoulli_bits(100, 0.6), 100), o.bernoulli(100, 0.6).astype(bool))
