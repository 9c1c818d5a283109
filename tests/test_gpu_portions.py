"""GPU: later portions of a Gemma session (tg_forward_tokens) against the same tokens one by one through the decode step.

Both are fp32 paths that differ in summation order only; with a near-continuous GeLU table they agree as the prompt and the
decode step agree with the checker in test_gpu_model.py (6 layers: 6e-6 measured there, bound 1.5e-5)."""
import numpy as np
import pytest

import golden_inputs as gi
from conftest import normrel

pytestmark = pytest.mark.gpu
TOL = 1.5e-5


@pytest.fixture(scope="module")
def sessions(tg, oracle, weight_images):
    model = tg.Transformer(tg.named_config("270m", 6))  # five local layers and a global one
    model.read_weights_mem(weight_images("270m", 6, 31))
    table = oracle.gelu_table(-4.0, 4.0, 1 << 20)
    return [model.session(gelu_table=table) for _ in range(2)]


# a portion of an empty session with several wanted places; portions in front of, at and across the 512 slots of the
# local rings; one longer than a ring; counts around the tiles of 16 and 32 queries; a long past for few queries; a portion of more
# rows than the last pass of the attention takes four parts at a time for
@pytest.mark.parametrize("prompt,portions", [(0, [40]), (3, [4, 17, 16]), (9, [3]), (480, [31, 5, 33]), (511, [32]), (512, [40]), (700, [33]), (300, [530]),
                                             (1, [600, 65]), (2500, [21, 4]), (5, [2060])])
def test_portions_equal_single_tokens(sessions, prompt, portions):
    a, b = sessions
    rng = np.random.default_rng(1000 + prompt)
    for s in (a, b):
        s.reset()
    if prompt:
        ids = gi.prompt_ids(50 + prompt, prompt)
        assert a.prefill(ids)[0] == b.prefill(ids)[0]
    for n in portions:
        ids = rng.integers(0, a.cfg.n_vocab, n).astype(np.int32)
        want = np.unique([0, n // 2, n - 2, n - 1] if n != 5 else [1, 3])  # once without the last place
        arg, logits = a.forward(ids, want)
        rows = {}
        for i, t in enumerate(ids):
            pick, lg = b.decode(t, want_logits=i in want or i == n - 1)
            rows[i] = lg
        worst = max(normrel(logits[k], rows[int(w)]) for k, w in enumerate(want))
        print(f"{prompt} + {n}: logits {worst:.1e}", flush=True)
        assert worst < TOL
        gap = np.sort(rows[n - 1])[-2:]
        assert arg == pick or gap[1] - gap[0] < 1e-4
        assert a.position == b.position
        for layer in (0, 4, 5):
            ka, va, pa, ba = a.kv(layer)
            kb, vb, pb, bb = b.kv(layer)
            assert (pa, ba) == (pb, bb)
            n_valid = min(pa, ka.shape[0])
            assert normrel(ka[:n_valid], kb[:n_valid]) < TOL and normrel(va[:n_valid], vb[:n_valid]) < TOL
            assert np.abs(ka - kb).max() < 1e-3 and np.abs(va - vb).max() < 1e-3  # every slot, also the untouched ones
        assert a.read_ids(1 << 15).tolist() == [arg]  # the log starts with the portion's pick
    # both go on: steps that read every slot the portions wrote
    tok = int(rng.integers(0, a.cfg.n_vocab))
    for _ in range(2):
        (pa, la), (pb, lb) = a.decode(tok), b.decode(tok)
        assert normrel(la, lb) < TOL
        tok = pa
    a.decode_enqueue(5)
    assert a.read_ids(64).size == 8


def test_short_portions_go_token_by_token(sessions):
    a, b = sessions
    for s in (a, b):
        s.reset()
        s.prefill(gi.prompt_ids(7, 30))
    a.forward([5, 6])
    for t in (5, 6):
        b.decode(t)
    assert np.array_equal(a.read_ids(64), b.read_ids(64)) and np.array_equal(a.kv(0)[0], b.kv(0)[0])


def test_context_end(sessions):
    """A portion that ends at the last position, and one that would pass it."""
    a, _ = sessions
    a.reset()
    n = a.cfg.n_pos
    a.prefill(gi.prompt_ids(8, n - 20), want_logits=False)
    with pytest.raises(Exception, match="context is full"):
        a.forward(np.zeros(21, np.int32))
    a.forward(np.arange(20, dtype=np.int32))
    assert a.position == n
    with pytest.raises(Exception, match="context is full"):
        a.forward([1, 2, 3])
