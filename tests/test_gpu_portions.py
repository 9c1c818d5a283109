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
@pytest.mark.parametrize("prompt,portions", [(0, [40]), (3, [4, 17, 16]), (9, [3, 4]), (480, [31, 5, 33]), (511, [32]), (512, [40]), (700, [33]), (300, [530]),
                                             (1, [600, 65]), (2500, [21, 4]), (5, [2060])])
def test_portions_equal_single_tokens(sessions, prompt, portions):
    a, b = sessions
    rng = np.random.default_rng(1000 + prompt)
    for s in (a, b):
        s.reset()
    log = []
    if prompt:
        ids = gi.prompt_ids(50 + prompt, prompt)
        log = [a.prefill(ids)[0]]
        assert log == [b.prefill(ids)[0]]
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
        log += [arg] if n > 3 else b.read_ids(1 << 15)[-n:].tolist()
        assert a.read_ids(1 << 15).tolist() == log  # the log goes on with the portion's pick, or with those of its single tokens
    # both go on: steps that read every slot the portions wrote
    tok = int(rng.integers(0, a.cfg.n_vocab))
    for _ in range(2):
        (pa, la), (pb, lb) = a.decode(tok), b.decode(tok)
        assert normrel(la, lb) < TOL
        tok = pa
    a.decode_enqueue(5)
    assert a.read_ids(1 << 15)[:len(log)].tolist() == log and a.read_ids(1 << 15).size == len(log) + 7


def layer_in_64_bits(image, cos, sin, ids, past, table):
    """Residual stream in front of, inside and behind the one layer of a 270m-shaped image for tokens behind `past` (its keys and
    values), and their keys and values; table: the session's GeLU table over [-4, 4)."""
    h, f, qo, at = 640, 2048, 1024, 0

    def take(count, dtype):
        nonlocal at
        a = np.frombuffer(image, dtype, count, at)
        at += a.nbytes
        return a

    def matrix(rows, cols):
        return take(rows * cols, np.int8).reshape(rows, cols), take(cols, np.float32)

    wte, wte_scales = matrix(262144, h)
    take(h, np.float32)
    m = {name: matrix(*shape) for name, shape in (("q", (h, qo)), ("k", (h, 256)), ("v", (h, 256)), ("o", (qo, h)))}
    qn, kn, apre, apost = (1.0 + take(n, np.float32).astype(np.float64) for n in (256, 256, h, h))
    m.update({name: matrix(*shape) for name, shape in (("up", (h, f)), ("gate", (h, f)), ("down", (f, h)))})
    mpre, mpost = (1.0 + take(h, np.float32).astype(np.float64) for _ in range(2))
    w = {name: a.astype(np.float64) * s.astype(np.float64) for name, (a, s) in m.items()}
    n, n_past = len(ids), past[0].shape[0]

    def rms(x, wt):
        return x / np.sqrt((x * x).mean(-1, keepdims=True) + 1e-6) * wt

    def rope(x):
        c, s = (t.reshape(-1, 256)[n_past:n_past + n, :128].astype(np.float64).reshape(n, *[1] * (x.ndim - 2), 128) for t in (cos, sin))
        u, v = x[..., :128], x[..., 128:]
        return np.concatenate([c * u - s * v, c * v + s * u], -1)

    x0 = np.sqrt(np.float64(h)) * wte[ids].astype(np.float64) * wte_scales.astype(np.float64)
    a = rms(x0, apre)
    q = rope(rms((a @ w["q"]).reshape(n, 4, 256), qn)) / 16.0
    k, v = rope(rms(a @ w["k"], kn)), a @ w["v"]
    keys, values = np.concatenate([past[0], k]), np.concatenate([past[1], v])
    scores = np.einsum("nhd,jd->nhj", q, keys)
    scores[np.broadcast_to((np.arange(n_past + n) > n_past + np.arange(n)[:, None])[:, None], scores.shape)] = -np.inf
    p = np.exp(scores - scores.max(-1, keepdims=True))
    att = np.einsum("nhj,jd->nhd", p / p.sum(-1, keepdims=True), values).reshape(n, qo)
    x1 = x0 + rms(att @ w["o"], apost)
    a = rms(x1, mpre)
    gate, up = a @ w["gate"], a @ w["up"]
    i = np.trunc((gate + 4.0) * (table.size / 8.0)).astype(np.int64)
    act = np.where(i < 0, 0.0, np.where(i < table.size, table.astype(np.float64)[np.clip(i, 0, table.size - 1)], gate))
    return x0, x1, x1 + rms((act * up) @ w["down"], mpost), k, v


@pytest.mark.parametrize("prompt,n", [(3, 5), (200, 61), (400, 100)])
def test_portions_are_as_exact_as_single_tokens(tg, oracle, weight_images, prompt, n):
    """The error of a portion's rows against 64 bits is not larger than that of the same tokens one by one, behind the same cached keys
    and values: of the portion's own keys and values, behind the attention and behind the feed-forward.  Gates far
    outside the table's range, so that its steps play no part; rows with few large entries, as a feed-forward's inside is."""
    image = weight_images("270m", 1, 31).copy()
    h, f = 640, 2048
    gate_scales = 262144 * h + 4 * h + 4 * h + sum(a * b + 4 * b for a, b in ((h, 1024), (h, 256), (h, 256), (1024, h), (h, f))) + 4 * (512 + 2 * h) + h * f
    image[gate_scales:gate_scales + 4 * f].view(np.float32)[:] *= 1e4
    model = tg.Transformer(tg.named_config("270m", 1))
    model.read_weights_mem(image)
    table = oracle.gelu_table(-4.0, 4.0, 1 << 20)
    cos, sin = oracle.rope_tables(10000.0, 32768)
    a, b = [model.session(rope_sw=(cos, sin), gelu_table=table) for _ in range(2)]
    for s in (a, b):
        s.prefill(gi.prompt_ids(9, prompt))
    past = [t[:prompt].astype(np.float64) for t in a.kv(0)[:2]]
    ids = np.random.default_rng(n).integers(0, 262144, n).astype(np.int32)
    x0, x1, x2, k, v = layer_in_64_bits(image, cos, sin, ids, past, table)
    a.forward(ids)
    got = {"portion": [a.tap(1, rows=n), a.tap(2, rows=n)], "steps": [[], []]}
    for t in ids:
        b.decode(int(t), want_logits=False)
        for i in range(2):
            got["steps"][i].append(b.tap(i + 1)[0])
    err = {}
    for name, s in (("portion", a), ("steps", b)):
        kk, vv = (t[prompt:prompt + n] for t in s.kv(0)[:2])
        y1, y2 = (np.array(t, np.float64) for t in got[name])
        err[name] = [normrel(kk, k), normrel(vv, v), normrel(y1 - x0, x1 - x0), normrel(y2 - y1, x2 - x1)]
    print(f"{prompt} + {n}: " + "; ".join(f"{name} {' '.join(f'{e:.2e}' for e in es)}" for name, es in err.items()), flush=True)
    assert all(p <= 1.1 * q for p, q in zip(err["portion"], err["steps"]))


def test_short_portions_go_token_by_token(sessions):
    a, b = sessions
    for s in (a, b):
        s.reset()
        s.prefill(gi.prompt_ids(7, 30))
    a.forward([5, 6])
    a.forward([7, 8, 9])
    for t in range(5, 10):
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


def test_the_log_keeps_earlier_answers(sessions):
    """Prompt, answer, next turn, answer, sampled tokens: the log read once at the end holds all picks in order."""
    a, b = sessions
    for s in (a, b):
        s.reset()
    prompt, turn = gi.prompt_ids(9, 20), gi.prompt_ids(10, 30)
    randf = np.random.default_rng(3).uniform(0, 1, 6).astype(np.float32)
    log = [a.prefill(prompt)[0]]
    a.decode_enqueue(5)
    log = a.read_ids(64).tolist()
    assert len(log) == 6
    log.append(a.forward(np.concatenate([[log[-1]], turn]).astype(np.int32))[0])
    a.decode_enqueue(4)
    a.decode_enqueue_sampled(6, 0.05, 1.0, randf)
    got = a.read_ids(64).tolist()
    assert got[:7] == log and len(got) == 17
    # the same with a read behind every call
    b.prefill(prompt)
    b.decode_enqueue(5)
    b.forward(np.concatenate([b.read_ids(64)[-1:], turn]).astype(np.int32))
    b.decode_enqueue(4)
    assert b.read_ids(64).tolist() == got[:11]
    b.decode_enqueue_sampled(6, 0.05, 1.0, randf)
    assert b.read_ids(64).tolist() == got


def test_reset_leaves_empty_caches(sessions):
    """A reset clears the rows written since the last one: behind a prompt longer than the local rings, portions, single tokens, steps and
    rows set one layer at a time, then behind a shorter request."""
    a, _ = sessions
    rng = np.random.default_rng(12)

    def rows(n):
        return rng.standard_normal((n, 256)).astype(np.float32)

    def long_request():
        a.prefill(gi.prompt_ids(11, 700))
        a.forward(gi.prompt_ids(12, 40))
        a.forward([1, 2])
        a.decode_enqueue(9)
        a.decode_enqueue_sampled(3, 0.1, 1.0, rng.uniform(0, 1, 3).astype(np.float32))

    def short_request():
        a.prefill(gi.prompt_ids(13, 20))
        a.decode_enqueue(2)

    def by_layer():
        for layer in (0, 5):
            a.kv_prefill(layer, rows(600), rows(600))
        for _ in range(3):
            a.block_attention(0, rng.standard_normal((1, 640)).astype(np.float32))

    def by_block():
        a.block_attention(5, rng.standard_normal((50, 640)).astype(np.float32))

    a.reset()
    for fill in (long_request, short_request, by_layer, by_block, short_request):
        fill()
        assert any(a.kv(layer)[0].any() for layer in range(6))
        a.reset()
        for layer in range(6):
            k, v, pos, _ = a.kv(layer)
            assert pos == 0 and not k.any() and not v.any(), (fill.__name__, layer)
