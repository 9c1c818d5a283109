"""The work that programs built on this framework have it do, as cases that can be timed and checked.

Three kinds, each through the package's public calls:

linear  the products of one feed-forward block on device-resident buffers (QWeight.gemv for one row, QWeight.gemm for more),
        as a program with its own model loop makes them.
gemma   requests to an int8 model of the Gemma shapes: a prompt, generated tokens (greedy or min-p), and, where the case has
        one, the user's next turn behind them with its own answer.
net     requests to a layer-list model opened from its folder (Madevik, Tutelix), in bfloat16 or float32: a prompt, whole or in
        portions, and generated tokens.

Weights are random.  Sublayers add little to the residual stream and the head's columns are the embeddings of the token
before, so that a pick is as decisive as a trained model's mostly is, and every step meets another token.
"""
import importlib.util
import json
import math
import os
import shutil
import struct
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
VOCAB = 262144
SHAPES = {"270m": (640, 2048, 18), "1B": (1152, 6912, 26)}  # hidden, feed-forward, layers
HEADS, HEAD_DIM, WINDOW, PATTERN = 4, 256, 512, 6
TEMPERATURE = 1.0


def package():
    if "tiny_gemma_amd" not in sys.modules:
        path = os.path.join(ROOT, "tiny-gemma_amd")
        spec = importlib.util.spec_from_file_location("tiny_gemma_amd", os.path.join(path, "__init__.py"), submodule_search_locations=[path])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["tiny_gemma_amd"] = mod
        spec.loader.exec_module(mod)
    sys.modules["tiny_gemma_amd"].init(0)
    return sys.modules["tiny_gemma_amd"]


# ---- the cases --------------------------------------------------------------------------------------------------------------
def linear(name, shape, rows):
    return {"name": name, "kind": "linear", "shape": shape, "rows": rows}


def gemma(name, shape, prompt, steps, turn=0, answer=0, minp=1.0):
    return {"name": name, "kind": "gemma", "shape": shape, "prompt": prompt, "steps": steps, "turn": turn, "answer": answer, "minp": minp}


def net(name, design, width, dtype, prompt, portion, steps):
    return {"name": name, "kind": "net", "design": design, "width": width, "dtype": dtype, "prompt": prompt, "portion": portion, "steps": steps}


def listed():
    return [
        # one token through a feed-forward block of the small shape: three launches, nothing but latency
        linear("products_270m_1_row", "270m", 1),
        # the same products of the large shape for a batch of rows that fills no tile
        linear("products_1b_777_rows", "1B", 777),
        # a short question and the first words of the answer: what a user waits for
        gemma("270m_9_tokens_16_steps", "270m", 9, 16),
        # a request of ordinary size to the small model
        gemma("270m_64_tokens_128_steps", "270m", 64, 128),
        # a long document and a short answer about it
        gemma("270m_16384_tokens_32_steps", "270m", 16384, 32),
        # the mean chat prompt and the beginning of its completion
        gemma("1b_178_tokens_128_steps", "1B", 178, 128),
        # a document read once, of which only the end is wanted (classification, the next token)
        gemma("1b_4096_tokens", "1B", 4096, 0),
        # a conversation: prompt, answer, the user's next turn, answer
        gemma("1b_chat_300_and_61_tokens", "1B", 300, 24, 61, 24),
        # a sampled completion behind a page of text
        gemma("1b_1000_tokens_48_sampled", "1B", 1000, 48, 0, 0, 0.1),
        # a layer-list model with experts, prompt of some pages, short answer
        net("madevik_640_1024_tokens_32_steps", "Madevik", 640, "bfloat16", 1024, 1024, 32),
        # a layer-list model that is fed its prompt in portions, as a server that interleaves requests does
        net("tutelix_1152_600_in_portions", "Tutelix", 1152, "bfloat16", 600, 130, 24),
        # full precision, as for checking a model's quality
        net("tutelix_640_f32_333_tokens_16_steps", "Tutelix", 640, "float32", 333, 333, 16),
    ]


def log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "gemma", "gemma", "gemma", "net", "net"])
    if kind == "linear":
        case = linear("", rng.choice(list(SHAPES)), log_int(rng, 1, 2000))
    elif kind == "gemma":
        shape = rng.choice(list(SHAPES))
        prompt = log_int(rng, 1, 16000 if shape == "270m" else 4000)
        steps = log_int(rng, 1, 100)
        turn = answer = 0
        if rng.random() < 0.35 and prompt <= 4000:
            turn, answer = log_int(rng, 2, 64), log_int(rng, 1, 24)
            steps = min(steps, 24)
        case = gemma("", shape, prompt, steps, turn, answer, 0.1 if rng.random() < 0.25 else 1.0)
    else:
        prompt = log_int(rng, 2, 1200)
        case = net("", *rng.choice([("Madevik", 640, "bfloat16"), ("Tutelix", 640, "bfloat16"), ("Tutelix", 1152, "bfloat16"), ("Tutelix", 640, "float32"),
                                    ("Madevik", 640, "float32")]), prompt, rng.choice([prompt, max(2, log_int(rng, 1 + prompt // 10, prompt))]), log_int(rng, 1, 32))
    del case["name"]
    return case


# ---- random weights, as the files hold them -------------------------------------------------------------------------------------
def normal(gen, shape, std, mean=0.0):
    return torch.randn(shape, generator=gen, device="cuda") * std + mean


def quantized(w):
    """int8 values and the fp32 scale of every column."""
    s = w.abs().amax(0) / 127.0
    return torch.round(w / s).to(torch.int8), s


def generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def gemma_tensors(shape, seed):
    """(name, tensor) in file order; a matrix as (int8 [in][out], fp32 scales)."""
    h, f, layers = SHAPES[shape]
    gen, qo = generator(seed), HEADS * HEAD_DIM

    def matrix(a, b):
        return quantized(normal(gen, (a, b), 0.02))

    wte = normal(gen, (VOCAB, h), 0.02)
    yield "wte", quantized(wte)
    yield "norm", normal(gen, (h,), 0.1, 2.0)
    head = quantized(torch.roll(wte, 1, 0).t().contiguous())
    del wte
    for l in range(layers):
        for name, a, b in (("q", h, qo), ("k", h, HEAD_DIM), ("v", h, HEAD_DIM), ("o", qo, h)):
            yield f"{l}.{name}", matrix(a, b)
        yield f"{l}.qn", normal(gen, (HEAD_DIM,), 0.1)
        yield f"{l}.kn", normal(gen, (HEAD_DIM,), 0.1)
        yield f"{l}.apre", normal(gen, (h,), 0.1)
        yield f"{l}.apost", normal(gen, (h,), 0.05, -0.85)
        for name, a, b in (("up", h, f), ("gate", h, f), ("down", f, h)):
            yield f"{l}.{name}", matrix(a, b)
        yield f"{l}.mpre", normal(gen, (h,), 0.1)
        yield f"{l}.mpost", normal(gen, (h,), 0.05, -0.85)
    yield "head", head


def gemma_image(shape, seed):
    parts = []
    for _, t in gemma_tensors(shape, seed):
        parts += [x.contiguous().view(torch.uint8).reshape(-1) for x in (t if isinstance(t, tuple) else (t,))]
    image = torch.cat(parts)
    del parts
    return image.cpu().numpy()


def net_config(design, width):
    def head(**more):
        return dict({"architecture": design, "width": width, "vocab": VOCAB, "norm": {"eps": 1e-5}}, **more)

    if design == "Madevik":
        gla = {"type": "gla", "mixer": {"heads": 4, "dim": 64, "vdim": 128, "tau": 16.0}}
        lat = {"type": "latent_attention", "mixer": {"heads": 4, "dim": 64, "vdim": 64, "kv_rank": 128, "scale": 0.125}}
        mlp = {"kind": "moe", "expert": {"ff": 768}, "router": {"experts": 8, "top": 2, "scale": 2.5}}
        return head(residual_mult=0.5, layers=[dict(lat if i % 3 == 2 else gla, mlp=mlp) for i in range(18)])

    def lat(heads, dim, rot, vdim, q, kv, window):
        return {"type": "latent_attention", "mixer": {"heads": heads, "dim": dim, "rot_dim": rot, "vdim": vdim, "q_rank": q, "kv_rank": kv, "mask": {"size": window},
                                                      "rot": {"base": 10000.0, "dims": rot}, "scale": (dim + rot) ** -0.5}}

    def att(heads, kv, dim, rot, window):
        return {"type": "attention", "mixer": {"heads": heads, "kv_heads": kv, "dim": dim, "vdim": dim, "mask": {"size": window},
                                               "rot": {"base": 1000000.0, "dims": rot}, "scale": dim ** -0.5}}

    def delta(heads, kv, dim, vdim):
        return {"type": "channel_delta", "mixer": {"heads": heads, "kv_heads": kv, "dim": dim, "vdim": vdim, "conv": 4}}

    if width == 640:
        mixers, ff, loop = [delta(4, 4, 64, 128), lat(4, 64, 32, 64, 256, 128, 1024), att(8, 2, 64, 32, 512)] * 6, 2304, (0, 1, 1)
    else:
        a, b, d = delta(4, 4, 128, 256), lat(8, 128, 64, 128, 512, 256, 1024), att(8, 2, 128, 64, 512)
        mixers, ff, loop = [a, a, d, b, a, a, d, b, a, b], 10368, (0, 8, 3)
    return head(embedding={"scale": 1.0}, layers=[dict(m, mlp={"kind": "dense", "ff": ff}) for m in mixers],
                loop={"start": loop[0], "stop": loop[1], "times": loop[2]})


def layer_runs(cfg):
    n, loop = len(cfg["layers"]), cfg.get("loop")
    if not loop:
        return list(range(n))
    a, b = loop["start"], loop["stop"]
    return list(range(a)) + list(range(a, b)) * loop["times"] + list(range(b, n))


def net_tensors(cfg, seed):
    """(name, bfloat16 tensor) in file order.  Output projections are scaled down by the depth of the residual stream."""
    gen, D = generator(seed), cfg["width"]
    small = (2 * len(layer_runs(cfg))) ** -0.5
    bf = torch.bfloat16

    def w(rows, cols, gain=1.0):
        return normal(gen, (rows, cols), gain * cols ** -0.5).to(bf)

    def vec(n, std, mean=0.0):
        return normal(gen, (n,), std, mean).to(bf)

    def dyt(name):
        return [(name, vec(D, 0.1, 1.0)), (name + ".b", vec(D, 0.1)), (name + ".alpha", torch.tensor(0.7, dtype=bf, device="cuda"))]

    embed = normal(gen, (VOCAB, D), 1.0).to(bf)
    yield "embed", embed
    head = (torch.roll(embed, 1, 0).float() * D ** -0.5).to(bf)
    for i, l in enumerate(cfg["layers"]):
        m, p, q = l["mixer"], f"l{i}.mix.", f"l{i}.mlp."
        H, d, v = m["heads"], m["dim"], m["vdim"]
        if cfg["architecture"] == "Madevik":
            yield from dyt(f"l{i}.norm1")
            yield p + "q", w(H * d, D)
            if l["type"] == "gla":
                yield from [(p + "k", w(H * d, D)), (p + "v", w(H * v, D)), (p + "g", w(H * v, D)), (p + "o", w(D, H * v, small)), (p + "norm", vec(v, 0.1, 1.0)),
                            (p + "a1", w(16, D)), (p + "a2", w(H * d, 16)), (p + "a2.b", vec(H * d, 0.5, 3.0))]
            else:
                r = m["kv_rank"]
                yield from [(p + "dkv", w(r, D)), (p + "dkv.norm", vec(r, 0.1, 1.0)), (p + "uk", w(H * d, r)), (p + "uv", w(H * v, r)), (p + "g", w(H, D)),
                            (p + "o", w(D, H * v, small))]
            yield from dyt(f"l{i}.norm2")
            E, ff = l["mlp"]["router"]["experts"], l["mlp"]["expert"]["ff"]
            for e in range(E):
                yield from [(f"{q}e{e}.gate", w(ff, D)), (f"{q}e{e}.up", w(ff, D)), (f"{q}e{e}.down", w(D, ff, small))]
            yield from [(q + "router", w(E, D)), (q + "correction", vec(E, 0.1))]
            continue
        yield from [(f"l{i}.norm1", vec(D, 0.1)), (f"l{i}.norm1b", vec(D, 0.1 * small, small - 1.0)), (f"l{i}.norm2", vec(D, 0.1)),
                    (f"l{i}.norm2b", vec(D, 0.1 * small, small - 1.0))]
        if l["type"] == "latent_attention":
            r, k, e = m["q_rank"], m["kv_rank"], m["rot_dim"]
            yield from [(p + "dq", w(r, D)), (p + "dq.norm", vec(r, 0.1, 1.0)), (p + "uq", w(H * (d + e), r)), (p + "dkv", w(k + e, D)),
                        (p + "dkv.norm", vec(k, 0.1, 1.0)), (p + "uk", w(H * d, k)), (p + "uv", w(H * v, k))]
        elif l["type"] == "attention":
            G = m["kv_heads"]
            yield from [(p + "q", w(H * d, D)), (p + "q.b", vec(H * d, 0.1)), (p + "k", w(G * d, D)), (p + "k.b", vec(G * d, 0.1))]
        else:
            G = m["kv_heads"]
            for name, rows in (("q", G * d), ("k", G * d), ("v", H * v)):
                yield from [(p + name, w(rows, D)), (f"{p}{name}.conv", w(rows, m["conv"]))]
            yield from [(p + "b", w(H, D)), (p + "A_log", vec(H, 0.1)), (p + "norm", vec(v, 0.1, 1.0)), (p + "a1", w(16, D)), (p + "a2", w(H * d, 16)),
                        (p + "dt_bias", vec(H * d, 0.5, -3.0)), (p + "g1", w(16, D)), (p + "g2", w(H * v, 16))]
        yield p + "o", w(D, H * v)
        yield from [(q + "up", w(l["mlp"]["ff"], D)), (q + "down", w(D, l["mlp"]["ff"]))]
    if cfg["architecture"] == "Madevik":
        yield from dyt("final.norm")
    else:
        yield "final.norm", vec(D, 0.1)
    yield "head", head


def write_folder(path, cfg, seed):
    with open(os.path.join(path, "config.json"), "w") as f:
        json.dump(cfg, f)
    head, parts, at = {}, [], 0
    for name, t in net_tensors(cfg, seed):
        n = 2 * t.numel()
        head[name] = {"dtype": "BF16", "shape": list(t.shape), "data_offsets": [at, at + n]}
        parts.append(t.contiguous().view(torch.uint8 if t.dim() else torch.int16).reshape(-1).view(torch.uint8))
        at += n
    data = torch.cat(parts)
    del parts
    text = json.dumps(head).encode()
    text += b" " * (-len(text) % 8)
    with open(os.path.join(path, "model.safetensors"), "wb") as f:
        f.write(struct.pack("<Q", len(text)) + text)
        data.cpu().numpy().tofile(f)


# ---- inputs -------------------------------------------------------------------------------------------------------------------------
def requests(case, seed):
    """Token ids and uniform numbers of a request, from the seed."""
    rng = np.random.default_rng(int(seed))
    r = {"prompt": rng.integers(0, VOCAB, case["prompt"]).astype(np.int32)}
    if case["kind"] == "gemma":
        r["turn"] = rng.integers(0, VOCAB, case["turn"]).astype(np.int32)
        r["rand"] = [rng.random(n, dtype=np.float32) for n in (case["steps"], case["answer"])]
    return r


def linear_inputs(case, seed):
    h, f, _ = SHAPES[case["shape"]]
    gen, m = generator(seed), case["rows"]
    weights = [quantized(normal(gen, s, 0.02)) for s in ((h, f), (h, f), (f, h))]
    # the feed-forward's inputs: a normed row, and the gated product, whose entries are mostly small
    x = normal(gen, (m, h), 1.0)
    hidden = normal(gen, (m, f), 1.0) * torch.nn.functional.gelu(normal(gen, (m, f), 1.0))
    return weights, x, hidden


class Buffer:
    """Device memory of a torch tensor, as the package's calls take it."""

    def __init__(self, t):
        self.t, self.p = t, t.data_ptr()


def prepare(case, seed):
    tg = package()
    if case["kind"] == "linear":
        weights, x, hidden = linear_inputs(case, seed)
        ws = [tg.QWeight(q.cpu().numpy(), s.cpu().numpy()) for q, s in weights]
        h, f, _ = SHAPES[case["shape"]]
        outs = [torch.empty((case["rows"], n), device="cuda") for n in (f, f, h)]
        return {"case": case, "weights": ws, "in": [Buffer(x), Buffer(x), Buffer(hidden)], "out": [Buffer(t) for t in outs]}
    state = dict(requests(case, seed), case=case)
    if case["kind"] == "gemma":
        model = tg.Transformer(tg.named_config(case["shape"]))
        model.read_weights_mem(gemma_image(case["shape"], seed))
        state["session"] = model.session()
    else:
        folder = tempfile.mkdtemp(prefix="model_", dir="/dev/shm" if os.access("/dev/shm", os.W_OK) else None)
        try:
            write_folder(folder, net_config(case["design"], case["width"]), seed)
            model = tg.Transformer.from_dir(folder, case["dtype"])
        finally:
            shutil.rmtree(folder, ignore_errors=True)
        state["session"] = model.open_session(case["prompt"] + case["steps"] + 1)
    state["model"] = model
    torch.cuda.empty_cache()
    return state


# ---- one pass -------------------------------------------------------------------------------------------------------------------------
def steps(session, n, minp, rand):
    """n generated tokens behind the last pick; the ids, the last pick among them."""
    if minp < 1.0:
        session.decode_enqueue_sampled(n, minp, TEMPERATURE, rand)
    else:
        session.decode_enqueue(n)
    return session.read_ids(1 << 15)[-(n + 1):]


def run(state):
    case = state["case"]
    if case["kind"] == "linear":
        for w, x, y in zip(state["weights"], state["in"], state["out"]):
            if case["rows"] == 1:
                w.gemv(y, x)
            else:
                w.gemm(y, x, case["rows"])
        return {"up": state["out"][0].t, "gate": state["out"][1].t, "down": state["out"][2].t}
    s = state["session"]
    s.reset()
    if case["kind"] == "net":
        ids, at = state["prompt"], 0
        while at < ids.size:
            _, logits = s.forward(ids[at:at + case["portion"]])
            at += case["portion"]
        out = {"logits": logits[0]}
        if case["steps"]:
            out["ids"] = steps(s, case["steps"], 1.0, None)
            out["last_logits"] = s.decode(out["ids"][-1])[1]
        return out
    pick, logits = s.prefill(state["prompt"])
    out = {"logits": logits, "ids": np.array([pick], np.int32)}
    if case["steps"]:
        out["ids"] = steps(s, case["steps"], case["minp"], state["rand"][0])
    if case["turn"]:
        _, out["turn_logits"] = s.forward(np.concatenate([out["ids"][-1:], state["turn"]]))
        out["answer"] = steps(s, case["answer"], case["minp"], state["rand"][1])
    if case["steps"]:
        out["last_logits"] = s.decode(out["answer" if case["turn"] else "ids"][-1])[1]
    return out


# ---- what a pass cannot do without ------------------------------------------------------------------------------------------------------
def gemma_params(shape):
    h, f, layers = SHAPES[shape]
    qo = HEADS * HEAD_DIM
    return layers * (h * (qo + 2 * HEAD_DIM) + qo * h + 3 * h * f), h * VOCAB, layers


def gemma_pass(shape, start, n):
    """bytes and flops of n tokens behind `start`: weights once, keys and values once, logits of the last."""
    body, head, layers = gemma_params(shape)
    glob = layers // PATTERN
    keys = sum(min(start + n, WINDOW + n) if i >= glob else start + n for i in range(layers))
    pairs = glob * (n * start + n * (n + 1) / 2) + (layers - glob) * n * min(start + (n + 1) / 2, WINDOW)
    return np.array([body + head + 8 * HEAD_DIM * keys + 4 * VOCAB, 2.0 * body * n + 2 * head + 4 * HEADS * HEAD_DIM * pairs])


def net_pass(cfg, dtype, start, n):
    D, size = cfg["width"], 2 if dtype == "bfloat16" else 4
    read = flops = 0.0
    for i in layer_runs(cfg):
        l = cfg["layers"][i]
        m = l["mixer"]
        H, d, v = m["heads"], m["dim"], m["vdim"]
        kind = l["type"]
        if kind in ("gla", "channel_delta"):
            w = D * (2 * m.get("kv_heads", H) * d + (3 if kind == "gla" else 2) * H * v)
            flops += n * 6 * H * d * v
            read += 8 * H * d * v
        elif kind == "attention":
            w = D * (2 * H * d + m["kv_heads"] * d)
            flops += n * 4 * H * d * min(start + (n + 1) / 2, m["mask"]["size"])
            read += size * m["kv_heads"] * d * min(start + n, m["mask"]["size"] + n)
        else:
            e, q = m.get("rot_dim", 0), m.get("q_rank", 0)
            w = D * (m["kv_rank"] + e + H * v) + (D * q + q * H * (d + e) if q else D * H * d) + m["kv_rank"] * H * (d + v)
            window = m.get("mask", {}).get("size", 1 << 30)
            flops += n * 2 * H * (d + e + v) * min(start + (n + 1) / 2, window)
            read += size * (m["kv_rank"] + e) * min(start + n, window + n)
        mlp = l["mlp"]
        if mlp["kind"] == "moe":
            E, top, one = mlp["router"]["experts"], mlp["router"]["top"], 3 * D * mlp["expert"]["ff"]
            read += size * (w + one * min(E, top * n))
            flops += 2.0 * n * (w + top * one)
        else:
            read += size * (w + 2 * D * mlp["ff"])
            flops += 2.0 * n * (w + 2 * D * mlp["ff"])
    return np.array([read + size * D * VOCAB + 4 * VOCAB, flops + 2 * D * VOCAB])


def work(case):
    if case["kind"] == "linear":
        h, f, _ = SHAPES[case["shape"]]
        m = case["rows"]
        return {"bytes": 3 * h * f + 4 * (2 * f + h) + 4 * m * (h + f) + 4 * m * (2 * f + h), "flops": 6.0 * m * h * f}
    if case["kind"] == "gemma":
        one = lambda at, n: gemma_pass(case["shape"], at, n)  # noqa: E731
    else:
        cfg = net_config(case["design"], case["width"])
        one = lambda at, n: net_pass(cfg, case["dtype"], at, n)  # noqa: E731
    total, at = np.zeros(2), 0
    while at < case["prompt"]:
        n = min(case.get("portion", case["prompt"]), case["prompt"] - at)
        total += one(at, n)
        at += n
    for n in [1] * case["steps"] + ([case["turn"] + 1] + [1] * case["answer"] if case.get("turn") else []) + [1] * (case["steps"] > 0):
        total += one(at, n)
        at += n
    return {"bytes": float(total[0]), "flops": float(total[1])}


def tolerance(case):
    if case["kind"] == "linear":
        return {"rel": 5e-6}
    if case["kind"] == "gemma":
        # the 1024-entry table of the gated product is a step function: a last bit moves a value to the next entry
        return {"rel": 1e-2, "max": 0.1, "differ": 0.005}
    return {"rel": 1e-2, "max": 0.1, "differ": 0.005} if case["dtype"] == "bfloat16" else {"rel": 1e-5, "max": 1e-4, "differ": 0.005}


# ---- the same in 64 bits ----------------------------------------------------------------------------------------------------------------
F = torch.float64


def rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


class GemmaExact:
    def __init__(self, shape, seed):
        self.h, self.f, self.layers = SHAPES[shape]
        self.t = {}
        for name, t in gemma_tensors(shape, seed):
            if isinstance(t, tuple):  # the two tables of the vocabulary stay as they are stored
                t = t if name in ("wte", "head") else t[0].to(F) * t[1].to(F)
            else:
                t = t.to(F) + 1.0
            self.t[name] = t
        x = np.float32(-4.0) + np.arange(1024, dtype=np.float32) * np.float32(8.0 / 1024)
        a = x.astype(np.float64)
        lut = (0.5 * a) * (1.0 + np.tanh(float(np.float32(0.7978845608)) * (a + float(np.float32(0.044715)) * a ** 3)))
        self.lut = torch.from_numpy(lut.astype(np.float32)).cuda().to(F)
        self.freq = {}
        for theta in (1e6, 1e4):
            e = (2 * np.arange(HEAD_DIM // 2)).astype(np.float32) / np.float32(HEAD_DIM)
            self.freq[theta] = torch.from_numpy((np.float32(1.0) / np.power(np.float32(theta), e)).astype(np.float32)).cuda()
        self.keys = [torch.empty((0, HEAD_DIM), dtype=F, device="cuda")] * self.layers
        self.values = list(self.keys)
        self.pos = 0

    def rope(self, x, at, theta):
        p = torch.arange(at, at + x.shape[0], dtype=torch.float32, device="cuda")
        a = (p[:, None] * self.freq[theta]).to(F)
        a = a if x.dim() == 2 else a[:, None]
        c, s, u, v = torch.cos(a), torch.sin(a), x[..., :HEAD_DIM // 2], x[..., HEAD_DIM // 2:]
        return torch.cat([c * u - s * v, c * v + s * u], -1)

    def attention(self, q, K, V, start, window):
        """q [n][heads][dim] behind `start` keys; `window`: keys that a token sees, itself among them (0: all)."""
        out = torch.empty_like(q)
        for a in range(0, q.shape[0], 512):
            b = min(a + 512, q.shape[0])
            lo = max(0, start + a - window + 1) if window else 0
            k, v = K[lo:start + b], V[lo:start + b]
            i = torch.arange(start + a, start + b, device="cuda")[:, None]
            j = torch.arange(lo, start + b, device="cuda")[None]
            bad = (j > i) | ((j <= i - window) if window else (j < 0))
            for hd in range(HEADS):
                s = (q[a:b, hd] @ k.t()) / math.sqrt(HEAD_DIM)
                out[a:b, hd] = torch.softmax(s.masked_fill(bad, -math.inf), -1) @ v
        return out

    def forward(self, ids, prefill):
        t, n, eps = self.t, len(ids), 1e-6
        q8, sc = t["wte"]
        x = math.sqrt(self.h) * q8[torch.as_tensor(np.asarray(ids), dtype=torch.long, device="cuda")].to(F) * sc.to(F)
        for l in range(self.layers):
            local = l % PATTERN != PATTERN - 1
            theta, p = (1e4 if local else 1e6), f"{l}."
            a = rms(x, t[p + "apre"], eps)
            q = self.rope(rms((a @ t[p + "q"]).view(n, HEADS, HEAD_DIM), t[p + "qn"], eps), self.pos, theta)
            k = self.rope(rms(a @ t[p + "k"], t[p + "kn"], eps), self.pos, theta)
            self.keys[l] = torch.cat([self.keys[l], k])
            self.values[l] = torch.cat([self.values[l], a @ t[p + "v"]])
            # a prompt's tokens see one key more of a local layer than the ring keeps
            o = self.attention(q, self.keys[l], self.values[l], self.pos, (WINDOW + (1 if prefill else 0)) if local else 0)
            x = x + rms(o.reshape(n, -1) @ t[p + "o"], t[p + "apost"], eps)
            a = rms(x, t[p + "mpre"], eps)
            gate = a @ t[p + "gate"]
            i = ((gate + 4.0) * 128.0).trunc().long()
            gate = torch.where(i < 0, torch.zeros_like(gate), torch.where(i < 1024, self.lut[i.clamp(0, 1023)], gate))
            x = x + rms((gate * (a @ t[p + "up"])) @ t[p + "down"], t[p + "mpost"], eps)
        self.pos += n
        last, (q8, sc) = rms(x[-1], t["norm"], eps), t["head"]
        logits = torch.empty(VOCAB, dtype=F, device="cuda")
        for a in range(0, VOCAB, 32768):
            logits[a:a + 32768] = (last @ q8[:, a:a + 32768].to(F)) * sc[a:a + 32768].to(F)
        return logits

    def generate(self, logits, n, minp, rand):
        ids = []
        for i in range(n + 1):
            # the pick behind a prompt is the most likely token; the ones behind it are drawn
            if minp < 1.0 and i > 0:
                p = torch.softmax(logits / TEMPERATURE, 0)
                p = p / p[p >= minp * p.max()].sum()
                over = torch.nonzero(torch.cumsum(p, 0) >= float(rand[i - 1]))
                ids.append(int(over[0, 0]) if over.numel() else 0)
            else:
                ids.append(int(torch.argmax(logits)))
            if i < n:
                logits = self.forward(ids[-1:], False)
        return ids


class NetExact:
    def __init__(self, case, seed):
        self.cfg = net_config(case["design"], case["width"])
        self.t = {name: t if name in ("embed", "head") else t.to(F) for name, t in net_tensors(self.cfg, seed)}
        self.runs = layer_runs(self.cfg)
        self.state = [{} for _ in self.runs]
        self.pos, self.eps, self.tanh = 0, self.cfg["norm"]["eps"], case["design"] == "Madevik"

    def norm(self, name, x):
        t = self.t
        return torch.tanh(t[name + ".alpha"] * x) * t[name] + t[name + ".b"] if self.tanh else rms(x, 1.0 + t[name], self.eps)

    def rotate(self, x, dims, base, pairs):
        """x [n, heads, size]: its first `dims` elements turned."""
        i = torch.arange(dims // 2, device="cuda", dtype=F)
        a = torch.arange(self.pos, self.pos + x.shape[0], device="cuda", dtype=F)[:, None, None] * base ** (-2.0 * i / dims)
        c, s = torch.cos(a), torch.sin(a)
        if pairs:
            u, v = x[..., 0:dims:2], x[..., 1:dims:2]
            turned = torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2)
        else:
            u, v = x[..., :dims // 2], x[..., dims // 2:dims]
            turned = torch.cat([u * c - v * s, v * c + u * s], -1)
        return torch.cat([turned, x[..., dims:]], -1)

    def softmax_sum(self, q, k, v, scale, window):
        """q [n, heads, e], k [keys, heads, e], v [keys, heads, f]."""
        n, keys = q.shape[0], k.shape[0]
        i = torch.arange(keys - n, keys, device="cuda")[:, None]
        j = torch.arange(keys, device="cuda")[None]
        out = torch.empty((n, q.shape[1], v.shape[2]), dtype=F, device="cuda")
        for a in range(q.shape[1]):
            s = (q[:, a] @ k[:, a].t()) * scale
            out[:, a] = torch.softmax(s.masked_fill((j > i) | (j <= i - window), -math.inf), -1) @ v[:, a]
        return out.flatten(1)

    def keep(self, state, name, x):
        state[name] = torch.cat([state[name], x]) if name in state else x
        return state[name]

    def conv(self, state, name, x, taps):
        past = state.get(name)
        n = taps.shape[1]
        past = torch.zeros((n - 1, x.shape[1]), dtype=F, device="cuda") if past is None else past
        all_ = torch.cat([past, x])
        state[name] = all_[all_.shape[0] - (n - 1):] if n > 1 else all_[:0]
        return torch.nn.functional.silu(sum(taps[:, i] * all_[i:i + x.shape[0]] for i in range(n)))

    def mixer(self, i, h, state):
        l, t, p, n = self.cfg["layers"][i], self.t, f"l{i}.mix.", h.shape[0]
        m = l["mixer"]
        H, d, v = m["heads"], m["dim"], m["vdim"]
        if l["type"] in ("gla", "channel_delta"):
            delta = l["type"] != "gla"
            z = (h @ t[p + "a1"].t()) @ t[p + "a2"].t()
            if delta:
                G = m["kv_heads"]
                q, k, x = (self.conv(state, c, h @ t[p + c].t(), t[f"{p}{c}.conv"]) for c in "qkv")
                unit = lambda a: a / torch.sqrt((a * a).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
                q, k = unit(q.view(n, G, d)) * d ** -0.5, unit(k.view(n, G, d))
                q, k = q.repeat_interleave(H // G, 1), k.repeat_interleave(H // G, 1)
                beta = torch.sigmoid(h @ t[p + "b"].t())
                decay = torch.exp(-torch.exp(t[p + "A_log"])[:, None] * torch.nn.functional.softplus((z + t[p + "dt_bias"]).view(n, H, d), threshold=1e9))
                gate = torch.sigmoid((h @ t[p + "g1"].t()) @ t[p + "g2"].t())
            else:
                q, k, x = (h @ t[p + "q"].t()).view(n, H, d) * d ** -0.5, (h @ t[p + "k"].t()).view(n, H, d), h @ t[p + "v"].t()
                decay = torch.exp(torch.nn.functional.logsigmoid(z + t[p + "a2.b"]) / m["tau"]).view(n, H, d)
                gate = torch.nn.functional.silu(h @ t[p + "g"].t())
            x = x.view(n, H, v)
            S = state.get("S")
            S = torch.zeros((H, d, v), dtype=F, device="cuda") if S is None else S
            out = torch.empty((n, H, v), dtype=F, device="cuda")
            for j in range(n):
                S = S * decay[j][..., None]
                u = beta[j][:, None] * (x[j] - (S * k[j][..., None]).sum(1)) if delta else x[j]
                S = S + k[j][..., None] * u[:, None]
                out[j] = (S * q[j][..., None]).sum(1)
            state["S"] = S
            return (rms(out, t[p + "norm"], self.eps).flatten(1) * gate) @ t[p + "o"].t()
        if l["type"] == "attention":
            G, rot = m["kv_heads"], m["rot"]
            key = (h @ t[p + "k"].t() + t[p + "k.b"]).view(n, G, d)
            q = self.rotate((h @ t[p + "q"].t() + t[p + "q.b"]).view(n, H, d), rot["dims"], rot["base"], False)
            val = self.keep(state, "v", key).repeat_interleave(H // G, 1)
            k = self.keep(state, "k", self.rotate(key, rot["dims"], rot["base"], False)).repeat_interleave(H // G, 1)
            return self.softmax_sum(q, k, val, m["scale"], m["mask"]["size"]) @ t[p + "o"].t()
        r, e = m["kv_rank"], m.get("rot_dim", 0)
        kv = h @ t[p + "dkv"].t()
        c = self.keep(state, "c", rms(kv[:, :r], t[p + "dkv.norm"], self.eps))
        hq = rms(h @ t[p + "dq"].t(), t[p + "dq.norm"], self.eps) @ t[p + "uq"].t() if e else h @ t[p + "q"].t()
        q = hq.view(n, H, d + e)
        k, val = (c @ t[p + "uk"].t()).view(-1, H, d), (c @ t[p + "uv"].t()).view(-1, H, v)
        if e:
            rot = m["rot"]
            kr = self.keep(state, "r", self.rotate(kv[:, None, r:], rot["dims"], rot["base"], True))
            q = torch.cat([q[..., :d], self.rotate(q[..., d:], rot["dims"], rot["base"], True)], -1)
            k = torch.cat([k, kr.expand(-1, H, -1)], -1)
        o = self.softmax_sum(q, k, val, m["scale"], m.get("mask", {}).get("size", 1 << 30))
        if self.tanh:
            o = (o.view(n, H, v) * torch.sigmoid(h @ t[p + "g"].t())[..., None]).flatten(1)
        return o @ t[p + "o"].t()

    def feed_forward(self, i, h):
        l, t, p = self.cfg["layers"][i], self.t, f"l{i}.mlp."
        if l["mlp"]["kind"] == "dense":
            return torch.nn.functional.gelu(h @ t[p + "up"].t()) @ t[p + "down"].t()
        r, out = l["mlp"]["router"], torch.zeros_like(h)
        score = torch.sigmoid(h @ t[p + "router"].t())
        chosen = torch.topk(score + t[p + "correction"], r["top"], -1).indices
        weight = torch.gather(score, 1, chosen)
        weight = weight / (weight.sum(-1, keepdim=True) + 1e-20) * r["scale"]
        for e in range(r["experts"]):
            row, place = torch.nonzero(chosen == e, as_tuple=True)
            if row.numel():
                x, q = h[row], f"{p}e{e}."
                out[row] += weight[row, place][:, None] * ((torch.nn.functional.silu(x @ t[q + "gate"].t()) * (x @ t[q + "up"].t())) @ t[q + "down"].t())
        return out

    def forward(self, ids):
        x = self.t["embed"][torch.as_tensor(np.asarray(ids), dtype=torch.long, device="cuda")].to(F)
        if not self.tanh:
            x = x * self.cfg["embedding"]["scale"]
        for run_, i in enumerate(self.runs):
            p = f"l{i}."
            a = self.mixer(i, self.norm(p + "norm1", x), self.state[run_])
            x = x + (self.cfg["residual_mult"] * a if self.tanh else self.norm(p + "norm1b", a))
            a = self.feed_forward(i, self.norm(p + "norm2", x))
            x = x + (self.cfg["residual_mult"] * a if self.tanh else self.norm(p + "norm2b", a))
        self.pos += len(ids)
        last, head = self.norm("final.norm", x[-1]), self.t["head"]
        return torch.cat([head[a:a + 32768].to(F) @ last for a in range(0, VOCAB, 32768)])


def exact(case, seed):
    if case["kind"] == "linear":
        weights, x, hidden = linear_inputs(case, seed)
        up, gate, down = (a.to(F) @ (q.to(F) * s.to(F)) for a, (q, s) in zip((x, x, hidden), weights))
        return {"up": up, "gate": gate, "down": down}
    r = requests(case, seed)
    if case["kind"] == "net":
        m = NetExact(case, seed)
        logits = m.forward(r["prompt"])
        out = {"logits": logits}
        if case["steps"]:
            ids = [int(torch.argmax(logits))]
            for _ in range(case["steps"]):
                ids.append(int(torch.argmax(m.forward(ids[-1:]))))
            out["ids"], out["last_logits"] = np.array(ids, np.int32), m.forward(ids[-1:])
        return out
    m = GemmaExact(case["shape"], seed)
    logits = m.forward(r["prompt"], True)
    ids = m.generate(logits, case["steps"], case["minp"], r["rand"][0])
    out = {"logits": logits, "ids": np.array(ids, np.int32)}
    if case["turn"]:
        out["turn_logits"] = m.forward(np.concatenate([ids[-1:], r["turn"]]), False)
        ids = m.generate(out["turn_logits"], case["answer"], case["minp"], r["rand"][1])
        out["answer"] = np.array(ids, np.int32)
    if case["steps"]:
        out["last_logits"] = m.forward(ids[-1:], False)
    return out
