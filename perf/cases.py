"""Timed cases of the token loop: what a program does with libember.so.

Every case is one call (or one enqueued call) of the public C API, made as
the ctypes binding makes it: ``ember_forward`` for a decode step,
``ember_prefill`` for a prompt or the next turn of a conversation,
``ehip_sample_noalloc`` for a token from logits on the device and
``ehip_quantize_rows`` for the requantizer's matrices.  The API has no entry
point for a single layer, so the model cases are whole calls that return the
logits; they cover the shapes of ``emberllm_amd.configs`` in the three weight
encodings of the format and with both KV cache types.

The models are the seeded synthetic files of ``emberllm_amd.configs`` (their
weights do not depend on the seed of a case; the token ids do).
"""
import ctypes
import math

import numpy as np
import torch

from emberllm_amd import _native, configs, emberllm

F32, Q8, Q4 = _native.DT_F32, _native.DT_Q8_0, _native.DT_Q4_0
WINDOW = 64          # decode steps before a decode case returns to its first position
MAX_SAMPLE = 262144  # logits that ehip_sample_noalloc takes


# ----------------------------------------------------------------- cases ----
def decode(name, model, depth, kv16=False, layers=0):
    return dict(name=name, kind="decode", model=model, depth=depth, kv16=kv16, layers=layers)


def prompt(name, model, n, kv16=False, layers=0):
    return dict(name=name, kind="prompt", model=model, n=n, kv16=kv16, layers=layers)


def turn(name, model, history, n, kv16=False, layers=0):
    return dict(name=name, kind="turn", model=model, history=history, n=n, kv16=kv16, layers=layers)


def listed():
    return [
        # a serving loop picking a token from logits it holds on the GPU: the
        # chat defaults over the largest vocabulary of the model shapes
        dict(name="sample_151936", kind="sample", n=151936, temperature=0.8, top_k=40, top_p=0.9, min_p=0.0, repeat=1.0),
        # generating text, one step at a time, each step's logits on the host:
        # a small model early in its context
        decode("decode_stories110m", "stories110m", 128),
        # a deep and narrow model, half-way through a long document, fp16 cache
        decode("decode_smollm2_f16kv", "smollm2_135m", 1000, kv16=True),
        # the headline: the 0.6B shape at the end of a 4k context
        decode("decode_qwen3_4096", "qwen3_06b", 4096),
        # the 4-bit file of the same shape at a chat's length
        decode("decode_qwen3_q4", "qwen3_06b_q4", 512),
        # a converted file that has not been quantized
        decode("decode_stories110m_f32", "stories110m_f32", 300),
        # a conversation: each pass is the next short message after everything
        # said so far, so no two passes have the same first position
        turn("turn_qwen3_23", "qwen3_06b", 517, 23, kv16=True),
        # the first prompt of a session: a short paragraph to the unquantized
        # file, a page to the shape with biases and the largest FFN (a third
        # of its layers: the comment at tolerance()), the benchmark's 512
        # tokens to the 4-bit file, a 4k document to the headline shape
        prompt("prompt_stories110m_f32", "stories110m_f32", 200),
        prompt("prompt_qwen25_257", "qwen25_05b", 257, layers=8),
        prompt("prompt_qwen3_q4_512", "qwen3_06b_q4", 512),
        prompt("prompt_qwen3_4096", "qwen3_06b", 4096),
        # preparing a file: the feed-forward matrices of one layer to Q8_0
        dict(name="quantize_ffn_q8", kind="quantize", rows=3072, cols=1024, count=3, target=Q8),
    ]


def log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prompt", "prompt", "prompt", "turn", "turn", "sample", "quantize"])
    if kind == "sample":
        greedy = rng.random() < 0.2
        return dict(kind="sample", n=log_uniform(rng, 20000, MAX_SAMPLE), temperature=0.0 if greedy else round(rng.uniform(0.3, 1.5), 3),
                    top_k=rng.randint(1, 64), top_p=rng.choice([0.0, round(rng.uniform(0.5, 0.99), 3)]),
                    min_p=rng.choice([0.0, 0.05]), repeat=rng.choice([1.0, 1.1]))
    if kind == "quantize":
        cols = 32 * log_uniform(rng, 4, 160)
        rows = log_uniform(rng, 64, 12000000 // cols)
        return dict(kind="quantize", rows=rows, cols=cols, count=rng.randint(1, max(1, min(7, 12000000 // (rows * cols)))),
                    target=rng.choice([Q8, Q4]))
    model = rng.choice(["stories110m", "smollm2_135m", "qwen25_05b", "qwen3_06b", "qwen3_06b_q4", "stories110m_f32"])
    case = dict(kind=kind, model=model, kv16=rng.random() < 0.4, layers=8 if model == "qwen25_05b" else 0)
    longest = min(config(case)["max_seq_len"], 6000)
    if kind == "decode":
        case["depth"] = log_uniform(rng, 4, longest - WINDOW)
    elif kind == "prompt":
        case["n"] = log_uniform(rng, 2, 512 if model == "stories110m_f32" else min(longest, 4000))
    else:
        case["history"] = log_uniform(rng, 16, min(longest, 3000) - 400)
        case["n"] = log_uniform(rng, 2, 300)
    return case


# ---------------------------------------------------------------- models ----
def config(case):
    model = case["model"]
    cfg = dict(configs.REAL[model[:-4] if model.endswith("_f32") else model])
    if model.endswith("_f32"):
        cfg["dtype"] = F32
    if case["layers"]:
        cfg["n_layers"] = case["layers"]
    return cfg


def model_file(case):
    cfg = config(case)
    return configs.model_path(f"perf_{case['model']}_{cfg['n_layers']}", cfg)


def context(case):
    """The context a program asks for: the next power of two that holds the
    case and the room it goes on in."""
    need = {"decode": lambda: case["depth"] + WINDOW, "prompt": lambda: case["n"] + 64,
            "turn": lambda: case["history"] + 24 * case["n"]}[case["kind"]]()
    cap = min(config(case)["max_seq_len"], 8192)
    return min(cap, max(512, 1 << (need - 1).bit_length()))


def token_ids(case, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(0, config(case)["vocab_size"], (context(case),), generator=g, dtype=torch.int32).numpy()


class Session:
    """A loaded model, one state and the conversation's token ids."""

    def __init__(self, case, seed):
        self.eng = emberllm.Engine(model_file(case), ctx=context(case), kv_fp16=case["kv16"])
        self.lib, self.m, self.st, self.vocab = self.eng.lib, self.eng.m, self.eng.st, self.eng.vocab
        self.ids = token_ids(case, seed)
        self.step = 0
        self.buffer = type("Logits", (ctypes.c_float * self.vocab,), {})

    def logits(self, p):
        """The state's own logits, which live as long as somebody holds them."""
        b = self.buffer.from_address(ctypes.addressof(p.contents))
        b.session = self
        return np.frombuffer(b, dtype=np.float32)

    def prefill(self, start, n):
        part = self.ids[start:start + n]
        return self.logits(self.lib.ember_prefill(self.m, self.st, part.ctypes.data_as(ctypes.POINTER(ctypes.c_int)), n, start))

    def forward(self, pos):
        return self.logits(self.lib.ember_forward(self.m, self.st, int(self.ids[pos]), pos))


def sampler_params(case, history_cap):
    smp = _native.EmberSampler()
    smp.temperature, smp.top_k, smp.top_p, smp.min_p = case["temperature"], case["top_k"], case["top_p"], case["min_p"]
    smp.repeat_penalty, smp.hist_cap = case["repeat"], history_cap
    return smp


def logits_of(case, seed):
    """Logits with the spread of a language model's: most tokens far below a few dozen candidates."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(case["n"], generator=g) * 2.5
    top = torch.randint(0, case["n"], (48,), generator=g)
    x[top] += 4.0 + 6.0 * torch.rand(48, generator=g)
    history = top[torch.randint(0, 48, (64,), generator=g)].to(torch.int32)
    return x, history


def matrices(case, seed):
    g = torch.Generator().manual_seed(seed)
    return [(torch.randn(case["rows"], case["cols"], generator=g) * 0.02).numpy() for _ in range(case["count"])]


# --------------------------------------------------------------- prepare ----
def prepare(case, seed):
    kind = case["kind"]
    if kind == "sample":
        x, history = logits_of(case, seed)
        dev = dict(logits=x.cuda(), rng=torch.tensor([seed * 2 + 1], dtype=torch.int64).cuda(), history=history.cuda(),
                   meta=torch.tensor([len(history), 0], dtype=torch.int32).cuda(), token=torch.zeros(1, dtype=torch.int32).cuda())
        lib = _native.lib()
        if lib.ehip_noalloc_setup() != 0:
            raise RuntimeError(_native.last_error())
        return dict(kind=kind, lib=lib, smp=sampler_params(case, len(history)), **dev)
    if kind == "quantize":
        src = matrices(case, seed)
        block = 34 if case["target"] == Q8 else 18
        dst = [np.zeros((case["rows"], case["cols"] // 32 * block), dtype=np.uint8) for _ in src]
        jobs = (_native.EhipQuantJob * len(src))()
        for j, a, b in zip(jobs, src, dst):
            j.src, j.rows, j.cols, j.dtype, j.dst = a.ctypes.data, case["rows"], case["cols"], case["target"], b.ctypes.data
        return dict(kind=kind, lib=_native.lib(), src=src, dst=dst, jobs=jobs)
    s = Session(case, seed)
    if kind == "decode":
        s.prefill(0, case["depth"])
    elif kind == "turn":
        s.prefill(0, case["history"])
    return dict(kind=kind, case=case, session=s, ctx=context(case))


# ------------------------------------------------------------------- run ----
def run(state):
    kind = state["kind"]
    if kind == "sample":
        t = state
        rc = t["lib"].ehip_sample_noalloc(t["logits"].data_ptr(), t["logits"].numel(), ctypes.byref(t["smp"]), t["rng"].data_ptr(),
                                          t["history"].data_ptr(), t["meta"].data_ptr(), t["token"].data_ptr(),
                                          torch.cuda.current_stream().cuda_stream)
        if rc != 0:
            raise RuntimeError(_native.last_error())
        return dict(token=t["token"], rng=t["rng"], history=t["history"], meta=t["meta"], logits=t["logits"])
    if kind == "quantize":
        if state["lib"].ehip_quantize_rows(state["jobs"], len(state["src"])) != 0:
            raise RuntimeError(_native.last_error())
        return state["dst"]
    s, case = state["session"], state["case"]
    if kind == "decode":
        pos = case["depth"] + s.step
        s.step = (s.step + 1) % WINDOW
        return s.forward(pos)
    if kind == "prompt":
        return s.prefill(0, case["n"])
    start = case["history"] + s.step * case["n"]
    s.step = s.step + 1 if start + 2 * case["n"] <= state["ctx"] else 0
    return s.prefill(start, case["n"])


# ------------------------------------------------------------------ work ----
def work(case):
    """Each weight, key, value and input read once, each output written once;
    the products' multiply-adds and causal attention's."""
    kind = case["kind"]
    if kind == "sample":
        return dict(bytes=4 * case["n"], flops=4 * case["n"])
    if kind == "quantize":
        values = case["rows"] * case["cols"] * case["count"]
        return dict(bytes=values * (4 + (34 if case["target"] == Q8 else 18) / 32), flops=4 * values)
    c = config(case)
    dim, hid, L, V = c["dim"], c["hidden_dim"], c["n_layers"], c["vocab_size"]
    qd, kvd = c["n_heads"] * c["head_dim"], c["n_kv_heads"] * c["head_dim"]
    per = {F32: 4.0, Q8: 34 / 32, Q4: 18 / 32}[c["dtype"]]
    head_per = 4.0 if c["dtype"] == F32 else 34 / 32
    layer = dim * (qd + 2 * kvd) + qd * dim + 3 * dim * hid
    n = 1 if kind == "decode" else case["n"]
    start = {"decode": lambda: case["depth"] + WINDOW // 2, "prompt": lambda: 0,
             "turn": lambda: (case["history"] + context(case)) // 2}[kind]()
    e = 2 if case["kv16"] else 4
    nbytes = L * layer * per + V * dim * head_per + n * dim * head_per + 2 * L * (start + n) * kvd * e + 4 * V
    keys = n * start + n * (n + 1) // 2
    return dict(bytes=nbytes, flops=2 * n * L * layer + 2 * V * dim + 4 * L * keys * qd)


# ------------------------------------------------------------- tolerance ----
def tolerance(case):
    """Sampling and quantizing give whole numbers and bytes: exact.

    An unquantized model's logits are sums in 32 bits: with its attention in
    another order of summation they move by 1.3e-6 relative L2 (6e-6 of the
    logits' size at most), and with an fp16 cache by 1.9e-5 (9e-5), a sum in
    another order moving cached values by one step of fp16.

    A quantized model quantizes the input of every product to Q8_0 (this is
    the format's arithmetic), so a change in the last bit of one sum can move
    an activation code, and the moved code goes through every layer after it.
    With the attention's sums in another order the logits move by 1.1e-2 to
    1.6e-2 (7e-2 at most); two builds of the reference implementation that
    sum in other orders differ by as much.  The shape with biases differs by
    2.4e-2 at its full depth (3.0e-2 at most) and by 1.7e-2 to 2.3e-2 with a
    third of its layers, which its cases therefore have."""
    if case["kind"] in ("sample", "quantize"):
        return "exact"
    if config(case)["dtype"] == F32:
        return {"rel": 8e-5, "max": 4e-4} if case["kv16"] else {"rel": 5e-6, "max": 2.5e-5}
    return {"rel": 0.03, "max": 0.2}


# ----------------------------------------------------------------- exact ----
class File:
    """The tensors of an .ember file as float64, read with numpy alone."""

    HEADER = np.dtype([("head", "S16"), ("shape", "<i4", 8), ("theta", "<f4"), ("eps", "<f4"), ("flags", "<u4"),
                       ("rope", "<i4"), ("ids", "<i4", 3), ("n_tensors", "<i4"), ("skip", "V16"), ("where", "<u8", 4)])
    ENTRY = np.dtype([("name", "S48"), ("dtype", "<i4"), ("ndim", "<i4"), ("shape", "<i4", 4), ("offset", "<u8"), ("nbytes", "<u8")])

    def __init__(self, path, device):
        self.raw, self.device = np.memmap(path, dtype=np.uint8, mode="r"), device
        h = self.raw[:self.HEADER.itemsize].view(self.HEADER)[0]
        table = int(h["where"][2])
        rows = self.raw[table:table + int(h["n_tensors"]) * self.ENTRY.itemsize].view(self.ENTRY)
        self.entry = {r["name"].decode(): r for r in rows}

    def __contains__(self, name):
        return name in self.entry

    def get(self, name, rows=None):
        t = self.entry[name]
        off, shape, dtype = int(t["offset"]), [int(v) for v in t["shape"][:int(t["ndim"])]], int(t["dtype"])
        b = np.asarray(self.raw[off:off + int(t["nbytes"])])
        if dtype == F32:
            w = b.view("<f4").reshape(shape)
            return torch.from_numpy(np.array(w if rows is None else w[rows])).to(self.device).double()
        w = b.reshape(shape[0], -1)
        w = torch.from_numpy(np.array(w if rows is None else w[rows])).to(self.device)
        w = w.reshape(w.shape[0], shape[1] // 32, -1)
        scale = w[:, :, :2].contiguous().view(torch.float16).double()
        q = w[:, :, 2:]
        q = q.view(torch.int8).double() if dtype == Q8 else torch.cat([(q & 15).double(), (q >> 4).double()], 2) - 8
        return (q * scale).reshape(w.shape[0], shape[1])


def exact_logits(case, ids):
    """The model's function on ids in 64 bits: nothing is rounded but the
    stored weights and the rotary angles, which the format has in 32 bits.
    (The Q8_0 inputs of the products are the path's precision, and are left
    out here: both sides of a comparison are then off by their size.)"""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    c = config(case)
    f = File(model_file(case), dev)
    hd, nh, nkv, n = c["head_dim"], c["n_heads"], c["n_kv_heads"], len(ids)
    base = np.float32(1) / np.power(float(c["rope_theta"]), 2.0 * np.arange(hd // 2) / hd).astype(np.float32)
    ang = torch.from_numpy(np.arange(n, dtype=np.float32)[:, None] * base[None, :]).to(dev).double()
    cos, sin = ang.cos()[:, None, :], ang.sin()[:, None, :]

    def norm(x, w):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + float(np.float32(c["norm_eps"]))) * w

    def rotate(x):
        if c["rope_style"] == _native.ROPE_NEOX:
            a, b = x[..., :hd // 2], x[..., hd // 2:]
            return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)

    hidden = torch.ones(n, n, dtype=torch.bool, device=dev).triu(1)
    x = f.get("tok_embeddings", np.asarray(ids))
    for l in range(c["n_layers"]):
        t = lambda s: f.get(f"layers.{l}.{s}")  # noqa: E731
        y = norm(x, t("attn_norm"))
        q, k, v = (y @ t(w).T + (t(w + "_bias") if f"layers.{l}.{w}_bias" in f else 0) for w in ("wq", "wk", "wv"))
        q, k, v = q.view(n, nh, hd), k.view(n, nkv, hd), v.view(n, nkv, hd)
        if f"layers.{l}.q_norm" in f:
            q, k = norm(q, t("q_norm")), norm(k, t("k_norm"))
        q, k = rotate(q), rotate(k)
        o = torch.empty(n, nh, hd, dtype=torch.float64, device=dev)
        for h in range(nh):
            g = h // (nh // nkv)
            p = (q[:, h] @ k[:, g].T.contiguous() / math.sqrt(hd)).masked_fill(hidden, -math.inf).softmax(-1)
            o[:, h] = p @ v[:, g]
        x = x + o.reshape(n, nh * hd) @ t("wo").T
        y = norm(x, t("ffn_norm"))
        x = x + (torch.nn.functional.silu(y @ t("w1").T) * (y @ t("w3").T)) @ t("w2").T
    y = norm(x[-1], f.get("final_norm"))
    return (f.get("lm_head" if "lm_head" in f else "tok_embeddings") @ y).cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "quantize":
        return None
    if kind == "sample":
        x, history = logits_of(case, seed)
        x = x.double()
        seen = history.unique().long()
        if case["repeat"] != 1.0:
            r = float(np.float32(case["repeat"]))
            x[seen] = torch.where(x[seen] > 0, x[seen] / r, x[seen] * r)
        return dict(token=None, rng=None, history=None, meta=None, logits=x.numpy())
    end = {"decode": lambda: case["depth"] + 1, "prompt": lambda: case["n"], "turn": lambda: case["history"] + case["n"]}[kind]()
    return exact_logits(case, token_ids(case, seed)[:end])
