"""The performance cases of this library: what its users have it do, at the sizes they do it.

Six kinds of work, each through the public Python face:

  linear    one fused decode+GEMV / GEMM call on packed tensors that share their activations (gemv, gemm)
  decode    decode steps of a Llama-shaped model: one sequence, or independent sequences with caches of their own
  prompt    a prompt of a Llama-shaped model entered in passes of 512 rows
  turn      a chat turn of a Gamilorn or Davasun model: a prompt, then decode steps of one sequence
  moe       a Mixtral-shaped mixture-of-experts feed-forward
  codec     packing a bf16 matrix on the GPU and unpacking it again

Decode steps are given their tokens (as when a text is scored, or a sampler outside the engine picks them), so that a run
always takes the same path.  Models have four layers: the layers of a deeper one repeat the same launches.
"""
import importlib.util
import json
import math
import os
import random
import shutil
import struct
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEV = "cuda"
VOCAB, LAYERS, EPS, THETA = 32000, 4, 1e-5, 500000.0
MAX_SEQ = 4352                        # positions of the one-sequence cache (largest prompt and some)
PROMPT_ROWS = 512                     # prompt tokens per pass of the layer stack
LLAMA = {2048: dict(n_embd=2048, n_head=16, n_head_kv=4, n_ff=8192), 4096: dict(n_embd=4096, n_head=32, n_head_kv=8, n_ff=14336)}
MOE = dict(experts=8, top_k=2, width=4096, ff=14336)


def package():
    """The package's folder name is no identifier: it is imported under the name its own tests use."""
    name = "turbo_lossless_amd"
    if name not in sys.modules:
        folder = os.path.join(ROOT, "turbo-lossless_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(folder, "__init__.py"), submodule_search_locations=[folder])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


def listed():
    return [
        # one attention output projection of a single sequence: the smallest call a decode step makes
        dict(name="linear_o_b1", kind="linear", rows="4096", K=4096, B=1),
        # three tensors of odd sizes that share a ragged batch of a few sequences
        dict(name="linear_ragged_b21", kind="linear", rows="5001,1250,1250", K=2560, B=21),
        # interactive use: one sequence in the middle of a conversation
        dict(name="decode_b1", kind="decode", width=4096, batch=1, context=700, steps=8),
        # a local server with a few users
        dict(name="decode_b8", kind="decode", width=4096, batch=8, context=1000, steps=4),
        # a busy server
        dict(name="decode_b64", kind="decode", width=4096, batch=64, context=1000, steps=2),
        # offline generation: as many sequences as the headline batch, short contexts
        dict(name="decode_b256", kind="decode", width=4096, batch=256, context=200, steps=2),
        # the time to the first token of a short question, and of a long document
        dict(name="prompt_100", kind="prompt", width=4096, tokens=100),
        dict(name="prompt_2048", kind="prompt", width=4096, tokens=2048),
        # chat turns of the two other families
        dict(name="gamilorn_turn", kind="turn", family="gamilorn", tokens=1500, steps=8),
        dict(name="davasun_turn", kind="turn", family="davasun", tokens=700, steps=8),
        # the feed-forward of a mixture of experts while a server decodes a batch of sequences
        dict(name="moe_40", kind="moe", tokens=40),
        # converting a checkpoint's largest layer tensor and reading it back
        dict(name="codec_gate", kind="codec", M=14336, K=4096),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "decode", "decode", "prompt", "turn", "moe", "codec"])
    if kind == "linear":
        K = rng.choice([2048, 2560, 4096, 5504, 8192, 14336, 64 * rng.randint(8, 128)])
        rows = [_log(rng, 256, 16384) for _ in range(rng.choice([1, 1, 2, 3]))]
        return dict(kind=kind, rows=",".join(str(r) for r in rows), K=K, B=_log(rng, 1, 512))
    if kind == "decode":
        batch = _log(rng, 1, 256)
        context = _log(rng, 8, min(1900, 65536 // batch))
        return dict(kind=kind, width=rng.choice(sorted(LLAMA)), batch=batch, context=context, steps=2 if batch > 16 else 4)
    if kind == "prompt":
        return dict(kind=kind, width=rng.choice(sorted(LLAMA)), tokens=_log(rng, 16, 2048))
    if kind == "turn":
        family = rng.choice(["gamilorn", "davasun"])
        return dict(kind=kind, family=family, tokens=_log(rng, 16, 1500 if family == "gamilorn" else 700), steps=8)
    if kind == "moe":
        return dict(kind=kind, tokens=_log(rng, 1, 256))
    return dict(kind=kind, M=_log(rng, 512, 14336), K=rng.choice([2048, 2560, 4096, rng.randint(500, 4096)]))


# ---- inputs ------------------------------------------------------------------------------------------------------------
def _gen(seed, k=0):
    return torch.Generator(device=DEV).manual_seed(1000003 * (seed + 1) + k)


def _weight(M, K, g, p_outlier=3e-4):
    """bf16 [M, K] ~ N(0, 0.02), a fraction of the entries 2 to 30 in size, of either sign: those need an escape.  (The
    smallest weights are kept inside the coded range and every outlier has a stretch of the matrix to itself, so that the length of
    the escape list does not depend on the seed.)"""
    w = torch.randn((M, K), generator=g, device=DEV) * 0.02
    w = torch.where(w.abs() < 2.0 ** -16, 2.0 ** -16, w).clamp_(-0.12, 0.12)
    n = int(M * K * p_outlier)
    if n:
        stretch = M * K // n
        at = torch.arange(n, device=DEV) * stretch + torch.randint(0, stretch, (n,), generator=g, device=DEV)
        big = 2.0 + 28.0 * torch.rand(n, generator=g, device=DEV)
        w.view(-1)[at] = torch.where(torch.rand(n, generator=g, device=DEV) < 0.5, -big, big)
    return w.to(torch.bfloat16)


def _linear_inputs(case, seed):
    g = _gen(seed)
    K = case["K"]
    W = [_weight(int(r), K, g) for r in case["rows"].split(",")]
    return W, torch.randn((case["B"], K), generator=g, device=DEV).to(torch.bfloat16)


def _moe_inputs(case, seed):
    g = _gen(seed)
    n, ff = MOE["width"], MOE["ff"]
    W = [[_weight(M, K, g, 0.0) for M, K in ((ff, n), (ff, n), (n, ff))] for _ in range(MOE["experts"])]
    X = torch.randn((case["tokens"], n), generator=g, device=DEV).to(torch.bfloat16)
    top, ids = torch.topk(torch.randn((case["tokens"], MOE["experts"]), generator=g, device=DEV), MOE["top_k"], dim=-1)
    return W, X, ids.contiguous(), torch.softmax(top, dim=-1).contiguous()


def _decode_inputs(case, seed):
    """Prompts of ragged lengths, and the tokens of the steps."""
    rng = random.Random(seed)
    prompts = [[rng.randrange(VOCAB) for _ in range(max(1, case["context"] - rng.randrange(case["context"] // 2 + 1)))] for _ in range(case["batch"])]
    return prompts, [[rng.randrange(VOCAB) for _ in range(case["batch"])] for _ in range(case["steps"])]


def _tokens(seed, n):
    rng = random.Random(seed)
    return [rng.randrange(VOCAB) for _ in range(n)]


def _gamilorn_config():
    left = {"heads": 16, "kv_heads": 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "mask": {"size": 1024, "keep_first": 4}}
    layer = {"type": "parallel", "mlp": {"kind": "dense", "ff": 8192},
             "mixer": {"left": left, "right": {"heads": 16, "dim": 64}, "left_scale": 1.0, "right_scale": 1.0}}
    return {"architecture": "Gamilorn", "layers": [layer] * LAYERS, "vocab": VOCAB, "width": 2048, "max_positions": 8192, "norm": {"eps": EPS},
            "logit_softcap": 30.0}


def _davasun_config():
    mlstm = {"type": "mlstm", "mixer": {"heads": 4, "dim": 256, "vdim": 512, "gate_cap": 15.0}, "mlp": None}
    latent = {"type": "latent_attention", "mlp": {"kind": "dense", "ff": 5504, "limit": 7.0},
              "mixer": {"heads": 16, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 256, "scale": 192 ** -0.5, "rot": {"dims": 64, "base": 10000.0}}}
    return {"architecture": "Davasun", "layers": [mlstm, latent] * (LAYERS // 2), "vocab": VOCAB, "width": 2048, "norm": {"eps": EPS},
            "logit_scale": 1.0, "loop": None}


def _family_checkpoint(family, seed):
    """(configuration, {name: bf16 tensor on the GPU}) of a random model, every mechanism at a working point."""
    g = _gen(seed)
    cfg = _gamilorn_config() if family == "gamilorn" else _davasun_config()
    n = cfg["width"]
    randn = lambda *s: torch.randn(s, generator=g, device=DEV)
    mat = lambda m, k, gain=1.0: randn(m, k) * (gain / math.sqrt(k))
    vec = lambda m, mean=0.0, dev=0.3: mean + dev * randn(m)
    gain = lambda: 0.6 + 0.9 * torch.rand((), generator=g, device=DEV)
    t = {"embed": randn(VOCAB, n), "head": mat(VOCAB, n)}
    for i, L in enumerate(cfg["layers"]):
        p, c = "l%d." % i, L["mixer"]
        if family == "gamilorn":
            a, b, ff, rank = c["left"], c["right"], L["mlp"]["ff"], 64
            d = b["heads"] * b["dim"]
            t[p + "norm1"], t[p + "norm2"] = vec(n), vec(n)
            for name, m in (("q", a["heads"] * a["dim"]), ("k", a["kv_heads"] * a["dim"]), ("v", a["kv_heads"] * a["vdim"])):
                t[p + "mix.left." + name], t[p + "mix.left.%s.b" % name] = mat(m, n), vec(m)
            t[p + "mix.left.pb"], t[p + "mix.left.o"] = vec(a["heads"], -4.0), mat(n, a["heads"] * a["vdim"], 0.7)
            for name in "rkvga":
                t[p + "mix.right." + name] = mat(d, n)
            t[p + "mix.right.a.b"], t[p + "mix.right.w0"] = vec(d, 0.0, 1.5), vec(d, -3.0, 3.0)
            t[p + "mix.right.w1"], t[p + "mix.right.w2"] = mat(rank, n), mat(d, rank)
            t[p + "mix.right.norm"], t[p + "mix.right.o"] = vec(d, 1.0), mat(n, d, 0.7)
            t[p + "mlp.up"], t[p + "mlp.down"], t[p + "mlp.act"] = mat(ff, n), mat(n, ff, 0.5), vec(2, 0.6, 0.4)
            continue
        H, hv = c["heads"], c["heads"] * c["vdim"]
        t[p + "norm1"], t[p + "norm1b"] = gain(), gain()
        if L["type"] == "mlstm":
            t[p + "mix.q"] = mat(H * c["dim"], n, 1.5)
            t[p + "mix.k"] = 0.8 * t[p + "mix.q"] + mat(H * c["dim"], n, 0.9)      # (keys like their queries: the normaliser seldom cancels)
            t[p + "mix.v"], t[p + "mix.g"], t[p + "mix.norm"] = mat(hv, n), mat(hv, n), vec(hv, 1.0)
            t[p + "mix.i"], t[p + "mix.i.b"] = mat(H, n, 2.0), vec(H, -1.0, 1.5)
            t[p + "mix.f"], t[p + "mix.f.b"] = mat(H, n, 2.0), vec(H, 3.0, 1.5)
        else:
            d, r, R = c["dim"], c["rot_dim"], c["kv_rank"]
            t[p + "mix.q"], t[p + "mix.g"] = mat(H * (d + r), n, 1.5), mat(H, n)
            t[p + "mix.dkv"], t[p + "mix.dkv.norm"] = mat(R + r, n, 1.2), vec(R, 1.0)
            t[p + "mix.uk"], t[p + "mix.uv"] = mat(H * d, R), mat(hv, R)
        t[p + "mix.o"] = mat(n, hv)
        if L["mlp"]:
            ff = L["mlp"]["ff"]
            t[p + "norm2"], t[p + "norm2b"] = gain(), gain()
            t[p + "mlp.gate"], t[p + "mlp.up"], t[p + "mlp.down"] = mat(ff, n, 1.5), mat(ff, n, 1.5), mat(n, ff)
    if family == "gamilorn":
        t["pos"], t["final.norm"] = 0.3 * randn(cfg["max_positions"], n), vec(n)
    else:
        t["embed.norm"], t["final.norm"] = gain(), gain()
    return cfg, {k: v.to(torch.bfloat16) for k, v in t.items()}


class _Folder:
    """A folder in memory where there is one, gone at the end of the block."""

    def __enter__(self):
        self.path = tempfile.mkdtemp(prefix="t12_cases_", dir="/dev/shm" if os.access("/dev/shm", os.W_OK) else None)
        return self.path

    def __exit__(self, *a):
        shutil.rmtree(self.path, ignore_errors=True)


def _write_checkpoint(path, cfg, tensors):
    with open(os.path.join(path, "config.json"), "w") as f:
        json.dump(cfg, f)
    header, at = {}, 0
    for name, t in tensors.items():
        header[name] = {"dtype": "BF16", "shape": list(t.shape), "data_offsets": [at, at + 2 * t.numel()]}
        at += 2 * t.numel()
    h = json.dumps(header).encode()
    h += b" " * (-len(h) % 8)
    with open(os.path.join(path, "model.safetensors"), "wb") as f:
        f.write(struct.pack("<Q", len(h)) + h)
        for t in tensors.values():
            f.write(memoryview(t.reshape(-1).view(torch.int16).cpu().numpy()).cast("B"))


class _Served:
    """An engine that is closed when its last reference goes."""

    def __init__(self, engine):
        self.engine = engine

    def __del__(self):
        try:
            self.engine.close()
        except Exception:  # the interpreter is ending
            pass


def _llama(case, seed, batch=1):
    t12 = package()
    cfg = dict(LLAMA[case["width"]], n_vocab=VOCAB, n_layer=LAYERS, n_ctx=MAX_SEQ, rope_theta=THETA, rms_norm_eps=EPS)
    # without outliers 0.02 % of the weights need an escape (the smallest ones); with them a random model's logits hang on a few of them
    return t12.Engine.synthetic(cfg, seed=7000 + 1000 * (seed % 100003), max_seq=MAX_SEQ, batch=batch, p_outlier=0.0,
                                per_sequence=2048 if batch > 1 else 0)


def prepare(case, seed):
    t12 = package()
    kind = case["kind"]
    if kind == "linear":
        W, X = _linear_inputs(case, seed)
        packed = [t12.pack_device(w) for w in W]
        X = X.view(torch.int16)
        shape = (lambda w: (w.M,)) if case["B"] == 1 else (lambda w: (case["B"], w.M))
        return dict(kind=kind, W=packed, X=X[0] if case["B"] == 1 else X, out=[torch.empty(shape(w), device=DEV) for w in packed])
    if kind == "decode":
        prompts, steps = _decode_inputs(case, seed)
        e = _llama(case, seed, case["batch"])
        for b, p in enumerate(prompts):
            if case["batch"] == 1:
                e.prefill_rows(p, PROMPT_ROWS)
            else:
                e.prefill(b, p)
        e.sync()
        return dict(kind=kind, e=_Served(e), at=[len(p) for p in prompts], steps=steps)
    if kind == "prompt":
        return dict(kind=kind, e=_Served(_llama(case, seed)), tokens=_tokens(seed, case["tokens"]), steps=[])
    if kind == "turn":
        cfg, tensors = _family_checkpoint(case["family"], seed)
        with _Folder() as path:
            _write_checkpoint(path, cfg, tensors)
            e = t12.Engine.load(path, batch=1)
        return dict(kind=kind, e=_Served(e), tokens=_tokens(seed, case["tokens"]), steps=[[t] for t in _tokens(seed + 77, case["steps"])])
    if kind == "moe":
        from turbo_lossless_amd import moe
        W, X, ids, w = _moe_inputs(case, seed)
        layer = moe.MoeLayer([moe.Expert(*[t12.pack_device(x) for x in e]) for e in W])
        return dict(kind=kind, layer=layer, X=X.view(torch.int16), ids=ids, w=w, out=torch.empty((case["tokens"], MOE["width"]), device=DEV))
    return dict(kind=kind, W=_weight(case["M"], case["K"], _gen(seed)), out=torch.empty((case["M"], case["K"]), dtype=torch.int16, device=DEV))


def run(s):
    t12 = package()
    kind = s["kind"]
    if kind == "linear":
        return (t12.gemv if s["X"].dim() == 1 else t12.gemm)(s["W"], s["X"], s["out"])
    if kind == "moe":
        return s["layer"](s["X"], s["ids"], s["w"], out=s["out"])
    if kind == "codec":
        p = t12.pack_device(s["W"])
        return [p.sm, p.gr, p.row_off, p.cols, p.correct, p.wrong, t12.decompress(p, out=s["out"])]
    e = s["e"].engine
    if kind == "decode":
        e.set_positions(s["at"])
    else:
        e.set_positions([0])
        e.prefill_rows(s["tokens"], PROMPT_ROWS)
    for tokens in s["steps"]:
        e.forward(tokens)
    return e.logits(VOCAB)


# ---- what a pass cannot do without -------------------------------------------------------------------------------------
def _llama_weights(width):
    c = LLAMA[width]
    n, kv = c["n_embd"], c["n_head_kv"] * (c["n_embd"] // c["n_head"])
    return LAYERS * (2 * n * n + 2 * n * kv + 3 * n * c["n_ff"]), n * VOCAB, kv


def _family_weights(family):
    n = 2048
    if family == "gamilorn":
        return LAYERS * (n * (2048 + 1024 + 5 * 1024 + 64) + n * (2048 + 1024) + 2 * n * 8192), n * VOCAB
    return LAYERS // 2 * (n * (2048 + 3 * 2048 + 8) + n * (16 * 192 + 256 + 64 + 16 + 2048) + 16 * 256 * 256 + 3 * n * 5504), n * VOCAB


def work(case):
    kind = case["kind"]
    if kind == "linear":
        M, K, B = sum(int(r) for r in case["rows"].split(",")), case["K"], case["B"]
        return dict(bytes=1.5 * M * K + 2 * B * K + 4 * B * M, flops=2.0 * M * K * B)
    if kind == "decode":
        layers, head, kv = _llama_weights(case["width"])
        B, heads = case["batch"], LLAMA[case["width"]]["n_embd"]
        keys = 0.75 * case["context"] * B * LAYERS                     # cache rows read per step
        step = dict(bytes=1.5 * (layers + head) + keys * 2 * (kv + kv // 32) + 4 * B * VOCAB, flops=2.0 * B * (layers + head) + 4.0 * keys * heads)
        return {k: case["steps"] * v for k, v in step.items()}
    if kind == "prompt":
        layers, head, kv = _llama_weights(case["width"])
        T, heads = case["tokens"], LLAMA[case["width"]]["n_embd"]
        passes = -(-T // PROMPT_ROWS)
        return dict(bytes=1.5 * (layers * passes + head) + 2.0 * kv * T * LAYERS * (passes + 1) / 2, flops=2.0 * (layers * T + head) + 2.0 * T * T * heads * LAYERS)
    if kind == "turn":
        layers, head = _family_weights(case["family"])
        passes = -(-case["tokens"] // PROMPT_ROWS)
        return dict(bytes=1.5 * (layers * (passes + case["steps"]) + head * (1 + case["steps"])), flops=2.0 * layers * (case["tokens"] + case["steps"]))
    if kind == "moe":
        E, n, ff, T = MOE["experts"], MOE["width"], MOE["ff"], case["tokens"]
        named = E * (1 - (1 - MOE["top_k"] / E) ** T)
        return dict(bytes=1.5 * named * 3 * n * ff + 6.0 * T * n, flops=2.0 * T * MOE["top_k"] * 3 * n * ff)
    n = case["M"] * case["K"]
    return dict(bytes=2.0 * n + 1.5 * n + 1.5 * n + 2.0 * n, flops=0)


# Four times what the path differs by when its sums are taken in another order or against the plain evaluation (measured):
# fp32 sums of exact products; bf16 activations between the kernels of a layer and of a model.
def tolerance(case):
    return {"linear": {"rel": 1e-5}, "decode": {"rel": 2e-2}, "prompt": {"rel": 2e-2}, "turn": {"rel": 3e-2}, "moe": {"rel": 6e-3},
            "codec": "exact"}[case["kind"]]


# ---- the same in 64 bits -----------------------------------------------------------------------------------------------
def _unpack(path, name):
    """A tensor of a saved model directory, in float64."""
    M, K, P, base = (int(x) for x in open(os.path.join(path, name + ".dims")).read().split())
    load = lambda ext, t: torch.from_numpy(np.fromfile(os.path.join(path, name + ext), t)).to(DEV)
    sm, gr = load(".sm.bin", np.uint8).int(), load(".gr.bin", np.uint8).int()
    group = torch.stack([gr & 15, gr >> 4], 1).view(-1)[:M * K]
    bits = ((sm & 128) << 8) | ((base + group) << 7) | (sm & 127)
    if P:
        off = load(".row_off.bin", np.int32).long()
        row = torch.repeat_interleave(torch.arange(M, device=DEV), off[1:] - off[:-1])
        bits[row * K + load(".patch_cols.bin", np.int32).long()] = load(".patch_correct.bin", np.int16).int() & 0xFFFF
    return (bits << 16).view(torch.float32).view(M, K).double()


def _rms(x, eps=EPS):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _rotate_half(x, at, base):
    """x [T, heads, d] at positions at [T]."""
    half = x.shape[-1] // 2
    a = at[:, None, None].double() * float(base) ** (-2.0 * torch.arange(half, device=DEV).double() / x.shape[-1])
    u, v = x[..., :half], x[..., half:]
    return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()], -1)


def _int8(x):
    """What a cache row holds: 127 steps either side of zero, per head."""
    s = x.abs().amax(-1, keepdim=True) / 127
    return torch.clamp(torch.round(x / torch.where(s > 0, s, 1.0)), -127, 127) * s


def _causal(q, k, v, scale):
    """q [T, H, d], k [T, G, d], v [T, G, e] of one sequence -> [T, H, e]."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    hide = torch.ones((T, T), dtype=torch.bool, device=DEV).triu(1)
    out = []
    for g in range(G):
        s = torch.matmul(q[:, g * (H // G):(g + 1) * (H // G)].transpose(0, 1), k[:, g].T.contiguous()) * scale
        p = torch.softmax(s.masked_fill(hide, float("-inf")), -1)
        out.append(torch.matmul(p, v[:, g].contiguous()).transpose(0, 1))
    return torch.cat(out, 1)


def _llama_exact(case, seed, sequences):
    """Logits after the last token of every sequence, [sequences, vocab]."""
    c = LLAMA[case["width"]]
    n, H, G = c["n_embd"], c["n_head"], c["n_head_kv"]
    hd = n // H
    with _Folder() as path:
        e = _Served(_llama(case, seed))
        e.engine.save(path)
        del e
        lens = [len(s) for s in sequences]
        at = torch.cat([torch.arange(k, device=DEV) for k in lens])
        table = torch.from_numpy(np.fromfile(os.path.join(path, "tok_embd.bin"), np.int16)).to(DEV).view(torch.bfloat16).view(VOCAB, n)
        x = table[torch.tensor([t for s in sequences for t in s], device=DEV)].double()
        norm = lambda name: torch.from_numpy(np.fromfile(os.path.join(path, name), np.float32)).to(DEV).double()
        for i in range(LAYERS):
            p = "layer.%d." % i
            h = _rms(x) * norm(p + "attn_norm.bin")
            lin = lambda name, y: y @ _unpack(path, p + name).T
            q = _rotate_half(lin("wq", h).view(-1, H, hd), at, THETA)
            k = _int8(_rotate_half(lin("wk", h).view(-1, G, hd), at, THETA))
            v = _int8(lin("wv", h).view(-1, G, hd))
            o = torch.cat([_causal(a, b, d, hd ** -0.5) for a, b, d in zip(q.split(lens), k.split(lens), v.split(lens))])
            x = x + lin("wo", o.reshape(-1, n))
            h = _rms(x) * norm(p + "ffn_norm.bin")
            x = x + lin("w_down", torch.nn.functional.silu(lin("w_gate", h)) * lin("w_up", h))
        last = torch.cumsum(torch.tensor(lens, device=DEV), 0) - 1
        return (_rms(x[last]) * norm("output_norm.bin")) @ _unpack(path, "output_proj").T


def _gamilorn_exact(cfg, t, tokens):
    W = lambda name: t[name].double()
    T = len(tokens)
    at = torch.arange(T, device=DEV)
    x = W("embed")[torch.tensor(tokens, device=DEV)] + W("pos")[:T]
    norm = lambda y, name: _rms(y) * (1 + W(name))
    for i, L in enumerate(cfg["layers"]):
        p, a, b = "l%d." % i, L["mixer"]["left"], L["mixer"]["right"]
        H, G, d, e = a["heads"], a["kv_heads"], a["dim"], a["vdim"]
        h = norm(x, p + "norm1")
        q, k, v = (h @ W(p + "mix.left." + j).T + W(p + "mix.left.%s.b" % j) for j in "qkv")
        dist = at[:, None] - at[None, :]
        see = (dist >= 0) & ((dist < a["mask"]["size"]) | (at[None, :] < a["mask"]["keep_first"]))
        o = []
        for j in range(H):
            g = j // (H // G)
            s = torch.sigmoid(q[:, j * d:(j + 1) * d] @ k[:, g * d:(g + 1) * d].T * a["scale"] + W(p + "mix.left.pb")[j]) * see
            o.append(s @ v[:, g * e:(g + 1) * e])
        left = torch.cat(o, 1) @ W(p + "mix.left.o").T
        N, D = b["heads"], b["dim"]
        r, k, v = ((h @ W(p + "mix.right." + j).T).view(T, N, D) for j in "rkv")
        w = torch.exp(-math.exp(-0.5) * torch.sigmoid(torch.tanh(h @ W(p + "mix.right.w1").T) @ W(p + "mix.right.w2").T + W(p + "mix.right.w0"))).view(T, N, D)
        rem = torch.sigmoid(h @ W(p + "mix.right.a").T + W(p + "mix.right.a.b")).view(T, N, D)
        u = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
        S, o = torch.zeros((N, D, D), dtype=torch.float64, device=DEV), []
        for s in range(T):                                             # S [head, key channel, value channel]
            S = w[s, :, :, None] * S - (rem[s] * u[s])[:, :, None] * (u[s][:, :, None] * S).sum(1, keepdim=True) + k[s, :, :, None] * v[s, :, None, :]
            o.append((r[s][:, :, None] * S).sum(1))
        o = _rms(torch.stack(o)).reshape(T, N * D) * W(p + "mix.right.norm") * torch.sigmoid(h @ W(p + "mix.right.g").T)
        x = x + L["mixer"]["left_scale"] * left + L["mixer"]["right_scale"] * (o @ W(p + "mix.right.o").T)
        z = norm(x, p + "norm2") @ W(p + "mlp.up").T
        f = torch.nn.functional.softplus(W(p + "mlp.act"))
        low = torch.clamp(z, max=0.0)
        z = torch.where(z > 0, f[0] * z * z + 0.5 * z, (0.5 + f[1]) * (torch.expm1(low) - low) + 0.5 * z)
        x = x + z @ W(p + "mlp.down").T
    cap = cfg["logit_softcap"]
    return cap * torch.tanh(norm(x[-1:], "final.norm") @ W("head").T / cap)


def _davasun_exact(cfg, t, tokens):
    W = lambda name: t[name].double()
    T = len(tokens)
    at = torch.arange(T, device=DEV)
    norm = lambda y, name: _rms(y) * W(name)
    x = norm(W("embed")[torch.tensor(tokens, device=DEV)], "embed.norm")
    for i, L in enumerate(cfg["layers"]):
        p, c = "l%d." % i, L["mixer"]
        H, d, e = c["heads"], c["dim"], c["vdim"]
        h = norm(x, p + "norm1")
        lin = lambda name: h @ W(p + "mix." + name).T
        if L["type"] == "mlstm":
            q, k, v = lin("q").view(T, H, d) / math.sqrt(d), lin("k").view(T, H, d), lin("v").view(T, H, e)
            cap = lambda y: c["gate_cap"] * torch.tanh(y / c["gate_cap"])
            ig, fg = cap(lin("i") + W(p + "mix.i.b")), torch.nn.functional.logsigmoid(cap(lin("f") + W(p + "mix.f.b")))
            S, nrm, m, o = torch.zeros((H, d, e), dtype=torch.float64, device=DEV), torch.zeros((H, d), dtype=torch.float64, device=DEV), torch.zeros(
                H, dtype=torch.float64, device=DEV), []
            for s in range(T):
                new = torch.maximum(fg[s] + m, ig[s])
                keep, enter = torch.exp(fg[s] + m - new), torch.exp(ig[s] - new)
                S = keep[:, None, None] * S + enter[:, None, None] * k[s][:, :, None] * v[s][:, None, :]
                nrm, m = keep[:, None] * nrm + enter[:, None] * k[s], new
                o.append((q[s][:, :, None] * S).sum(1) / (torch.maximum((nrm * q[s]).sum(-1).abs(), torch.exp(-m)) + 1e-6)[:, None])
            y = _rms(torch.stack(o)).reshape(T, -1) * W(p + "mix.norm") * torch.sigmoid(lin("g"))
        else:
            R, base = c["kv_rank"], c["rot"]["base"]
            q, low = lin("q").view(T, H, -1), lin("dkv")
            q = torch.cat([q[..., :d], _rotate_half(q[..., d:], at, base)], -1)
            lat, rot = norm(low[:, :R], p + "mix.dkv.norm"), _rotate_half(low[:, None, R:], at, base)
            k = torch.cat([(lat @ W(p + "mix.uk").T).view(T, H, d), rot.expand(T, H, -1)], -1)
            y = _causal(q, k, (lat @ W(p + "mix.uv").T).view(T, H, e), c["scale"]) * torch.sigmoid(lin("g"))[:, :, None]
            y = y.reshape(T, -1)
        x = x + norm(y @ W(p + "mix.o").T, p + "norm1b")
        if L["mlp"]:
            h, lim = norm(x, p + "norm2"), L["mlp"]["limit"]
            g, u = torch.clamp(h @ W(p + "mlp.gate").T, max=lim), torch.clamp(h @ W(p + "mlp.up").T, -lim, lim)
            x = x + norm((g * torch.sigmoid(1.702 * g) * (u + 1)) @ W(p + "mlp.down").T, p + "norm2b")
    return norm(x[-1:], "final.norm") @ W("head").T * cfg["logit_scale"]


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        W, X = _linear_inputs(case, seed)
        out = [X.double() @ w.double().T for w in W]
        return [o[0] for o in out] if case["B"] == 1 else out
    if kind == "decode":
        prompts, steps = _decode_inputs(case, seed)
        return _llama_exact(case, seed, [p + [s[b] for s in steps] for b, p in enumerate(prompts)])
    if kind == "prompt":
        return _llama_exact(case, seed, [_tokens(seed, case["tokens"])])
    if kind == "turn":
        cfg, t = _family_checkpoint(case["family"], seed)
        tokens = _tokens(seed, case["tokens"]) + _tokens(seed + 77, case["steps"])
        return (_gamilorn_exact if case["family"] == "gamilorn" else _davasun_exact)(cfg, t, tokens)
    if kind == "moe":
        W, X, ids, w = _moe_inputs(case, seed)
        x, out = X.double(), torch.zeros((case["tokens"], MOE["width"]), dtype=torch.float64, device=DEV)
        for e, (w1, w3, w2) in enumerate(W):
            share = (w.double() * (ids == e)).sum(-1, keepdim=True)
            out += share * ((torch.nn.functional.silu(x @ w1.double().T) * (x @ w3.double().T)) @ w2.double().T)
        return out
    return None                                                        # the codec's outputs are whole numbers
