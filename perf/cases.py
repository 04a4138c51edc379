"""The work this framework is used for, as cases that can be timed and compared: what is run, over which sizes, and what it must give.

Llama2 stages in fp16 (and the small whole model in fp32) and the run-time sized designs in bf16, each in both directions the path has:
decode, one token of every context, and prefill, many tokens of some contexts.  A case is a dict of plain values:

  path     "decode" | "prefill" of a Llama2 stage, "design-decode" | "design-prefill" of a design
  model    a stage configuration's name, or the design's
  dtype    storage type
  layers   hosted layers (designs: layers of the model)
  batch    contexts
  lo, hi   keys a context holds when a decode step is over, spread evenly between the two
  tokens   prompt tokens per context of a prefill
"""
from __future__ import annotations

import json
import math
import os
import random
import shutil
import struct
import tempfile

import numpy as np
import torch

from glinthawk_amd import ops, stage

SHAPES = {   # dim, heads, kv heads, hidden, positions, layers
    "stories15m": (288, 6, 6, 768, 256, 6),
    "llama2-7b": (4096, 32, 32, 11008, 2048, 32),
    "llama2-13b-4k": (5120, 40, 40, 13824, 4096, 40),
    "llama2-70b-4k": (8192, 64, 8, 28672, 4096, 80),
}
VOCAB = 32000
EPS = 1e-5
# the designs at the layer sizes of the benchmark's w4096 models, with a small vocabulary
WIDTH, HIDDEN, HEADS, DIM, DESIGN_VOCAB = 4096, 11008, 32, 128, 4096
WINDOW, KEEP, BIAS_ROWS, BIAS_MAX, GATE_CAP = 1024, 4, 32, 512, 15.0
M_HEADS, M_DIM, M_VDIM = 8, 256, 512
PASSES = 2
TEMP_COEF, TEMP_EVERY = 0.1, 512
ROOM = 6000          # positions a design's contexts have beyond the first decoded one


# ---- the cases -----------------------------------------------------------------------------------
def listed():
    def llama(name, path, model, layers, batch, **sizes):
        return dict(name=name, path=path, model=model, dtype="f32" if model == "stories15m" else "f16", layers=layers, batch=batch, **sizes)

    def design(name, path, model, batch, **sizes):
        return dict(name=name, path=path, model=model, dtype="bf16", layers=2, batch=batch, **sizes)

    return [
        # a whole small model generating for a few users: nothing but latency
        llama("15m-decode-b4", "decode", "stories15m", 6, 4, lo=40, hi=256),
        # one interactive user of a large model's stage: a product of few rows is a stream of the weights
        llama("70b-decode-b1", "decode", "llama2-70b-4k", 4, 1, lo=1537, hi=1537),
        # a stage of a multi-head model at an ordinary batch
        llama("7b-decode-b32", "decode", "llama2-7b", 4, 32, lo=1024, hi=1024),
        # the headline serving step: a full batch at long contexts
        llama("70b-decode-b64", "decode", "llama2-70b-4k", 4, 64, lo=4096, hi=4096),
        # many slots in service at once, at whatever lengths they have reached
        llama("70b-decode-b256-ragged", "decode", "llama2-70b-4k", 2, 256, lo=17, hi=4096),
        # a short question to an idle stage: time to the first token
        llama("7b-prompt-77", "prefill", "llama2-7b", 4, 1, tokens=77),
        # slots that finished are refilled with new prompts between decode steps
        llama("70b-refill-26x128", "prefill", "llama2-70b-4k", 4, 26, tokens=128),
        # long documents come in
        llama("13b-prefill-8x2048", "prefill", "llama2-13b-4k", 4, 8, tokens=2048),
        # the designs, serving and taking prompts
        design("famidra-decode-b32", "design-decode", "famidra", 32, lo=1025, hi=1025),
        design("famidra-prefill-8x1024", "design-prefill", "famidra", 8, tokens=1024),
        design("dirozen-decode-b32", "design-decode", "dirozen", 32, lo=1025, hi=1025),
        design("dirozen-prefill-4x2048", "design-prefill", "dirozen", 4, tokens=2048),
    ]


def draw(rng: random.Random):
    def log(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))

    kind = rng.choice(["15m", "7b", "70b-few", "70b", "70b-many", "prompt", "refill", "13b", "famidra", "famidra-prefill", "dirozen", "dirozen-prefill"])
    if kind == "15m":
        hi = rng.randint(20, 256)
        return dict(path="decode", model="stories15m", dtype="f32", layers=6, batch=log(1, 16), lo=rng.randint(2, hi), hi=hi)
    if kind == "7b":
        hi = log(96, 2048)
        return dict(path="decode", model="llama2-7b", dtype="f16", layers=rng.choice([2, 4]), batch=log(4, 64), lo=rng.choice([hi, rng.randint(2, hi)]), hi=hi)
    if kind in ("70b-few", "70b", "70b-many"):
        few, some = kind == "70b-few", kind == "70b"
        hi = log(128, 4096)
        lo = rng.choice([hi, rng.randint(2, hi)]) if kind != "70b-many" else rng.randint(2, hi)
        return dict(path="decode", model="llama2-70b-4k", dtype="f16", layers=2, batch=log(1, 9) if few else log(10, 96) if some else rng.randint(97, 256), lo=lo, hi=hi)
    if kind == "prompt":
        return dict(path="prefill", model="llama2-7b", dtype="f16", layers=rng.choice([2, 4]), batch=rng.randint(1, 3), tokens=log(5, 120))
    if kind == "refill":
        return dict(path="prefill", model="llama2-70b-4k", dtype="f16", layers=2, batch=rng.randint(4, 32), tokens=rng.randint(33, 160))
    if kind == "13b":
        tokens = log(200, 2048)
        return dict(path="prefill", model="llama2-13b-4k", dtype="f16", layers=rng.choice([2, 4]), batch=rng.randint(1, max(1, min(8, 16384 // tokens))), tokens=tokens)
    if kind in ("famidra", "dirozen"):
        keys = log(64, 2048)
        return dict(path="design-decode", model=kind, dtype="bf16", layers=2, batch=log(1, 48), lo=keys, hi=keys)
    tokens = log(100, 2048)
    return dict(path="design-prefill", model=kind.split("-")[0], dtype="bf16", layers=2, batch=rng.randint(1, max(1, min(8, 8192 // tokens))), tokens=tokens)


# ---- what a case's values are, from its seed -------------------------------------------------------
class _Draws:
    """Normal values on the GPU, a stream of their own for every (seed, tag)."""

    def __init__(self, seed):
        self.seed, self.g = seed, torch.Generator(device="cuda")

    def fill(self, view, tag, std=1.0, mean=0.0):
        self.g.manual_seed((self.seed * 1_000_003 + hash_tag(tag)) & 0x7FFFFFFFFFFF)
        return view.normal_(mean, std, generator=self.g)

    def new(self, shape, dtype, tag, std=1.0, mean=0.0):
        return self.fill(torch.empty(shape, dtype=dtype, device="cuda"), tag, std, mean)


def hash_tag(tag):
    h = 2166136261
    for c in str(tag).encode():
        h = ((h ^ c) * 16777619) & 0xFFFFFFFF
    return h


def lengths(case, seed):
    """Keys per context, the current token among them: an even spread in an order of the seed's."""
    n = case["batch"]
    spread = [case["lo"] + (case["hi"] - case["lo"]) * (2 * i + 1) // (2 * n) for i in range(n)] if case["hi"] > case["lo"] else [case["hi"]] * n
    random.Random(seed).shuffle(spread)
    return spread


def elem(case):
    return {"f16": torch.float16, "f32": torch.float32, "bf16": torch.bfloat16}[case["dtype"]]


class _Memory:
    """Device memory of a stage's as torch sees it; the stage lives as long as a tensor over it does."""

    def __init__(self, owner, ptr, shape, dtype):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr={torch.float16: "<f2", torch.float32: "<f4"}[dtype], data=(ptr, False), strides=None, version=3)


def view(owner, ptr, shape, dtype):
    return torch.as_tensor(_Memory(owner, ptr, shape, dtype), device="cuda")


class _Host:
    """A host buffer of a stage's state, likewise."""

    def __init__(self, owner, array):
        self.owner, self.__array_interface__ = owner, array.__array_interface__


# ---- Llama2 stages -------------------------------------------------------------------------------------
def first_layer(case):
    """A stage in the middle of the pipeline; a whole model starts at its embedding."""
    return 0 if case["layers"] == SHAPES[case["model"]][5] else 8


def layer_shapes(model):
    d, heads, kv_heads, hidden, _, _ = SHAPES[model]
    kv = d // heads * kv_heads
    return {"rms_att_weight": (d,), "wq": (d, d), "wkv": (2 * kv, d), "wo": (d, d), "rms_ffn_weight": (d,), "w1": (hidden, d), "w2": (d, hidden), "w3": (hidden, d)}


def base_shapes(case):
    """The base tensors a whole model has beside its layers (its classifier is the embedding)."""
    d = SHAPES[case["model"]][0]
    return {"token_embedding_table": (VOCAB, d), "rms_final_weight": (d,)} if first_layer(case) == 0 else {}


def tensor_values(draws, name, layer, out):
    norm, embedding = name.startswith("rms"), name == "token_embedding_table"
    return draws.fill(out, f"{name}{layer}", 0.1 if norm else 1.0 if embedding else 0.02, 1.0 if norm else 0.0)


def cached_rows(draws, layer, context, out):
    return draws.fill(out, f"kv{layer}.{context}")


def prepare_llama(case, seed):
    ops.init(0)
    d, heads, kv_heads, _, positions, _ = SHAPES[case["model"]]
    kv, dt, batch, first, n = d // heads * kv_heads, elem(case), case["batch"], first_layer(case), case["layers"]
    whole = first == 0
    st = stage.Stage(case["model"], case["dtype"], first, n, batch, batch, with_cls=whole)
    draws, lib = _Draws(seed), stage.host_lib()
    count = stage.C.c_uint64(0)
    for name, shape in base_shapes(case).items():
        tensor_values(draws, name, "", view(st, lib.glint_stage_base_tensor_ptr(st._h, stage.BASE_TENSORS.index(name), stage.C.byref(count)), shape, dt))
    for l in range(first, first + n):
        for name, shape in layer_shapes(case["model"]).items():
            tensor_values(draws, name, l, view(st, lib.glint_stage_layer_tensor_ptr(st._h, l, stage.LAYER_TENSORS.index(name), stage.C.byref(count)), shape, dt))
    ids = np.arange(100, 100 + batch, dtype=np.uint32)
    decode = case["path"] == "decode"
    pos = np.array([k - 1 for k in lengths(case, seed)] if decode else [0] * batch, dtype=np.uint32)
    tokens = np.random.default_rng(seed).integers(3, VOCAB, batch).astype(np.uint32)
    st.new_state(batch, next_layer=first)
    st.set_prompts(ids, tokens, pos)
    assert st.acquire_contexts()
    s = dict(case=case, stage=st, ids=ids, pos=pos, tokens=tokens, first=first, rows=[], logits=None)
    # what a pass appends to the caches: all of it, or that of evenly chosen contexts where there are many
    seen = range(0, batch, -(-batch * n // 60))
    new = 1 if decode else case["tokens"]
    for l in range(first, first + n):
        for i in range(batch):
            rows = view(st, st.context_layer_ptr(i, l), (positions, 2 * kv), dt)
            if decode and pos[i] > 0:
                cached_rows(draws, l, i, rows[: int(pos[i])])
            if i in seen:
                s["rows"].append(rows[int(pos[i]): int(pos[i]) + new])
    if not whole:
        x = draws.new((batch * new, d), dt, "x").cpu().numpy()
        s["x"], s["y"] = ops.pinned_empty(x.shape, x.dtype), None if decode else ops.pinned_empty(x.shape, x.dtype)
        s["x"][:] = x
    else:
        s["logits"] = view(st, st.scratch_ptr("logits"), (batch, VOCAB), dt)
    torch.cuda.synchronize()
    return s


def run_llama(s):
    st, case = s["stage"], s["case"]
    if case["path"] == "prefill":
        out, _ = st.prefill(s["ids"], s["pos"], case["tokens"], s["first"], activations=s["x"], out=s["y"])
        return {"activations": out, "rows": s["rows"]}
    st.new_state(case["batch"], next_layer=s["first"])
    st.set_prompts(s["ids"], s["tokens"], s["pos"])
    if s["first"] > 0:
        st.activations(allocate=True)[:] = s["x"].reshape(-1)
    st.forward()
    return {"activations": s["logits"] if s["first"] == 0 else np.asarray(_Host(st, st.activations())), "rows": s["rows"]}


def rms_norm(x, w, eps=EPS):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def causal(q, k, v, scale, first, bias=None, window=None, keep=0):
    """q (T, H, d) of positions first ..., k and v (first + T, G, d): the attention of one context, (T, H, dv)."""
    T, H, _ = q.shape
    n, G = k.shape[0], k.shape[1]
    out = torch.empty((T, H, v.shape[2]), dtype=q.dtype, device=q.device)
    i, j = torch.arange(first, first + T, device=q.device)[:, None], torch.arange(n, device=q.device)[None, :]
    hidden = j > i
    if window is not None:
        hidden |= (i - j >= window) & (j >= keep)
    far = (i - j).clamp(min=0) if bias is not None else None
    for g in range(G):
        hs = slice(g * (H // G), (g + 1) * (H // G))
        score = torch.einsum("thd,nd->htn", q[:, hs], k[:, g].contiguous()) * scale
        if bias is not None:
            score += bias[:, hs].T[:, far]
        out[:, hs] = torch.einsum("htn,nd->thd", score.masked_fill(hidden, -math.inf).softmax(-1), v[:, g].contiguous())
    return out


def rotate(x, re, im):
    """x (T, heads, d), tables (T, d / 2): neighbouring pairs."""
    a, b = x[..., 0::2], x[..., 1::2]
    re, im = re[:, None], im[:, None]
    return torch.stack([a * re - b * im, a * im + b * re], -1).flatten(-2)


def exact_llama(case, seed):
    d, heads, kv_heads, _, positions, _ = SHAPES[case["model"]]
    hd, dt, batch, first, n = d // heads, elem(case), case["batch"], first_layer(case), case["layers"]
    kv, decode = hd * kv_heads, case["path"] == "decode"
    draws, new = _Draws(seed), 1 if case["path"] == "decode" else case["tokens"]
    pos = [k - 1 for k in lengths(case, seed)] if decode else [0] * batch
    freq = np.float32(1.0) / np.power(np.float32(10000.0), np.arange(0, hd, 2, dtype=np.float32) / np.float32(hd))
    angle = torch.from_numpy(np.arange(positions, dtype=np.float32)[:, None] * freq).double().cuda()
    re, im = torch.cos(angle).to(dt).double(), torch.sin(angle).to(dt).double()
    if first == 0:
        tokens = np.random.default_rng(seed).integers(3, VOCAB, batch)
        base = {name: tensor_values(draws, name, "", torch.empty(shape, dtype=dt, device="cuda")).double() for name, shape in base_shapes(case).items()}
        x = base["token_embedding_table"][torch.from_numpy(tokens).cuda()]
    else:
        x = draws.new((batch * new, d), dt, "x").double()
    seen, kept = range(0, batch, -(-batch * n // 60)), []
    for l in range(first, first + n):
        w = {}
        for name, shape in layer_shapes(case["model"]).items():
            w[name] = tensor_values(draws, name, l, torch.empty(shape, dtype=dt, device="cuda"))
        h = rms_norm(x, w["rms_att_weight"].double())
        q, appended = (h @ w["wq"].double().T).view(batch, new, heads, hd), (h @ w["wkv"].double().T).view(batch, new, 2, kv_heads, hd)
        mixed = torch.empty((batch, new, d), dtype=torch.float64, device="cuda")
        for i in range(batch):
            at = slice(pos[i], pos[i] + new)
            row = torch.stack([rotate(appended[i, :, 0], re[at], im[at]), appended[i, :, 1]], 1)
            old = cached_rows(draws, l, i, torch.empty((pos[i], 2 * kv), dtype=dt, device="cuda")) if pos[i] else torch.empty((0, 2 * kv), dtype=dt, device="cuda")
            both = torch.cat([old.double().view(-1, 2, kv_heads, hd), row])
            mixed[i] = causal(rotate(q[i], re[at], im[at]), both[:, 0], both[:, 1], hd ** -0.5, pos[i]).reshape(new, d)
            if i in seen:
                kept.append(row.reshape(new, 2 * kv))
        x = x + mixed.view(batch * new, d) @ w["wo"].double().T
        h = rms_norm(x, w["rms_ffn_weight"].double())
        x = x + (torch.nn.functional.silu(h @ w["w1"].double().T) * (h @ w["w3"].double().T)) @ w["w2"].double().T
    if first == 0:
        x = rms_norm(x, base["rms_final_weight"]) @ base["token_embedding_table"].T
    return {"activations": x if first == 0 or not decode else x.reshape(-1), "rows": kept}


# ---- the designs ----------------------------------------------------------------------------------------
def design_config(case):
    """config.json and the tensors of model.safetensors: name -> (shape, std, mean)."""
    positions = (case["lo"] if case["path"] == "design-decode" else case["tokens"]) + ROOM
    mlp = {"kind": "dense", "ff": HIDDEN}
    t = {"embed": ((DESIGN_VOCAB, WIDTH), 1.0, 0.0)}

    def lin(name, rows, cols, gain=1.0):
        t[name] = ((rows, cols), gain / math.sqrt(cols), 0.0)

    if case["model"] == "famidra":
        layers = [{"type": "mlstm", "mixer": dict(heads=M_HEADS, dim=M_DIM, vdim=M_VDIM, gate_cap=GATE_CAP), "mlp": None},
                  {"type": "attention", "mlp": mlp, "mixer": dict(heads=HEADS, kv_heads=HEADS, dim=DIM, vdim=DIM, scale=DIM ** -0.5, bias_max=BIAS_MAX,
                                                                  mask=dict(size=WINDOW, keep_first=KEEP))}]
        config = {"architecture": "Famidra", "width": WIDTH, "vocab": DESIGN_VOCAB, "max_positions": positions, "norm": {"eps": EPS}, "logit_scale": 0.5,
                  "layers": layers, "loop": {"start": 0, "stop": 2, "times": PASSES}}
        t["pos"], t["final.norm"] = ((positions, WIDTH), 0.4, 0.0), ((WIDTH,), 0.2, 1.0)
        lin("loop.in", WIDTH, 2 * WIDTH, 1.4)
        t["loop.step"] = ((PASSES, WIDTH), 0.5, 0.0)
        for l in (0, 1):
            t[f"l{l}.norm1"] = t[f"l{l}.norm1b"] = ((WIDTH,), 0.2, 1.0)
        hk, hv = M_HEADS * M_DIM, M_HEADS * M_VDIM
        for name, rows, gain in (("q", hk, 1.0), ("k", hk, 1.0), ("v", hv, 1.0), ("g", hv, 1.0), ("i", M_HEADS, 2.0), ("f", M_HEADS, 2.0)):
            lin("l0.mix." + name, rows, WIDTH, gain)
        t["l0.mix.i.b"], t["l0.mix.f.b"], t["l0.mix.norm"] = ((M_HEADS,), 1.0, 0.0), ((M_HEADS,), 2.0, 3.0), ((hv,), 0.2, 1.0)
        lin("l0.mix.o", WIDTH, hv)
        for name in ("q", "k", "v"):
            lin("l1.mix." + name, HEADS * DIM, WIDTH)
            t[f"l1.mix.{name}.b"] = ((HEADS * DIM,), 0.3, 0.0)
        t["l1.mix.q.norm"] = t["l1.mix.k.norm"] = ((HEADS * DIM,), 0.2, 1.2)
        t["l1.mix.rel"] = ((BIAS_ROWS, HEADS), 1.0, 0.0)
        lin("l1.mix.o", WIDTH, HEADS * DIM)
        t["l1.norm2"] = t["l1.norm2b"] = ((WIDTH,), 0.2, 1.0)
        for name, rows, cols in (("gate", HIDDEN, WIDTH), ("up", HIDDEN, WIDTH), ("down", WIDTH, HIDDEN)):
            lin("l1.mlp." + name, rows, cols)
            t[f"l1.mlp.{name}.b"] = ((rows,), 0.2, 0.0)
    else:
        layer = {"type": "attention", "mlp": mlp, "mixer": dict(heads=HEADS, kv_heads=HEADS, dim=DIM, vdim=DIM, scale=DIM ** -0.5,
                                                                q_temp=dict(coef=TEMP_COEF, every=TEMP_EVERY))}
        config = {"architecture": "Dirozen", "width": WIDTH, "vocab": DESIGN_VOCAB, "norm": {"eps": EPS}, "layers": [layer] * case["layers"]}
        lin("head", DESIGN_VOCAB, WIDTH)
        t["final.norm"] = ((WIDTH,), 0.2, 0.0)
        for l in range(case["layers"]):
            t[f"l{l}.norm1"] = ((WIDTH,), 0.2, 0.0)
            for name, rows, gain in (("q", HEADS * DIM, 1.0), ("k", HEADS * DIM, 1.0), ("g", HEADS, 2.0), ("o", WIDTH, 1.5)):
                lin(f"l{l}.mix.{name}", rows, HEADS * DIM if name == "o" else WIDTH, gain)
            for name, rows, cols in (("gate", HIDDEN, WIDTH), ("up", HIDDEN, WIDTH), ("down", WIDTH, HIDDEN)):
                lin(f"l{l}.mlp.{name}", rows, cols)
    return config, t, positions


def design_weights(tensors, seed):
    draws = _Draws(seed)
    for name, (shape, std, mean) in tensors.items():
        yield name, draws.new(shape, torch.bfloat16, name, std, mean)


def design_tokens(case, seed):
    """(batch, tokens): the prompts, for decode with the tokens fed after them."""
    n = case["tokens"] if case["path"] == "design-prefill" else case["lo"] + ROOM
    return np.random.default_rng(seed).integers(0, DESIGN_VOCAB, (case["batch"], n)).astype(np.uint32)


def prepare_design(case, seed):
    ops.init(0)
    config, tensors, positions = design_config(case)
    batch, tokens = case["batch"], design_tokens(case, seed)
    folder = tempfile.mkdtemp(dir="/dev/shm" if os.access("/dev/shm", os.W_OK) else None)
    try:
        with open(os.path.join(folder, "config.json"), "w") as f:
            json.dump(config, f)
        header, at = {}, 0
        for name, (shape, _, _) in tensors.items():
            size = 2 * math.prod(shape)
            header[name] = {"dtype": "BF16", "shape": list(shape), "data_offsets": [at, at + size]}
            at += size
        raw = json.dumps(header).encode()
        with open(os.path.join(folder, "model.safetensors"), "wb") as f:
            f.write(struct.pack("<Q", len(raw)) + raw)
            for _, w in design_weights(tensors, seed):
                w.view(torch.int16).cpu().numpy().tofile(f)
        st = stage.DesignStage(folder, case["dtype"], batch, batch, max_positions=positions)
    finally:
        shutil.rmtree(folder, ignore_errors=True)
    s = dict(case=case, stage=st, ids=np.arange(batch, dtype=np.uint32), tokens=tokens, positions=positions)
    if case["path"] == "design-decode":
        take_prompts(s)
    torch.cuda.synchronize()
    return s


def take_prompts(s):
    """Every context at its length of the first decoded token, a few contexts at a time."""
    prompt = s["case"]["lo"] - 1
    per = max(1, 8192 // prompt)
    for i in range(0, s["case"]["batch"], per):
        part = s["ids"][i: i + per]
        s["stage"].prefill_logits(part, [0] * len(part), s["tokens"][i: i + per, :prompt])
    s["at"] = prompt


def run_design(s):
    st, case = s["stage"], s["case"]
    if case["path"] == "design-prefill":
        batch, n = s["tokens"].shape
        logits, _, _ = st.prefill_logits(s["ids"], [0] * batch, s["tokens"], want=[(i + 1) * n - 1 for i in range(batch)])
        return logits
    batch = case["batch"]
    if s["at"] == s["positions"]:       # contexts full: the conversations start again
        take_prompts(s)
    st.new_state(batch)
    st.set_prompts(s["ids"], s["tokens"][:, s["at"]], np.full(batch, s["at"], np.uint32), max_completion_length=s["positions"])
    st.forward()
    s["at"] += 1
    return st.logits(batch)


def unit(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def distance_bias(table, distances):
    """(distances, heads) of a table that has a row a distance up to half of its rows, then rows that widen with the logarithm."""
    half, rows = table.shape[0] // 2, []
    for n in range(distances):
        rows.append(n if n < half else min(table.shape[0] - 1, half + int(math.floor(math.log(n / half) / math.log(BIAS_MAX / half) * (table.shape[0] - half) + 1e-9))))
    return table[torch.tensor(rows, device=table.device)]


def matrix_memory(q, k, v, log_i, log_f):
    """q, k (T, H, d), v (T, H, dv), log gates (T, H) of one context: every token against all before it, the maximum taken out."""
    T, H, _ = q.shape
    total = log_f.cumsum(0)
    out = torch.empty((T, H, v.shape[2]), dtype=q.dtype, device=q.device)
    later = torch.ones((T, T), dtype=torch.bool, device=q.device).triu(1)
    for h in range(H):
        weight = (total[:, None, h] - total[None, :, h] + log_i[None, :, h]).masked_fill(later, -math.inf)
        m = torch.maximum(weight.amax(1), total[:, h])
        mixed = (q[:, h].contiguous() @ k[:, h].T.contiguous()) * torch.exp(weight - m[:, None])
        out[:, h] = (mixed @ v[:, h].contiguous()) / (torch.maximum(mixed.sum(1).abs(), torch.exp(-m)) + 1e-6)[:, None]
    return out


def exact_design(case, seed):
    _, tensors, _ = design_config(case)
    w = dict(design_weights(tensors, seed))
    tokens = torch.from_numpy(design_tokens(case, seed).astype(np.int64)).cuda()
    tokens = tokens[:, : case["lo"]] if case["path"] == "design-decode" else tokens
    batch, T = tokens.shape

    def by(x, name):
        return x @ w[name].double().T

    def each(mixer, *parts):
        return torch.cat([mixer(*[p[i * T: (i + 1) * T] for p in parts]) for i in range(batch)])

    x = w["embed"].double()[tokens.reshape(-1)]
    if case["model"] == "dirozen":
        at = torch.arange(T, device="cuda")
        heat = 1 + TEMP_COEF * torch.log(((at + 1) // TEMP_EVERY + 1).double())[:, None, None]
        for l in range(case["layers"]):
            h = unit(x) * (1 + w[f"l{l}.norm1"].double())
            q, k = by(h, f"l{l}.mix.q").view(-1, HEADS, DIM), by(h, f"l{l}.mix.k").view(-1, HEADS, DIM)
            o = each(lambda q, k: causal(unit(q) * heat, unit(k), k, DIM ** -0.5, 0), q, k) * torch.sigmoid(by(h, f"l{l}.mix.g"))[:, :, None]
            x = x + by(o.reshape(batch * T, -1), f"l{l}.mix.o") + by(torch.nn.functional.silu(by(h, f"l{l}.mlp.gate")) * by(h, f"l{l}.mlp.up"), f"l{l}.mlp.down")
        last = x.view(batch, T, WIDTH)[:, -1]
        return by(unit(last) * (1 + w["final.norm"].double()), "head")
    x = x + w["pos"].double()[:T].repeat(batch, 1)
    start, bias = x, distance_bias(w["l1.mix.rel"].double(), T)
    for t in range(PASSES):
        x = by(torch.cat([x, start], -1), "loop.in") + w["loop.step"][t].double()
        h = rms_norm(x, w["l0.norm1"].double())
        heads = {n: by(h, "l0.mix." + n).view(batch * T, M_HEADS, -1) for n in ("q", "k", "v")}
        log_i, log_f = (GATE_CAP * torch.tanh((by(h, f"l0.mix.{n}") + w[f"l0.mix.{n}.b"].double()) / GATE_CAP) for n in ("i", "f"))
        o = each(matrix_memory, heads["q"] * M_DIM ** -0.5, heads["k"], heads["v"], log_i, torch.nn.functional.logsigmoid(log_f))
        o = unit(o).reshape(batch * T, -1) * w["l0.mix.norm"].double() * torch.sigmoid(by(h, "l0.mix.g"))
        x = x + rms_norm(by(o, "l0.mix.o"), w["l0.norm1b"].double())
        h = rms_norm(x, w["l1.norm1"].double())
        q, k, v = (by(h, f"l1.mix.{n}") + w[f"l1.mix.{n}.b"].double() for n in ("q", "k", "v"))
        q, k = rms_norm(q, w["l1.mix.q.norm"].double()), rms_norm(k, w["l1.mix.k.norm"].double())
        q, k, v = (a.view(batch * T, HEADS, DIM) for a in (q, k, v))
        o = each(lambda q, k, v: causal(q, k, v, DIM ** -0.5, 0, bias, WINDOW, KEEP), q, k, v)
        x = x + rms_norm(by(o.reshape(batch * T, -1), "l1.mix.o"), w["l1.norm1b"].double())
        h = rms_norm(x, w["l1.norm2"].double())
        gate, up = (by(h, f"l1.mlp.{n}") + w[f"l1.mlp.{n}.b"].double() for n in ("gate", "up"))
        y = by(torch.nn.functional.gelu(gate, approximate="tanh") * up, "l1.mlp.down") + w["l1.mlp.down.b"].double()
        x = x + rms_norm(y, w["l1.norm2b"].double())
    return 0.5 * by(rms_norm(x.view(batch, T, WIDTH)[:, -1], w["final.norm"].double()), "embed")


# ---- the interface ------------------------------------------------------------------------------------
def prepare(case, seed):
    return prepare_design(case, seed) if case["path"].startswith("design") else prepare_llama(case, seed)


def run(state):
    return run_design(state) if state["case"]["path"].startswith("design") else run_llama(state)


def exact(case, seed):
    return exact_design(case, seed) if case["path"].startswith("design") else exact_llama(case, seed)


def work(case):
    """Weights once, cached rows once, inputs and outputs once; products and attention over the keys that are seen."""
    batch, dec = case["batch"], case["path"].endswith("decode")
    rows = batch if dec else batch * case["tokens"]
    size = 4 if case["dtype"] == "f32" else 2
    if not case["path"].startswith("design"):
        d, heads, kv_heads, _, _, _ = SHAPES[case["model"]]
        kv = d // heads * kv_heads
        params = case["layers"] * sum(math.prod(s) for s in layer_shapes(case["model"]).values())
        head = VOCAB * d if first_layer(case) == 0 else 0
        keys = sum(lengths(case, 0)) if dec else batch * case["tokens"] * (case["tokens"] + 1) // 2
        cached = keys if dec else rows
        moved = params + head + case["layers"] * 2 * kv * cached + rows * (VOCAB + d if head else 2 * d)
        return {"bytes": size * moved, "flops": 2 * rows * (params + head) + case["layers"] * 4 * d * keys}
    n = case["lo"] if dec else case["tokens"]
    attention = HEADS * DIM
    if case["model"] == "dirozen":
        runs, seen, row = case["layers"], n if dec else n * (n + 1) // 2, attention
        used = params = runs * (3 * WIDTH * attention + WIDTH * HEADS + 3 * WIDTH * HIDDEN)
        states, mixed = 0, 4 * attention * seen * batch * runs
    else:
        runs, row = PASSES, 2 * attention
        seen = min(n, WINDOW + KEEP) if dec else sum(min(i + 1, WINDOW + KEEP) for i in range(n))
        hk, hv = M_HEADS * M_DIM, M_HEADS * M_VDIM
        params = WIDTH * (2 * hk + 3 * hv + 2 * M_HEADS) + 4 * WIDTH * attention + 3 * WIDTH * HIDDEN + 2 * WIDTH * WIDTH
        used = runs * params
        states = runs * batch * M_HEADS * M_DIM * (M_VDIM + 1) * 4 * (2 if dec else 1)
        mixed = runs * batch * (4 * attention * seen + (n if not dec else 1) * 6 * M_HEADS * M_DIM * M_VDIM)
    logits = DESIGN_VOCAB * batch
    cached = runs * row * batch * (seen if dec else n)
    return {"bytes": 2 * (params + DESIGN_VOCAB * WIDTH + cached) + states + 4 * logits, "flops": 2 * rows * used + 2 * logits * WIDTH + mixed}


def tolerance(case):
    """Largest distance of another correct implementation with the same storage types: about four times what this one is off the exact
    values, of which rounding between the ops of a layer is nearly all.  Measured: fp32 1e-6 (cache rows), fp16 2e-3, Dirozen 3.6e-3,
    Famidra 7.5e-3 (its recurrence divides by a sum that cancels)."""
    if case["dtype"] == "f32":
        return {"rel": 5e-6}
    return {"rel": 8e-3} if case["dtype"] == "f16" else {"rel": 1.5e-2} if case["model"] == "dirozen" else {"rel": 3e-2}
