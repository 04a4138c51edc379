"""The Famidra design on the GPU against the plain implementation (plain_famidra.py): every mechanism alone, then whole models through the
stage, the compute kernel and the trace runner -- whole prompts, portions, token by token, batches, slots that are used again."""
import json
import os
import subprocess

import numpy as np
import pytest

import famidra_models as M
import plain_famidra as P

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DTYPES = ("f32", "bf16")
# root mean square of the difference over that of the expected values, worst row
MODEL_TOL = {"f32": 5e-5, "bf16": 8e-2}


def torch_dtype(dtype):
    import torch
    return torch.float32 if dtype == "f32" else torch.bfloat16


def dev(a, dtype):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda().to(torch_dtype(dtype)).contiguous()


def back(t):
    return t.float().cpu().numpy().astype(np.float64)


def row_error(got, want):
    got, want = np.asarray(got, np.float64), np.asarray(want, np.float64)
    return np.sqrt(((got - want) ** 2).mean(-1)) / np.sqrt((want ** 2).mean())


def assert_rows(got, want, tol, what="", stretch=1.0):
    """`stretch`: one row in fifty may be off by that many times more (a head whose output almost cancels is blown up by its norm,
    rounding included)."""
    e = row_error(got, want)
    ok = bool(np.isfinite(got).all()) and e.max() <= tol * stretch and (e > tol).sum() <= max(1, e.size // 50)
    assert ok if stretch > 1 else bool(np.isfinite(got).all()) and e.max() <= tol, f"{what}: worst row {int(e.argmax())} of {e.size} off by {e.max():.2e} (tol {tol})"


def logit_error(got, want):
    d = np.asarray(got, np.float64) - want
    d -= d.mean(-1, keepdims=True)
    w = want - want.mean(-1, keepdims=True)
    return np.sqrt((d ** 2).mean(-1)) / np.sqrt((w ** 2).mean())


def assert_logits(got, want, dtype, what=""):
    """fp32 storage holds every position; in bf16 a few may stray further, where a norm blows up the rounding of a small vector."""
    e, tol = logit_error(got, want), MODEL_TOL[dtype]
    ok = e.max() <= tol if dtype == "f32" else e.max() <= 5 * tol and (e > tol).sum() <= max(1, e.size // 25)
    assert ok, f"{what}: row {int(e.argmax())} of {e.size} off by {e.max():.2e} (tol {tol})"


# ---- mechanisms alone ----------------------------------------------------------------------------
@pytest.mark.parametrize("b,s,r", [(1, 64, 40), (3, 52, 17), (7, 256, 512), (70, 136, 200), (200, 256, 384), (300, 512, 2048), (200, 512, 8), (333, 1024, 24), (1030, 2048, 32), (2048, 1024, 8192)])
def test_bf16_products(b, s, r):
    import torch
    from glinthawk_amd import ops
    g = torch.Generator().manual_seed(b * s + r)
    x = torch.randn((b, s), generator=g).cuda().bfloat16()
    w = (torch.randn((r, s), generator=g) / s ** 0.5).cuda().bfloat16()
    want = x.float() @ w.float().T
    got = ops.matmul(x, w).float()
    assert (got - want).abs().max() <= 2 ** -8 * want.abs().max() + 1e-6
    assert (ops.matmul_scaled(x, w, 0.5) - 0.5 * want).abs().max() <= 1e-5 * want.abs().max()


# K ranges that leave a wave of the few weight rows' kernel one piece of 64, three and five
@pytest.mark.parametrize("b,s,r", [(200, 256, 8), (225, 768, 17), (333, 1280, 32)])
def test_bf16_products_of_few_weight_rows(b, s, r):
    test_bf16_products(b, s, r)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,s,width", [(1, 24, 52), (5, 128, 128), (33, 40, 1000), (200, 64, 256), (260, 64, 50)])
def test_stream_step(dtype, rows, s, width):
    """Every part of the residual update: bias, norm behind the projection, sum or replacement, added vector, norm in front of the next product."""
    import torch
    from glinthawk_amd import ops
    rng = np.random.default_rng(rows * width)
    rnd = lambda *shape: M.to_bf16(rng.standard_normal(shape))
    inp, w, bias, post, add, nxt = rnd(rows, s), rnd(width, s), rnd(width), 1 + 0.3 * rnd(width), rnd(width), 1 + 0.3 * rnd(width)
    post, nxt = M.to_bf16(post), M.to_bf16(nxt)
    x0 = rng.standard_normal((rows, width)).astype(np.float32)
    y = inp.astype(np.float64) @ w.T
    eps = 2e-3
    for parts in (dict(bias=bias, post_norm=post, accumulate=True, next_norm=nxt), dict(accumulate=False, add=add, next_norm=nxt), dict(post_norm=post, accumulate=True),
                  dict(bias=bias, accumulate=True, next_norm=None)):
        v = y + (parts["bias"] if "bias" in parts else 0)
        if "post_norm" in parts:
            v = P.rms_norm(v, eps, post.astype(np.float64))
        want = (x0 if parts["accumulate"] else 0) + v + (parts["add"] if "add" in parts else 0)
        out = torch.zeros((rows, 2 * width), dtype=torch_dtype(dtype), device="cuda")      # a row stride of its own
        x = torch.from_numpy(x0).cuda()
        dparts = {k: (dev(a, dtype) if isinstance(a, np.ndarray) else a) for k, a in parts.items()}
        ops.matmul_stream(x, dev(inp, dtype), dev(w, dtype), eps, out=out[:, width:], **dparts)
        want_out = P.rms_norm(want, eps, nxt.astype(np.float64)) if parts.get("next_norm") is not None else want
        tol = 1e-5 if dtype == "f32" else 1e-2
        assert_rows(back(x), want, tol, f"stream {sorted(parts)}")
        assert_rows(back(out[:, width:]), want_out, tol, f"out {sorted(parts)}")
        assert float(out[:, :width].abs().max()) == 0.0
    one = torch.zeros((rows, width), dtype=torch_dtype(dtype), device="cuda")
    ops.stream_out(torch.from_numpy(x0).cuda(), one, dev(nxt, dtype), eps)
    assert_rows(back(one), P.rms_norm(x0.astype(np.float64), eps, nxt.astype(np.float64)), 1e-5 if dtype == "f32" else 5e-3, "norm alone")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,s,hidden", [(1, 32, 20), (9, 64, 30), (64, 256, 128), (210, 64, 72)])
def test_gate(dtype, rows, s, hidden):
    from glinthawk_amd import ops
    rng = np.random.default_rng(hidden)
    x, w, b = (M.to_bf16(rng.standard_normal(n)) for n in ((rows, s), (2 * hidden, s), (2 * hidden,)))
    w = M.to_bf16(w / np.sqrt(s))
    y = x.astype(np.float64) @ w.T + b
    want = P.gelu_tanh(y[:, :hidden]) * y[:, hidden:]
    assert_rows(back(ops.matmul_gate(dev(x, dtype), dev(w, dtype), dev(b, dtype))), want, 1e-5 if dtype == "f32" else 1e-2)


def test_embedding():
    import torch
    from glinthawk_amd import ops
    rng = np.random.default_rng(1)
    e, p = rng.standard_normal((31, 20)).astype(np.float32), rng.standard_normal((40, 20)).astype(np.float32)
    tok = rng.integers(0, 31, (2, 5)).astype(np.int32)
    copy = torch.zeros((10, 40), device="cuda")
    x = ops.embed_positions(torch.from_numpy(tok.reshape(-1)).cuda(), torch.tensor([0, 33], dtype=torch.int32, device="cuda"), 5, dev(e, "f32"), dev(p, "f32"), copy[:, 20:])
    want = e[tok] + np.stack([p[0:5], p[33:38]])
    assert np.array_equal(x.cpu().numpy().reshape(2, 5, 20), want) and np.array_equal(copy[:, 20:].cpu().numpy(), x.cpu().numpy())


# threads of a row with one, two, four and eight groups of columns, a row that ends inside them, widths that are not of fours; read in place, uploaded, or pageable
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width,batch,n_tokens,pinned", [(4096, 3, 1, True), (288, 5, 1, True), (4100, 2, 7, True), (16388, 1, 2, True), (32768, 2, 1, False), (30, 4, 1, True),
                                                         (64, 256, 1, True), (64, 257, 1, True), (1028, 2, 600, True)])
def test_start_of_a_step(dtype, width, batch, n_tokens, pinned):
    """As the upload, the embedding and the norm one by one: the same bits but for the norm, whose sums of squares may be contracted otherwise (some 2^-22)."""
    import torch
    from glinthawk_amd import ops
    g, rows = torch.Generator(device="cuda").manual_seed(width), batch * n_tokens
    e, p, nw = (torch.randn(s, generator=g, device="cuda").to(torch_dtype(dtype)) for s in ((50, width), (700, width), (width,)))
    size = (rows + batch) * 4 + 12
    host = ops.pinned_empty((size // 16 * 16,), np.uint8) if pinned else np.empty((size // 16 * 16,), np.uint8)
    words, rng = host.view(np.int32), np.random.default_rng(width)
    words[:] = 0
    words[:batch], words[batch: batch + rows] = rng.integers(0, 80, batch), rng.integers(0, 50, rows)
    words[batch] = 1000                      # a row without a context may hold anything
    for pos, copied, norm, base in ((p, True, nw, 0.0), (None, False, nw, 1.0), (p, True, None, 0.0)):
        copies = [torch.zeros((rows, 2 * width), device="cuda", dtype=torch_dtype(dtype)) for _ in range(2)]
        outs = [torch.zeros((rows, width), device="cuda", dtype=torch_dtype(dtype)) for _ in range(2)]
        table = torch.zeros(host.shape, dtype=torch.uint8, device="cuda")
        got = ops.embed_step(table, host, 4 * batch, 0, batch, n_tokens, e, outs[0], pos, copies[0][:, width:] if copied else None, norm, 1e-5, base)
        torch.cuda.synchronize()
        assert np.array_equal(table.cpu().numpy(), host)
        on_device = torch.from_numpy(words.copy()).cuda()
        want = ops.embed_positions(on_device[batch: batch + rows].contiguous(), on_device[:batch].contiguous(), n_tokens, e, pos, copies[1][:, width:] if copied else None)
        ops.stream_out(want, outs[1], norm, 1e-5, base)
        assert torch.equal(got, want) and torch.equal(copies[0], copies[1])
        tol = 2.0 ** -8 if dtype == "bf16" else 1e-6    # one unit in the last place of bf16
        assert torch.allclose(outs[0].float(), outs[1].float(), rtol=tol, atol=0.0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,s,r", [(32, 4096, 4096), (1, 64, 4), (3, 100, 36), (5, 256, 8196), (2, 64, 32000), (200, 128, 1000), (4, 64, 30), (3, 64, 65536),
                                      (7, 64, 65540), (8, 64, 65540)])
def test_scaled_product_with_its_argmax(dtype, rows, s, r):
    """The same bits as the product and the argmax one after the other: ties, NaN first and elsewhere, rows of -inf."""
    import torch
    from glinthawk_amd import ops
    g = torch.Generator(device="cuda").manual_seed(r)
    x, w = (torch.randn(shape, generator=g, device="cuda").to(torch_dtype(dtype)) for shape in ((rows, s), (r, s)))
    w[r // 2] = w[r - 1]
    if rows > 2:
        w[0, 0], x[0, 0], x[1, 1:], x[2] = float("inf"), 0.0, 0.0, -float("inf")   # NaN at column 0; +-inf or 0; -inf, inf and NaN
        w[r // 3, 0] = float("inf")
    logits, best = ops.matmul_scaled_argmax(x, w, 0.5)
    want = ops.matmul_scaled(x, w, 0.5)
    assert torch.equal(logits.view(torch.int32), want.view(torch.int32))
    assert best.tolist() == ops.argmax(want)


ATTENTIONS = {
    # heads, kv heads, dim, vdim, window, kept, table rows, bias_max
    "grouped": (6, 2, 24, 16, 11, 3, 10, 40),
    "matrix": (8, 2, 64, 64, 40, 5, 16, 64),
    "ten": (10, 1, 72, 40, 30, 20, 8, 33),
    "own": (3, 3, 128, 96, 70, 0, 32, 100),
    "deep": (2, 1, 200, 136, 17, 1, 6, 25),
    "deeper": (1, 1, 300, 280, 20, 2, 4, 9),
    "open": (4, 2, 32, 32, 0, 0, 12, 50),        # no window
}


# streams of keys (rows x heads) up to the CUs, cut into splits and not; up to two, four times as many and more; short and long; heads that do not divide by
# two or four; head sizes that leave lanes idle; long streams whose work-groups are cut because they would leave CUs idle, up to the CUs and beyond
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("heads,dim,vdim,rows,keys", [(4, 128, 128, 1, 1500), (2, 72, 128, 40, 2100), (3, 96, 96, 5, 40), (32, 128, 128, 1, 64), (8, 128, 104, 40, 250),
                                                      (4, 72, 72, 70, 3100), (4, 128, 128, 150, 70), (6, 80, 72, 100, 33), (4, 128, 128, 300, 150), (4, 72, 128, 300, 250),
                                                      (5, 128, 128, 240, 200), (6, 96, 96, 24, 4200), (6, 72, 72, 52, 4200), (6, 72, 80, 100, 4200), (5, 128, 128, 120, 33),
                                                      (2, 96, 96, 1, 5000), (12, 72, 72, 50, 8500)])
def test_decode_of_heads_with_keys_of_their_own(heads, dim, vdim, rows, keys, shared):
    """Against 64 bits: a rounding to bf16 and fp32 sums.  Contexts of all lengths and none, a window with kept keys, a bias by distance, keys whose scores are -inf."""
    import torch
    from glinthawk_amd import ops
    vdim = dim if shared else vdim
    window, keep, n_dist = (keys // 2 + 1, 5, 0) if heads % 4 == 0 else (0, 0, 0 if shared else 17)
    a = ops.window_attn(heads, heads, dim, vdim, dim ** -0.5, window, keep, n_dist, shared)
    g = torch.Generator(device="cuda").manual_seed(rows + keys)
    row = heads * (dim if shared else dim + vdim)
    cache = torch.randn((rows, keys, row), generator=g, device="cuda").bfloat16()
    groups = -(-keys // 32)                                           # GH_WINDOW_FACTOR_GROUP keys side by side
    factors = torch.rand((rows, groups, heads, 32), generator=g, device="cuda") + 0.5
    memory = torch.cat([cache.view(rows, -1).view(torch.uint8), factors.view(rows, -1).view(torch.uint8)], 1).contiguous()
    lengths = torch.randint(1, keys + 1, (rows,), generator=g, device="cuda")
    lengths[-1], lengths[0] = 1, keys
    missing = rows // 2 if rows > 2 else -1
    table = ops.row_table([0 if i == missing else memory[i].data_ptr() for i in range(rows)])
    q = torch.randn((rows, heads, dim), generator=g, device="cuda").bfloat16()
    bias = torch.randn((heads, n_dist), generator=g, device="cuda") if n_dist else None
    if rows > 2:
        memory[0].view(torch.bfloat16)[3 * row] = -float("inf")            # a key of the first head: -inf or inf by the query's sign
        q[0, 0, 0] = 1.0
        cache[0, 3, 0] = -float("inf")
    got = ops.attn_window(q.view(rows, -1), a, table, (lengths - 1).int(), 1, keys - 1, bias, 0, cache[0].numel() * 2).double().view(rows, heads, vdim)
    j = torch.arange(keys, device="cuda")
    for i in range(rows):
        if i == missing:
            assert (got[i] == 0).all()
            continue
        p = int(lengths[i]) - 1
        k = cache[i, :p + 1, :heads * dim].view(p + 1, heads, dim).double()
        v = k if shared else cache[i, :p + 1, heads * dim:].view(p + 1, heads, vdim).double()
        score = (k * q[i].double()).sum(-1) * dim ** -0.5
        if shared:
            score = score * factors[i].permute(0, 2, 1).reshape(-1, heads)[:p + 1].double()
        if bias is not None:
            score = score + bias.double().T[(p - j[:p + 1]).clamp(max=n_dist - 1)]
        hidden = (p - j[:p + 1] >= window) & (j[:p + 1] >= keep) if window else torch.zeros(p + 1, dtype=torch.bool, device="cuda")
        weight = score.masked_fill(hidden[:, None], -float("inf")).softmax(0)
        if shared and i == 0:
            v = v.clone()
            v[v.isinf()] = 0.0
            got[0, 0, 0] = 0.0                                             # 0 x inf
        want = (weight[:, :, None] * v).sum(0)
        if shared and i == 0:
            want[0, 0] = 0.0
        assert ((got[i] - want).abs() <= 2.0 ** -8 * want.abs() + 2e-5).all(), i


# of a wave's 32 columns and 64 keys at a time: (heads, kv heads, head sizes), (window, kept tokens, distances, scale), (starts, tokens).  Tables of one
# distance, of fewer than a tile, with room for the entries around it and without, and none; windows that end inside a wave, kept tokens that reach into
# it; first positions on both sides of a tile's edge, portions past the last full wave; keys that are values too, of a size with an odd number of blocks
@pytest.mark.parametrize("heads,kv,dim,vdim,shared", [(4, 4, 128, 128, False), (8, 2, 72, 40, False), (6, 2, 128, 64, False), (2, 2, 96, 96, True), (4, 4, 128, 128, True)])
@pytest.mark.parametrize("window,keep,n_dist,scale", [(0, 0, 0, 1.0), (0, 0, 0, -1.0), (97, 5, 1, 1.0), (64, 70, 17, 1.0), (150, 200, 90, -1.0), (300, 3, 2000, 1.0), (31, 64, 7900, 1.0)])
@pytest.mark.parametrize("starts,T", [([0, 64], 16), ([1, 257], 131), ([95, 0], 290)])
def test_tiles_of_keys_by_waves(heads, kv, dim, vdim, shared, window, keep, n_dist, scale, starts, T):
    """Against 64 bits: a rounding to bf16 and weights in two terms of bf16, whose error is below 2^-17 of the largest value."""
    import torch
    from glinthawk_amd import ops
    a = ops.window_attn(heads, kv, dim, vdim, scale * dim ** -0.5, window, keep, n_dist, shared)
    g = torch.Generator(device="cuda").manual_seed(T + n_dist)
    keys = max(starts) + T
    cache = torch.randn((2, keys, kv * (dim if shared else dim + vdim)), generator=g, device="cuda").bfloat16()
    groups = -(-keys // 32)
    factors = torch.rand((2, groups, kv, 32), generator=g, device="cuda") + 0.5
    memory = torch.cat([cache.view(2, -1).view(torch.uint8), factors.view(2, -1).view(torch.uint8)], 1).contiguous()
    q = torch.randn((2, T, heads, dim), generator=g, device="cuda").bfloat16()
    bias = 2.0 * torch.randn((heads, n_dist), generator=g, device="cuda") if n_dist else None
    got = ops.attn_window(q.view(2 * T, -1), a, ops.row_table([m.data_ptr() for m in memory]), torch.tensor(starts, dtype=torch.int32, device="cuda"), T, max(starts), bias, 0,
                          cache[0].numel() * 2).double().view(2, T, heads, vdim)
    for i, start in enumerate(starts):
        n = start + T
        k = cache[i, :n, :kv * dim].view(n, kv, dim).double().repeat_interleave(heads // kv, 1)
        v = k if shared else cache[i, :n, kv * dim:].view(n, kv, vdim).double().repeat_interleave(heads // kv, 1)
        distance = torch.arange(start, n, device="cuda")[:, None] - torch.arange(n, device="cuda")
        score = (k.permute(1, 0, 2)[:, None] * q[i].permute(1, 0, 2)[:, :, None].double()).sum(-1) * (scale * dim ** -0.5)     # (heads, tokens, keys)
        if shared:
            score = score * factors[i].permute(0, 2, 1).reshape(-1, kv)[:n].double().T.repeat_interleave(heads // kv, 0)[:, None]
        if n_dist:
            score = score + bias.double()[:, distance.clamp(0, n_dist - 1)]
        hidden = distance < 0
        if window:
            hidden = hidden | ((distance >= window) & (torch.arange(n, device="cuda") >= keep))
        weight = score.masked_fill(hidden, -float("inf")).softmax(-1)
        want = torch.stack([weight[h] @ v[:, h] for h in range(heads)], 1)
        assert ((got[i] - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -17 * v.abs().max() + 2e-5).all(), start


# two groups of work-groups an XCD, the second one smaller, of which some have no head
@pytest.mark.parametrize("window,keep,n_dist,scale", [(0, 0, 0, 1.0), (0, 0, 0, -1.0), (97, 5, 1, 1.0), (64, 70, 17, 1.0), (150, 200, 90, -1.0), (300, 3, 2000, 1.0), (31, 64, 7900, 1.0)])
@pytest.mark.parametrize("starts,T", [([0, 64], 16), ([1, 257], 131), ([95, 0], 290)])
def test_tiles_of_keys_of_many_heads(window, keep, n_dist, scale, starts, T):
    test_tiles_of_keys_by_waves(33, 33, 64, 64, False, window, keep, n_dist, scale, starts, T)


class Cache:
    """One attention layer's cache rows of a few contexts, filled by hand (heads padded to 8 elements with zeros)."""

    def __init__(self, shape, k, v, dtype, offset=256):
        import torch
        from glinthawk_amd import ops
        heads, kv, d, dv, window, keep, rows, bias_max = shape
        self.attn = ops.window_attn(heads, kv, d, dv, d ** -0.5, window, keep, int(bias_max) + 1)
        dp, vp = -(-d // 8) * 8, -(-dv // 8) * 8
        self.offset = offset
        self.regions = []
        for kk, vv in zip(k, v):
            T = kk.shape[0]
            full = np.zeros((T, kv * (dp + vp)), np.float32)
            full[:, : kv * dp].reshape(T, kv, dp)[:, :, :d] = kk
            full[:, kv * dp:].reshape(T, kv, vp)[:, :, :dv] = vv
            t = dev(full, dtype)
            assert t.shape[1] * t.element_size() == ops.window_row_bytes(self.attn, t.dtype)
            pad = torch.full((offset // t.element_size(),), float("nan"), dtype=t.dtype, device="cuda")
            self.regions.append(torch.cat([pad, t.reshape(-1)]).contiguous())
        self.rows = ops.row_table([r.data_ptr() for r in self.regions])
        self.dp = dp


def attend(shape, q, k, v, rel, start, n, dtype):
    """Rows [start_i, start_i + n) of every sequence as one call."""
    import torch
    from glinthawk_amd import ops
    heads, kv, d, dv, window, keep, rows, bias_max = shape
    cache = Cache(shape, k, v, dtype)
    qp = np.zeros((len(q), n, heads, cache.dp), np.float32)
    for i, (qq, s) in enumerate(zip(q, start)):
        qp[i, :, :, :d] = qq[s:s + n]
    bias = np.array([[rel[P.distance_bucket(t, rows, bias_max), h] for t in range(int(bias_max) + 1)] for h in range(heads)], np.float32)
    out = ops.attn_window(dev(qp.reshape(len(q) * n, -1), dtype), cache.attn, cache.rows, torch.tensor(start, dtype=torch.int32, device="cuda"), n, max(start),
                          torch.from_numpy(bias).cuda(), cache.offset)
    return back(out).reshape(len(q), n, heads, dv)


def attention_case(name, T, seed, n_seq=1, sharp=False):
    shape = ATTENTIONS[name]
    heads, kv, d, dv, window, keep, rows, bias_max = shape
    rng = np.random.default_rng(seed)
    q = [M.to_bf16(rng.standard_normal((T, heads, d))) for _ in range(n_seq)]
    k = [M.to_bf16(rng.standard_normal((T, kv, d))) for _ in range(n_seq)]
    v = [M.to_bf16(rng.standard_normal((T, kv, dv))) for _ in range(n_seq)]
    rel = rng.standard_normal((rows, heads)).astype(np.float32)
    want = [P.windowed_attention(*(a.astype(np.float64) for a in (qq, kk, vv)), d ** -0.5, rel.astype(np.float64), bias_max, window or T + 1, keep)
            for qq, kk, vv in zip(q, k, v)]
    return shape, q, k, v, rel, want


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", list(ATTENTIONS))
def test_windowed_attention(name, dtype):
    """A whole prompt, portions from anywhere, single tokens at and around the window's edges, two sequences in a call."""
    T = 150
    shape, q, k, v, rel, want = attention_case(name, T, 3, n_seq=2)
    tol = 1e-5 if dtype == "f32" else 8e-3
    assert_rows(np.stack(attend(shape, q, k, v, rel, [0, 0], T, dtype)).reshape(2 * T, -1), np.stack(want).reshape(2 * T, -1), tol, "whole")
    window, keep = shape[4], shape[5]
    for start, n in (([0, 70], 2), ([13, 90], 33), ([64, 1], 64), ([100, 37], 17), ([16, 48], 80)):
        w = np.stack([a[s:s + n] for a, s in zip(want, start)])
        assert_rows(attend(shape, q, k, v, rel, start, n, dtype).reshape(2 * n, -1), w.reshape(2 * n, -1), tol, f"portion {start}+{n}")
    for p in sorted({0, 1, max(0, keep - 1), keep, window - 1, window, window + 1, window + keep, T - 1} & set(range(T))):
        w = np.stack([a[p] for a in want])
        assert_rows(attend(shape, q, k, v, rel, [p, p], 1, dtype)[:, 0].reshape(2, -1), w.reshape(2, -1), tol, f"token {p}")


# more work-groups than the CUs hold (two blocks of heads each, where their number is even), as many as they hold and few (eight waves on a row's keys)
@pytest.mark.parametrize("contexts", [400, 40, 3])
@pytest.mark.parametrize("name", ["grouped", "matrix", "own", "open"])
def test_windowed_attention_of_many_contexts(name, contexts):
    """Single tokens at another position in every context, an uneven number of keys to every wave."""
    T = 150
    shape, q, k, v, rel, want = attention_case(name, T, 5, n_seq=2)
    start = [(37 * i + 11) % T for i in range(contexts)]
    pick = [i % 2 for i in range(contexts)]
    got = attend(shape, [q[i] for i in pick], [k[i] for i in pick], [v[i] for i in pick], rel, start, 1, "bf16")
    assert_rows(got[:, 0].reshape(contexts, -1), np.stack([want[i][s] for i, s in zip(pick, start)]).reshape(contexts, -1), 8e-3, "tokens")


@pytest.mark.parametrize("dtype", DTYPES)
def test_windowed_attention_over_many_splits(dtype):
    """Single tokens behind thousands of keys, in more splits than their merge takes at once (64 at most), and than a head has values; contexts that end in
    the first of them and in the middle."""
    T = 5000
    heads, kv, d, dv, _, _, rows, bias_max = shape = ATTENTIONS["open"]
    rng = np.random.default_rng(9)
    start = [T - 1, 40, 2600]
    q, k, v = ([M.to_bf16(rng.standard_normal((T, n, e))) for _ in start] for n, e in ((heads, d), (kv, d), (kv, dv)))
    rel = rng.standard_normal((rows, heads)).astype(np.float32)
    want = np.zeros((3, heads, dv))
    for i, s in enumerate(start):
        bias = rel[[P.distance_bucket(s - j, rows, bias_max) for j in range(s + 1)]].astype(np.float64)
        for h in range(heads):
            score = (k[i][: s + 1, h // (heads // kv)].astype(np.float64) @ q[i][s, h]) * d ** -0.5 + bias[:, h]
            p = np.exp(score - score.max())
            want[i, h] = p / p.sum() @ v[i][: s + 1, h // (heads // kv)].astype(np.float64)
    tol = 1e-5 if dtype == "f32" else 8e-3
    for n in (3, 1):
        got = attend(shape, q[:n], k[:n], v[:n], rel, start[:n], 1, dtype)
        assert_rows(got.reshape(n, -1), want[:n].reshape(n, -1), tol, f"{n} contexts")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["grouped", "matrix", "ten", "own"])
def test_one_key_stands_out(name, dtype):
    """Every key in turn made the one that its query's score picks: seen exactly where the window or the kept tokens show it, and just
    not seen one position further."""
    shape = ATTENTIONS[name]
    heads, kv, d, dv, window, keep, rows, bias_max = shape
    T = window + keep + 70
    rng = np.random.default_rng(4)
    q0 = rng.standard_normal((heads, d))
    q0 *= np.sqrt(d) * 4 / np.linalg.norm(q0, axis=-1, keepdims=True)
    q = M.to_bf16(np.broadcast_to(q0, (T, heads, d)))
    v = M.to_bf16(rng.standard_normal((T, kv, dv)))
    rel = np.zeros((rows, heads), np.float32)
    for j in (0, keep - 1, keep, keep + 1, 31, T - 2 * window // 3):
        if j < 0:
            continue
        k = M.to_bf16(0.02 * rng.standard_normal((T, kv, d)))
        k[j] = M.to_bf16(np.stack([q[0, g * (heads // kv)] for g in range(kv)]))
        want = P.windowed_attention(*(a.astype(np.float64) for a in (q, k, v)), d ** -0.5, rel.astype(np.float64), bias_max, window, keep)
        got = attend(shape, [q], [k], [v], rel, [0], T, dtype)[0]
        tol = 1e-5 if dtype == "f32" else 1e-2
        assert_rows(got.reshape(T, -1), want.reshape(T, -1), tol, f"key {j} in a prompt")
        seen = np.abs(got[:, 0] - v[j, 0]).max(-1) < 0.2
        expect = [P.visible(i, j, window, keep) for i in range(T)]
        assert seen.tolist() == expect, f"key {j}"
        for p in (j, j + window - 1, j + window, T - 1):
            if p < T:
                one = attend(shape, [q], [k], [v], rel, [p], 1, dtype)[0]
                assert_rows(one.reshape(1, -1), want[p].reshape(1, -1), tol, f"key {j} decoded at {p}")


@pytest.mark.parametrize("dtype", DTYPES)
def test_bias_by_distance_in_every_row_of_the_table(dtype):
    """Scores from the bias alone: each query's output is the bias-weighted mean of the values."""
    shape = (4, 2, 16, 24, 90, 8, 14, 77)
    T = 130
    rng = np.random.default_rng(5)
    q, k = np.zeros((T, 4, 16), np.float32), np.zeros((T, 2, 16), np.float32)
    v = M.to_bf16(rng.standard_normal((T, 2, 24)))
    rel = (3 * rng.standard_normal((14, 4))).astype(np.float32)
    want = P.windowed_attention(*(a.astype(np.float64) for a in (q, k, v)), 0.25, rel.astype(np.float64), 77, 90, 8)
    got = attend(shape, [q], [k], [v], rel, [0], T, dtype)[0]
    assert_rows(got.reshape(T, -1), want.reshape(T, -1), 1e-5 if dtype == "f32" else 5e-3)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n_tokens", [1, 4, 250, 600])
def test_query_key_norm_and_append(dtype, n_tokens):
    import torch
    from glinthawk_amd import ops
    heads, kv, d, dv, width, eps = 6, 3, 20, 12, 88, 2e-3
    rng = np.random.default_rng(6)
    nq, nk, nv = heads * d, kv * d, kv * dv
    a = ops.window_attn(heads, kv, d, dv, 1.0, 9, 2, 5)
    x = M.to_bf16(rng.standard_normal((2 * n_tokens, width)))
    w, b = M.to_bf16(rng.standard_normal((nq + nk + nv, width)) / 9), M.to_bf16(rng.standard_normal(nq + nk + nv))
    qn, kn = M.to_bf16(1 + 0.3 * rng.standard_normal(nq)), M.to_bf16(1 + 0.3 * rng.standard_normal(nk))
    y = x.astype(np.float64) @ w.T + b
    T = n_tokens + 40
    row = ops.window_row_bytes(a, torch_dtype(dtype)) // (4 if dtype == "f32" else 2)
    regions = [torch.full((T, row), 7.0, dtype=torch_dtype(dtype), device="cuda") for _ in range(3)]
    start = [3, 39]
    q = ops.matmul_window_append(dev(x, dtype), dev(w, dtype), a, ops.row_table([regions[0].data_ptr(), regions[1].data_ptr()]),
                                 torch.tensor(start, dtype=torch.int32, device="cuda"), n_tokens, dev(b, dtype), dev(qn, dtype), dev(kn, dtype), eps)
    tol = 1e-5 if dtype == "f32" else 1e-2
    dp, vp = 24, 16
    got_q = back(q).reshape(-1, heads, dp)
    assert_rows(got_q[:, :, :d].reshape(len(x), -1), P.rms_norm(y[:, :nq], eps, qn.astype(np.float64)), tol, "q")
    assert np.abs(got_q[:, :, d:]).max() == 0
    for i in range(2):
        c = back(regions[i])
        part = y[i * n_tokens:(i + 1) * n_tokens]
        mine = c[start[i]:start[i] + n_tokens]
        gk, gv = mine[:, : kv * dp].reshape(-1, kv, dp), mine[:, kv * dp:].reshape(-1, kv, vp)
        assert_rows(gk[:, :, :d].reshape(n_tokens, -1), P.rms_norm(part[:, nq:nq + nk], eps, kn.astype(np.float64)), tol, "k")
        assert_rows(gv[:, :, :dv].reshape(n_tokens, -1), part[:, nq + nk:], tol, "v")
        assert np.abs(gk[:, :, d:]).max() == 0 and np.abs(gv[:, :, dv:]).max() == 0
        c[start[i]:start[i] + n_tokens] = 7.0
        assert (c == 7.0).all(), "rows outside the call were written"


# work-groups that take several tokens each, some one less; 16 bytes and 8 at a time, padded heads, more heads than keys have, a row that ends inside a group
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,kv,d,dv,n_tokens", [(32, 32, 128, 128, 521), (40, 8, 128, 64, 1111), (60, 20, 52, 36, 1301), (25, 5, 104, 72, 1201)])
def test_query_key_norm_and_append_of_many_tokens(dtype, heads, kv, d, dv, n_tokens):
    """Three contexts, the second without one: its tokens are passed over.  Against 64 bits, bound as above."""
    import torch
    from glinthawk_amd import ops
    width, eps = 64, 2e-3
    g = torch.Generator(device="cuda").manual_seed(heads)

    def draw(*shape):
        return torch.randn(shape, generator=g, device="cuda").bfloat16().to(torch_dtype(dtype))

    nq, nk, nv = heads * d, kv * d, kv * dv
    a = ops.window_attn(heads, kv, d, dv, 1.0, 9, 2, 5)
    x, w, b, qn, kn = draw(3 * n_tokens, width), draw(nq + nk + nv, width) / 8, draw(nq + nk + nv), 1 + draw(nq) / 4, 1 + draw(nk) / 4
    y = x.double() @ w.double().T + b.double()
    row = ops.window_row_bytes(a, torch_dtype(dtype)) // (4 if dtype == "f32" else 2)
    regions = [torch.full((n_tokens + 11, row), 7.0, dtype=torch_dtype(dtype), device="cuda") for _ in range(2)]
    start = [3, 0, 11]
    q = ops.matmul_window_append(x, w, a, ops.row_table([regions[0].data_ptr(), 0, regions[1].data_ptr()]), torch.tensor(start, dtype=torch.int32, device="cuda"),
                                 n_tokens, b, qn, kn, eps)

    def unit(v, weight):
        return v / torch.sqrt((v * v).mean(-1, keepdim=True) + eps) * weight.double()

    def close(got, want, size, what):
        got = got.double().reshape(len(want), -1, (size + 7) // 8 * 8)
        assert got[:, :, size:].abs().sum() == 0, what
        assert_rows(got[:, :, :size].reshape(len(want), -1).cpu().numpy(), want.cpu().numpy(), 1e-5 if dtype == "f32" else 1e-2, what)

    kp = kv * ((d + 7) // 8 * 8)
    assert q[n_tokens:2 * n_tokens].abs().sum() == 0
    for i, region in ((0, regions[0]), (2, regions[1])):
        at = slice(i * n_tokens, (i + 1) * n_tokens)
        mine = region[start[i]:start[i] + n_tokens]
        close(q[at], unit(y[at, :nq], qn), d, "q")
        close(mine[:, :kp], unit(y[at, nq:nq + nk], kn), d, "k")
        close(mine[:, kp:], y[at, nq + nk:], dv, "v")
        assert (region[:start[i]] == 7.0).all() and (region[start[i] + n_tokens:] == 7.0).all(), "rows outside the call were written"


# long rows of many tokens, which work-groups take in turn, some one less
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,kv,d,dv,n_tokens", [(32, 32, 128, 128, 1100), (64, 16, 128, 40, 1301)])
def test_query_key_norm_and_append_of_long_rows(dtype, heads, kv, d, dv, n_tokens):
    test_query_key_norm_and_append_of_many_tokens(dtype, heads, kv, d, dv, n_tokens)


MLSTMS = {"small": (3, 12, 20, 9.0), "round": (2, 64, 64, 15.0), "tall": (1, 130, 40, 5.0), "broad": (2, 32, 200, 15.0), "big": (1, 256, 136, 15.0), "huge": (1, 300, 70, 15.0)}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", list(MLSTMS))
def test_mlstm(name, dtype):
    """Mixer up to its output projection, for gates from never forgetting to forgetting at once: a whole prompt, portions, token by token;
    the state behind the last token as well."""
    import torch
    from glinthawk_amd import ops
    H, d, dv, cap = MLSTMS[name]
    width, eps, T = 72, 1e-4, 214
    from glinthawk_amd._lib import GhMlstm
    m = GhMlstm(H, d, dv, cap, eps)
    rng = np.random.default_rng(8)
    rows, gate_row = ops.mlstm_weight_rows(m)
    hd, hv = H * d, H * dv
    w = np.zeros((rows, width), np.float32)
    w[:2 * hd + 2 * hv] = rng.standard_normal((2 * hd + 2 * hv, width)) / np.sqrt(width)
    w[gate_row:gate_row + 2 * H] = rng.standard_normal((2 * H, width)) / 3
    w = M.to_bf16(w)
    bi, bf = M.to_bf16(2 * rng.standard_normal(H)), M.to_bf16(np.linspace(-6, 7, H) if H > 1 else np.array([3.0]))
    norm = M.to_bf16(1 + 0.2 * rng.standard_normal(hv))
    x = M.to_bf16(rng.standard_normal((T, width)))
    X, W = x.astype(np.float64), w.astype(np.float64)
    split = np.split(W[:2 * hd + 2 * hv], [hd, 2 * hd, 2 * hd + hv])
    q = (X @ split[0].T).reshape(T, H, d) * d ** -0.5
    k, v, g = (X @ split[1].T).reshape(T, H, d), (X @ split[2].T).reshape(T, H, dv), X @ split[3].T
    li = P.soft_cap(X @ W[gate_row:gate_row + H].T + bi, cap)
    lf = P.log_sigmoid(P.soft_cap(X @ W[gate_row + H:gate_row + 2 * H].T + bf, cap))
    o, (S, n, mm) = P.mlstm_recurrence(q, k, v, li, lf)
    want = P.rms_norm(o, eps).reshape(T, hv) * norm / (1 + np.exp(-g))
    tol = 5e-5 if dtype == "f32" else 4e-2
    weights = [dev(a, dtype) for a in (w, bi, bf, norm)]
    offset = 512

    def run(cuts, label):
        state = torch.full((offset // 4 + ops.mlstm_state_bytes(m) // 4,), float("nan"), device="cuda")     # position 0 needs no cleared slot
        table = ops.row_table([state.data_ptr()])
        outs, at = [], 0
        for c in cuts:
            outs.append(back(ops.mlstm_forward(dev(x[at:at + c], dtype), weights[0], m, *weights[1:], table, torch.tensor([at], dtype=torch.int32, device="cuda"), c, offset)))
            at += c
        got = np.concatenate(outs)
        assert_rows(got, want[:at], tol, label, 1.0 if dtype == "f32" else 5.0)
        if at == T:
            vp = -(-dv // 4) * 4
            st = state[offset // 4:].cpu().numpy().astype(np.float64)
            gS = st[:H * d * vp].reshape(H, d, vp)
            assert_rows(gS[:, :, :dv].reshape(H, -1), S.reshape(H, -1), tol, label + ": S")
            assert_rows(st[H * d * vp:H * d * vp + H * d].reshape(1, -1), n.reshape(1, -1), tol, label + ": n")
            assert np.abs(st[-H:] - mm).max() <= (1e-4 if dtype == "f32" else 5e-2), label + ": m"

    run([T], "whole")
    run([2, 3, 5, 64, 1, 63, 65, 11], "portions")
    run([130, 1, 1, 1, 81], "tokens between portions")
    run([1] * 40, "token by token")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width,batch", [(4096, 1), (4096, 7), (4096, 32), (1000, 5), (4096, 200), (4104, 200)])
def test_mlstm_gates_of_many_planes(width, batch, dtype):
    """Two tokens of each context, one a call: the walk adds up the gates' sums over the K ranges that the product left, a plane a lane (in 16 bits
    sixteen of them; where the gates of 192 rows and more are a product of their own, one or, by the width, sixteen).  The state's m is made of the gates alone."""
    import torch
    from glinthawk_amd import ops
    from glinthawk_amd._lib import GhMlstm
    H, d, dv, cap, eps = 2, 16, 24, 15.0, 1e-4
    m = GhMlstm(H, d, dv, cap, eps)
    rng = np.random.default_rng(width + batch)
    rows, gate_row = ops.mlstm_weight_rows(m)
    hd, hv = H * d, H * dv
    w = np.zeros((rows, width), np.float32)
    w[:2 * hd + 2 * hv] = rng.standard_normal((2 * hd + 2 * hv, width)) / np.sqrt(width)
    w[gate_row:gate_row + 2 * H] = 3 * rng.standard_normal((2 * H, width)) / np.sqrt(width)
    w = M.to_bf16(w)
    bi, bf, norm = M.to_bf16(rng.standard_normal(H)), M.to_bf16(np.array([-2.0, 3.0])), M.to_bf16(1 + 0.2 * rng.standard_normal(hv))
    x = M.to_bf16(rng.standard_normal((2, batch, width)))
    X, W = x.astype(np.float64), w.astype(np.float64)
    split = np.split(W[:2 * hd + 2 * hv], [hd, 2 * hd, 2 * hd + hv])
    q, k = (X @ split[0].T).reshape(2, batch, H, d) * d ** -0.5, (X @ split[1].T).reshape(2, batch, H, d)
    v, g = (X @ split[2].T).reshape(2, batch, H, dv), X @ split[3].T
    li = P.soft_cap(X @ W[gate_row:gate_row + H].T + bi, cap)
    lf = P.log_sigmoid(P.soft_cap(X @ W[gate_row + H:gate_row + 2 * H].T + bf, cap))
    weights = [dev(a, dtype) for a in (w, bi, bf, norm)]
    state = torch.full((batch, ops.mlstm_state_bytes(m) // 4), float("nan"), device="cuda")
    table = ops.row_table([state[i].data_ptr() for i in range(batch)])
    tol = 5e-5 if dtype == "f32" else 4e-2
    for t in range(2):
        got = back(ops.mlstm_forward(dev(x[t], dtype), weights[0], m, *weights[1:], table, torch.full((batch,), t, dtype=torch.int32, device="cuda"), 1))
        at = state.cpu().numpy().astype(np.float64)
        for i in range(batch):
            o, (S, n, mm) = P.mlstm_recurrence(q[:t + 1, i], k[:t + 1, i], v[:t + 1, i], li[:t + 1, i], lf[:t + 1, i])
            want = P.rms_norm(o, eps).reshape(t + 1, hv) * norm / (1 + np.exp(-g[:t + 1, i]))
            # the output is divided by n . q and normed, whose rounding, some 2e-6 of |n| |q|, grows by as much as they cancel: up to ten times is looked at
            if (np.abs((n * q[t, i]).sum(-1)) >= 0.1 * np.linalg.norm(n, axis=-1) * np.linalg.norm(q[t, i], axis=-1)).all():
                assert_rows(got[i:i + 1], want[t:], tol, f"{t} {i}", 1.0 if dtype == "f32" else 5.0)
            # at 200 rows of 16 bits k and v are rounded, the gates' sums are not
            assert_rows(at[i, :hd * dv].reshape(H, -1), S.reshape(H, -1), tol, f"{t} {i}: S")
            assert_rows(at[i, hd * dv:hd * dv + hd].reshape(1, -1), n.reshape(1, -1), tol, f"{t} {i}: n")
            # fp32 sums of exact products: a few units of 2^-24 of sqrt(width) terms of size 3 / sqrt(width), through gates whose slopes are at most 1
            assert np.abs(at[i, -H:] - mm).max() <= 1e-4, f"{t} {i}: m"


@pytest.mark.parametrize("dtype", DTYPES)
def test_mlstm_extreme_gates(dtype):
    """A far token written once with a strong input gate and kept by open forget gates must still be read, and a closed forget gate
    must wipe it."""
    import torch
    from glinthawk_amd import ops
    from glinthawk_amd._lib import GhMlstm
    H, d, dv, cap, T = 2, 16, 24, 15.0, 300
    m = GhMlstm(H, d, dv, cap, 1e-5)
    rows, gate_row = ops.mlstm_weight_rows(m)
    width = d + dv + 4
    # input columns: [key | value | query switch, unused, input gate, forget gate]
    w = np.zeros((rows, width), np.float32)
    for h in range(H):
        w[h * d:(h + 1) * d, :d] = np.eye(d) * np.sqrt(d)
        w[H * d + h * d:H * d + (h + 1) * d, :d] = np.eye(d)
        w[2 * H * d + h * dv:2 * H * d + (h + 1) * dv, d:d + dv] = np.eye(dv)
        w[gate_row + h, d + dv + 2] = 1
        w[gate_row + H + h, d + dv + 3] = 1 if h == 0 else -1        # the second head forgets where the first keeps
    rng = np.random.default_rng(2)
    x = np.zeros((T, width), np.float32)
    x[:, d:d + dv] = rng.standard_normal((T, dv))
    x[:, :d] = 0.05 * rng.standard_normal((T, d))
    x[:, d + dv + 2] = -8.0
    x[:, d + dv + 3] = 12.0
    x[5, 3], x[5, d + dv + 2] = 4.0, 6.0
    x[T - 1, 3] = 4.0
    x, w = M.to_bf16(x), M.to_bf16(w)
    X, W = x.astype(np.float64), w.astype(np.float64)
    q = (X @ W[:H * d].T).reshape(T, H, d) * d ** -0.5
    k, v = (X @ W[H * d:2 * H * d].T).reshape(T, H, d), (X @ W[2 * H * d:2 * H * d + H * dv].T).reshape(T, H, dv)
    li, lf = P.soft_cap(X @ W[gate_row:gate_row + H].T, cap), P.log_sigmoid(P.soft_cap(X @ W[gate_row + H:gate_row + 2 * H].T, cap))
    o, _ = P.mlstm_recurrence(q, k, v, li, lf)
    want = P.rms_norm(o, 1e-5).reshape(T, -1) / 2           # the output gate sees zero
    far = P.rms_norm(v[5], 1e-5)
    assert np.abs(want[-1, :dv] * 2 - far[0]).max() < 0.05 and np.abs(want[-1, dv:] * 2 - far[1]).max() > 0.5
    zeros, ones = dev(np.zeros(H), dtype), dev(np.ones(H * dv), dtype)
    for cuts in ([T], [100, 7, 193], [299, 1]):
        state = torch.empty((ops.mlstm_state_bytes(m) // 4,), device="cuda").fill_(float("nan"))
        table, at = ops.row_table([state.data_ptr()]), 0
        for c in cuts:
            got = back(ops.mlstm_forward(dev(x[at:at + c], dtype), dev(w, dtype), m, zeros, zeros, ones, table, torch.tensor([at], dtype=torch.int32, device="cuda"), c))
            assert_rows(got, want[at:at + c], 1e-4 if dtype == "f32" else 3e-2, f"{cuts} at {at}")
            at += c


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,d,dv,batch", [(4, 256, 384, 7), (8, 64, 64, 1), (3, 130, 136, 11), (1, 12, 20, 9), (2, 300, 70, 5)])
def test_mlstm_walk_of_many_contexts(H, d, dv, batch, dtype):
    """Work-groups take (context, head) pairs by eights and the rest as they come: every context as in a call of its own, where there are too few pairs for
    that, bit for bit (small whole numbers: the projections are exact in any order of their sums), and a slot without a context is left alone."""
    import torch
    from glinthawk_amd import ops
    from glinthawk_amd._lib import GhMlstm
    width, empty = 8, batch // 2 if batch > 1 else None
    m = GhMlstm(H, d, dv, 15.0, 1e-5)
    rows, _ = ops.mlstm_weight_rows(m)
    rng = np.random.default_rng(batch)
    w = dev(rng.integers(-2, 3, (rows, width)).astype(np.float32), dtype)
    bias, norm = dev(np.linspace(-3, 3, H), dtype), dev(np.ones(H * dv), dtype)
    n = ops.mlstm_state_bytes(m) // 4
    state0 = torch.from_numpy(rng.standard_normal((batch, n)).astype(np.float32)).cuda()
    start = torch.from_numpy((np.arange(batch) % 3).astype(np.int32)).cuda()  # some start anew
    for n_tokens in (1, 3):
        x = dev(rng.integers(-2, 3, (batch * n_tokens, width)).astype(np.float32), dtype)
        state = state0.clone()
        got = ops.mlstm_forward(x, w, m, bias, bias, norm, ops.row_table([0 if i == empty else state[i].data_ptr() for i in range(batch)]), start, n_tokens)
        for i in range(batch):
            alone = state0[i].clone()
            if i != empty:
                one = ops.mlstm_forward(x[i * n_tokens:(i + 1) * n_tokens].contiguous(), w, m, bias, bias, norm, ops.row_table([alone.data_ptr()]), start[i:i + 1].contiguous(),
                                        n_tokens)
                assert torch.equal(got[i * n_tokens:(i + 1) * n_tokens], one), i
            assert torch.equal(state[i], alone), i


# head sizes below and at each of the kernel's three, that leave part of a step of 32 or of a tile of 64 columns idle; one slice of columns and several;
# portions of one chunk, of the sixteen that the scan takes at once, of more, all with a last chunk of few tokens
@pytest.mark.parametrize("H,d,dv", [(3, 40, 8), (2, 64, 136), (1, 72, 64), (4, 128, 72), (2, 232, 200), (1, 256, 64)])
@pytest.mark.parametrize("cuts", [(24, 65), (1025, 127), (1100,), (33, 1024)])
def test_mlstm_chunks(H, d, dv, cuts):
    """Against 64 bits, two contexts and a slot without one.  Weights of the keys and the state meet their partners in two bf16 terms (2^-17); a log gate is
    off by 2^-22 of itself, and what it is summed over decays with it: weights that matter, above e^-20, are off by 20 x 2^-22 < 2^-17.  Four such errors are
    allowed to the sums of absolute values, for the numerator and for the denominator; the state is allowed two."""
    import torch
    from glinthawk_amd import ops
    from glinthawk_amd._lib import GhMlstm
    width, T, B, eps = 8, sum(cuts), 3, 1e-4
    m = GhMlstm(H, d, dv, 15.0, eps)
    rows, gate_row = ops.mlstm_weight_rows(m)
    rng = np.random.default_rng(d + dv)
    w = rng.integers(-2, 3, (rows, width)).astype(np.float32)             # small whole numbers: the projections are exact
    w[gate_row:gate_row + 2 * H] *= 0.5
    bias_i, bias_f, norm = np.linspace(-2, 2, H).astype(np.float32), np.linspace(1, 5, H).astype(np.float32), np.ones(H * dv, np.float32)
    bias_i, bias_f = M.to_bf16(bias_i), M.to_bf16(bias_f)
    x = rng.integers(-1, 2, (B, T, width)).astype(np.float32)
    state = torch.full((B, ops.mlstm_state_bytes(m) // 4), float("nan"), device="cuda")
    table = ops.row_table([0 if i == 1 else state[i].data_ptr() for i in range(B)])
    got, at = [], 0
    for c in cuts:
        out = ops.mlstm_forward(dev(x[:, at:at + c].reshape(B * c, width), "bf16"), dev(w, "bf16"), m, dev(bias_i, "bf16"), dev(bias_f, "bf16"), dev(norm, "bf16"), table,
                                torch.full((B,), at, dtype=torch.int32, device="cuda"), c)
        got.append(back(out).reshape(B, c, H, dv))
        at += c
    got = np.concatenate(got, 1)
    assert (got[1] == 0).all()
    for b in (0, 2):
        y = x[b].astype(np.float64) @ w.T
        q, k, v = (a.reshape(T, H, -1) for a in np.split(y[:, :2 * H * d + H * dv], [H * d, 2 * H * d], 1))
        q = q * d ** -0.5
        gate = 1 / (1 + np.exp(-y[:, 2 * H * d + H * dv:2 * H * (d + dv)].reshape(T, H, dv)))
        li = P.soft_cap(y[:, gate_row:gate_row + H] + bias_i, 15.0)
        lf = P.log_sigmoid(P.soft_cap(y[:, gate_row + H:gate_row + 2 * H] + bias_f, 15.0))
        S, n, S_abs, n_abs, top = np.zeros((H, d, dv)), np.zeros((H, d)), np.zeros((H, d, dv)), np.zeros((H, d)), np.zeros(H)
        for t in range(T):
            m_new = np.maximum(lf[t] + top, li[t])
            f, i = np.exp(lf[t] + top - m_new), np.exp(li[t] - m_new)
            kv = k[t][:, :, None] * v[t][:, None]
            S, n = f[:, None, None] * S + i[:, None, None] * kv, f[:, None] * n + i[:, None] * k[t]
            S_abs, n_abs = f[:, None, None] * S_abs + i[:, None, None] * np.abs(kv), f[:, None] * n_abs + i[:, None] * np.abs(k[t])
            top = m_new
            den = np.maximum(np.abs((n * q[t]).sum(1)), np.exp(-top))[:, None] + 1e-6
            o = (S * q[t][:, :, None]).sum(1) / den
            off = 2.0 ** -15 * ((S_abs * np.abs(q[t])[:, :, None]).sum(1) + np.abs(o) * (n_abs * np.abs(q[t])).sum(1)[:, None]) / den
            rms = np.sqrt((o ** 2).mean(1) + eps)[:, None]
            off = (off + np.abs(o) * np.sqrt((off ** 2).mean(1))[:, None] / rms) / rms * gate[t]
            want = o / rms * gate[t]
            assert (np.abs(got[b, t] - want) <= 2.0 ** -8 * np.abs(want) + off + 1e-6).all(), (b, t)
        vp = -(-dv // 4) * 4
        st = state[b].cpu().numpy().astype(np.float64)
        assert (np.abs(st[:H * d * vp].reshape(H, d, vp)[:, :, :dv] - S) <= 2.0 ** -16 * S_abs + 1e-9).all(), b
        assert (np.abs(st[H * d * vp:H * d * (vp + 1)].reshape(H, d) - n) <= 2.0 ** -16 * n_abs + 1e-9).all(), b
        assert (np.abs(st[-H:] - top) <= 2.0 ** -22 * np.abs(lf).sum(0) + 2.0 ** -20 * 15).all(), b


@pytest.mark.parametrize("d,dv,T", [(64, 64, 320), (128, 192, 257), (256, 512, 512)])
def test_mlstm_same_bits_twice(d, dv, T):
    """The chunks of a prompt share their LDS tiles: with enough work-groups for the waves of one to drift apart, the same inputs give the
    same bits, outputs and state."""
    import torch
    from glinthawk_amd import ops
    from glinthawk_amd._lib import GhMlstm
    H, width, batch = 8, 64, 8
    m = GhMlstm(H, d, dv, 15.0, 1e-5)
    rows, _ = ops.mlstm_weight_rows(m)
    gen = torch.Generator(device="cuda").manual_seed(3)
    x, w = (torch.randn(n, width, generator=gen, device="cuda").to(torch.bfloat16) for n in (batch * T, rows))
    w *= width ** -0.5
    zeros, ones = torch.zeros(H, dtype=torch.bfloat16, device="cuda"), torch.ones(H * dv, dtype=torch.bfloat16, device="cuda")
    start = torch.zeros(batch, dtype=torch.int32, device="cuda")
    first = None
    for _ in range(4):
        state = torch.zeros((batch, ops.mlstm_state_bytes(m) // 4), device="cuda")
        table = ops.row_table([state[i].data_ptr() for i in range(batch)])
        out = ops.mlstm_forward(x, w, m, zeros, zeros, ones, table, start, T)
        got = (out.cpu(), state.cpu())
        first = first or got
        assert torch.equal(got[0], first[0]) and torch.equal(got[1], first[1])


# ---- whole models ---------------------------------------------------------------------------------
@pytest.fixture(scope="module")
def models(tmp_path_factory):
    made = {}

    def get(name, T=120):
        if name not in made:
            cfg = M.CONFIGS[name]
            weights = M.random_weights(cfg, seed=sum(map(ord, name)))
            path = M.write_model(tmp_path_factory.mktemp(name), cfg, weights)
            rng = np.random.default_rng(11)
            # At a first token a head's normed output is v times the sign of k . q: where that product almost vanishes, rounding decides.
            # Sequences that rounding errors of weights in bf16 throw off like that say nothing about the code and are drawn again.
            noisy = {k: a * (1 + 2.0 ** -9 * rng.standard_normal(a.shape)) for k, a in weights.items()}
            seqs, want, residuals = [], [], []
            while len(seqs) < 4:
                s, res = rng.integers(0, cfg["vocab"], T), []
                w = P.forward(cfg, weights, s, residuals=res)
                if np.sort(logit_error(P.forward(cfg, noisy, s), w))[-2:].mean() < 0.06:
                    seqs.append(s)
                    want.append(w)
                    residuals = residuals or res
            made[name] = (path, cfg, weights, seqs, want, residuals)
        return made[name]

    return get


def open_stage(path, dtype, n=4, **kw):
    from glinthawk_amd.stage import DesignStage
    return DesignStage(path, dtype, n, n, **kw)


NAMES = list(M.CONFIGS)


def decode_step(st, ids, tokens, positions):
    st.new_state(len(ids))
    st.set_prompts(ids, tokens, positions, prompt_length=1, max_completion_length=st.max_positions)
    assert st.forward()
    return st.logits(len(ids))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", NAMES)
def test_prompt_and_residual_stream(models, name, dtype):
    path, cfg, _, seqs, want, residuals = models(name)
    st = open_stage(path, dtype)
    T = len(seqs[0])
    logits, nxt, res = st.prefill_logits([5], [0], seqs[0][None], range(T), True, cfg["width"])
    for i, (a, b) in enumerate(zip(res, residuals)):
        assert_rows(a, b, MODEL_TOL[dtype], f"stream behind run {i}", 1.0 if dtype == "f32" else 5.0)
    assert_logits(logits, want[0], dtype)
    assert int(nxt[0]) == int(np.argmax(logits[-1]))
    if dtype == "f32":
        assert (np.argmax(logits, -1) == np.argmax(want[0], -1)).all()
    st.close()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", NAMES)
def test_decoding_token_by_token(models, name, dtype):
    path, cfg, _, seqs, want, _ = models(name)
    st = open_stage(path, dtype)
    got = []
    for i, tok in enumerate(seqs[1]):
        got.append(decode_step(st, [3], [tok], [i])[0])
    assert_logits(np.stack(got), want[1], dtype)
    st.close()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("cuts", [[2] * 30 + [60], [3, 7, 2, 64, 5, 39], [65, 2, 53], [119, 1], [31, 33, 1, 1, 54]])
def test_portions(models, name, dtype, cuts):
    path, cfg, _, seqs, want, _ = models(name)
    st = open_stage(path, dtype)
    at, got = 0, []
    for c in cuts:
        part = seqs[0][at:at + c]
        logits = decode_step(st, [9], part, [at]) if c == 1 else st.prefill_logits([9], [at], part[None], range(c))[0]
        got.append(logits)
        at += c
    assert_logits(np.concatenate(got), want[0], dtype)
    st.close()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("paged", [False, True])
def test_unequal_requests_in_a_batch_and_slots_used_again(models, name, dtype, paged):
    """Four requests of different lengths, prefilled in pairs at different positions and decoded together, then all over again in the
    slots they gave back: each answers as if it were alone."""
    path, cfg, _, seqs, want, _ = models(name)
    st = open_stage(path, dtype, 4, paged=paged)
    for turn in range(2):
        ids = [10 * turn + k for k in range(4)]
        order = [0, 1, 2, 3] if turn == 0 else [2, 0, 3, 1]            # other sequences in other slots the second time
        at = [0, 0, 0, 0]

        def go(which, n):
            toks = np.stack([seqs[order[k]][at[k]:at[k] + n] for k in which])
            logits, _, _ = st.prefill_logits([ids[k] for k in which], [at[k] for k in which], toks, range(len(which) * n))
            w = np.concatenate([want[order[k]][at[k]:at[k] + n] for k in which])
            assert_logits(logits, w, dtype, f"turn {turn}, contexts {which}")
            for k in which:
                at[k] += n

        go([0], 40)
        go([1], 7)
        go([2, 3], 21)
        go([1, 2], 30)          # at positions 7 and 21
        for _ in range(12):
            logits = decode_step(st, ids, [seqs[order[k]][at[k]] for k in range(4)], at)
            w = np.stack([want[order[k]][at[k]] for k in range(4)])
            assert_logits(logits, w, dtype, f"turn {turn}, decoding at {at}")
            at = [a + 1 for a in at]
        go([3, 0, 2], 20)
        assert st.slot_counts() == dict(free=0, allocated=4, total=4)
        assert st.prefill_logits([99], [0], seqs[0][None, :3]) is None       # no slot left: nothing runs
        for i in ids:
            assert st.release_context(i)
    if paged:
        assert st.paging_info(0, 0)["clears"] >= 1
    # a context that starts again without being given back
    st.prefill_logits([77], [0], seqs[3][None, :50])
    logits, _, _ = st.prefill_logits([77], [0], seqs[1][None, :60], range(60))
    assert_logits(logits, want[1][:60], dtype)
    st.close()


@pytest.mark.parametrize("name", ["odd", "round"])
def test_tokens_out_of_order_are_refused(models, name):
    from glinthawk_amd._lib import GlintError
    path, cfg, _, seqs, want, _ = models(name)
    st = open_stage(path, "f32")
    st.prefill_logits([1], [0], seqs[0][None, :10])
    with pytest.raises(GlintError):
        st.prefill_logits([1], [12], seqs[0][None, 12:20])
    with pytest.raises(GlintError):
        decode_step(st, [1], [3], [9])
    with pytest.raises(GlintError):
        st.prefill_logits([2], [0], np.zeros((1, cfg["max_positions"] + 1), int))
    with pytest.raises(GlintError):
        decode_step(st, [1, 1], [3, 4], [10, 10])
    logits, _, _ = st.prefill_logits([1], [10], seqs[0][None, 10:20], range(10))       # and nothing of that has touched the context
    assert_logits(logits, want[0][10:20], "f32")
    st.close()


@pytest.mark.parametrize("dtype", DTYPES)
def test_long_decoding(models, dtype):
    """Decoding far beyond the window, the table of distances and the prompt, up to the last position the model has."""
    path, cfg, weights, _, _, _ = models("odd")
    T = cfg["max_positions"]
    seq = np.random.default_rng(5).integers(0, cfg["vocab"], T)
    want = P.forward(cfg, weights, seq)
    st = open_stage(path, dtype, 2)
    st.prefill_logits([4], [0], seq[None, :10])
    got = [decode_step(st, [4], [seq[i]], [i])[0] for i in range(10, T)]
    assert_logits(np.stack(got), want[10:], dtype)
    assert st.row(0)["finished"]
    st.close()


@pytest.mark.parametrize("name", ["odd", "round"])
def test_greedy_generation_through_the_compute_kernel(models, name):
    """The serving entry point: states pushed and popped as wire records, prompts fed token by token, then the sampled tokens; each row
    must get the tokens the plain implementation generates."""
    from glinthawk_amd import stage as S, wire
    from glinthawk_amd.kernel import ComputeKernel
    path, cfg, weights, seqs, _, _ = models(name)
    prompts = [list(map(int, seqs[0][:5])), list(map(int, seqs[1][:9])), list(map(int, seqs[2][:1]))]
    new = 12
    want = []
    for p in prompts:
        toks = list(p)
        for _ in range(new):
            toks.append(int(np.argmax(P.forward(cfg, weights, toks)[-1])))
        want.append(toks[len(p):])
    kernel = ComputeKernel(model_dir=path, dtype="f32", concurrency=3, max_contexts=3)
    rows = wire.new_prompts(3)
    rows["active"], rows["kv_tier"], rows["context_id"] = 1, 0, [21, 22, 23]
    rows["prompt_length"], rows["max_completion_length"] = [len(p) for p in prompts], new
    rows["token"] = [p[0] for p in prompts]
    got = [[] for _ in prompts]
    meta = dict(dtype=wire.DTYPE_CODE["f32"], next_layer=0, next_stage=S.STAGE_PRE)
    for _ in range(max(map(len, prompts)) + new + 2):
        if not rows["active"].any():
            break
        kernel.push(wire.pack_state(meta, rows))
        assert kernel.wait(30.0)
        kernel.read_event()
        _, rows, *_ = wire.unpack_state(kernel.pop(), 0, 0)
        for i, p in enumerate(prompts):
            if not rows["active"][i]:
                continue
            pos = int(rows["token_pos"][i])
            if pos < len(p):
                rows["token"][i] = p[pos]                    # still inside the prompt: the sampled token is not used
            else:
                got[i].append(int(rows["token"][i]))
                if len(got[i]) == new:
                    rows["active"][i] = 0
    assert got == want
    kernel.close()


def test_float32_weights_load_as_well(models, tmp_path):
    path, cfg, weights, seqs, want, _ = models("odd")
    st = open_stage(M.write_model(tmp_path / "f32", cfg, weights, dtype="F32"), "f32")
    assert_logits(st.prefill_logits([1], [0], seqs[0][None, :30], range(30))[0], want[0][:30], "f32")
    st.close()


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_trace_runner(models, tmp_path, dtype):
    path, cfg, _, seqs, want, _ = models("odd")
    steps = [
        {"step": 0, "entries": [{"id": "a", "tokens": seqs[0][:30].tolist(), "want": [0, 7, 29]}], "end": []},
        {"step": 1, "entries": [{"id": "b", "tokens": seqs[1][:2].tolist(), "want": []}], "end": []},
        {"step": 2, "entries": [{"id": "a", "tokens": [int(seqs[0][30])], "want": [0]}, {"id": "b", "tokens": [int(seqs[1][2])], "want": [0]}], "end": ["a"]},
        {"step": 5, "entries": [{"id": "b", "tokens": seqs[1][3:50].tolist(), "want": [46]}, {"id": "c", "tokens": [int(seqs[2][0])], "want": [0]}], "end": ["b", "c"]},
        {"step": 6, "entries": [{"id": "a", "tokens": seqs[3][:9].tolist(), "want": [8]}], "end": ["a"]},
    ]
    expect = {0: want[0][[0, 7, 29]], 2: np.stack([want[0][30], want[1][2]]), 5: np.stack([want[1][49], want[2][0]]), 6: want[3][8:9]}
    run = subprocess.run([os.path.join(ROOT, "bin", "trace_run"), "--model", path, "--dtype", dtype, "--out", str(tmp_path), "--max-tokens", "100"],
                         input="".join(json.dumps(s) + "\n" for s in steps), capture_output=True, text=True, timeout=110)
    assert run.returncode == 0, run.stderr
    assert [l for l in run.stdout.splitlines() if l.startswith("done")] == [f"done {s['step']}" for s in steps]
    for n, w in expect.items():
        got = np.fromfile(tmp_path / f"{n}.f32", np.float32).reshape(-1, cfg["vocab"])
        assert got.shape == w.shape
        assert_logits(got, w, "f32" if dtype == "float32" else "bf16", f"step {n}")
    assert not (tmp_path / "1.f32").exists()
