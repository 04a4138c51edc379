"""Bits of kernels whose order of sums models depend on.  A design whose layers feed each other for a thousand tokens turns a last bit into a difference of a
token's logits that can be far larger than that of any of its parts, so a faster kernel here keeps the order of its sums, and what is pinned are checksums of whole
outputs.  Inputs are whole numbers over powers of two from a generator of numpy's, and products in front of the kernel are exact in any order."""
import zlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def draw(rng, shape, spread=0, dtype="bfloat16"):
    """Up to seven significant bits, over `spread` + 1 powers of two."""
    import torch
    v = rng.integers(-127, 128, shape).astype(np.float32) / 64.0
    if spread:
        v = np.ldexp(v, -rng.integers(0, spread + 1, shape))
    return torch.from_numpy(v.astype(np.float32)).cuda().to(getattr(torch, dtype))


def checksum(*tensors):
    import torch
    c = 0
    for t in tensors:
        c = zlib.crc32(t.contiguous().view(torch.uint8).cpu().numpy().tobytes(), c)
    return c


MLSTM = {(3, 40, 8, 24, 65): 3122385930, (2, 64, 136, 33, 256): 1821903039, (4, 128, 72, 64, 300): 579374656, (2, 232, 200, 130, 127): 3581533614,
         (8, 256, 512, 1025, 64): 3581607802}


def mlstm_bits(H, d, dv, *cuts):
    """Two contexts and a slot without one, in two portions: outputs, then the state."""
    import torch
    from glinthawk_amd import ops
    from glinthawk_amd._lib import GhMlstm
    rng = np.random.default_rng(d + dv)
    m, width, B = GhMlstm(H, d, dv, 15.0, 1e-4), 8, 3
    rows, gate_row = ops.mlstm_weight_rows(m)
    w = rng.integers(-2, 3, (rows, width)) * np.where(np.arange(rows) >= gate_row, 0.5, 1.0)[:, None]
    w = torch.from_numpy(w.astype(np.float32)).cuda().bfloat16()
    x = torch.from_numpy(rng.integers(-1, 2, (B, sum(cuts), width)).astype(np.float32)).cuda().bfloat16()
    bias_i, bias_f, norm = draw(rng, H), draw(rng, H) + 3, draw(rng, H * dv) / 8 + 1
    state = torch.zeros((B, ops.mlstm_state_bytes(m) // 4), device="cuda")
    table, out, at = ops.row_table([0 if i == 1 else state[i].data_ptr() for i in range(B)]), [], 0
    for c in cuts:
        start = torch.full((B,), at, dtype=torch.int32, device="cuda")
        out.append(ops.mlstm_forward(x[:, at:at + c].reshape(B * c, width).contiguous(), w, m, bias_i, bias_f, norm, table, start, c))
        at += c
    return checksum(*out, state)


@pytest.mark.parametrize("shape", MLSTM)
def test_mlstm(shape):
    assert mlstm_bits(*shape) == MLSTM[shape]


# (heads, kv heads, head sizes, values are keys), (window, kept tokens, distances), tokens: no bias, one that ends before the keys do, one too long for room around it
WINDOW = {(4, 4, 128, 128, False, 0, 0, 0, 290): 322941296, (8, 2, 72, 40, False, 97, 5, 1, 131): 2589682963, (4, 4, 128, 128, False, 300, 4, 64, 700): 43964091,
          (4, 4, 128, 128, True, 0, 0, 90, 290): 2409675448, (2, 2, 96, 96, True, 64, 70, 17, 131): 4132586507, (6, 2, 128, 64, False, 31, 64, 7900, 131): 382486082}


def window_bits(heads, kv, dim, vdim, shared, window, keep, n_dist, T):
    """Two contexts, one of them with keys in front."""
    import torch
    from glinthawk_amd import ops
    rng = np.random.default_rng(dim + T)
    a, starts = ops.window_attn(heads, kv, dim, vdim, dim ** -0.5, window, keep, n_dist, shared), [0, 77]
    keys = max(starts) + T
    cache, factors = draw(rng, (2, keys, kv * (dim if shared else dim + vdim)), 2), draw(rng, (2, -(-keys // 32) * kv * 32), 0, "float32") / 4 + 1
    memory = torch.cat([cache.view(2, -1).view(torch.uint8), factors.view(torch.uint8)], 1).contiguous()
    bias = draw(rng, (heads, n_dist), 2, "float32") if n_dist else None
    return checksum(ops.attn_window(draw(rng, (2 * T, heads * dim), 2), a, ops.row_table([m.data_ptr() for m in memory]), torch.tensor(starts, dtype=torch.int32, device="cuda"), T,
                                    max(starts), bias, 0, cache[0].numel() * 2))


@pytest.mark.parametrize("shape", WINDOW)
def test_window_attention(shape):
    assert window_bits(*shape) == WINDOW[shape]


# (k, activation rows, weight rows): work-groups whose waves get one piece of 64 k or two, some of them one more or none; one tile of weight rows and two
FEW_ROWS = {(256, 200, 8): 1210123369, (768, 225, 17): 3488112410, (1280, 333, 32): 1850897936, (512, 193, 1): 827850632, (4096, 1000, 16): 916273720}


def few_rows_bits(s, b, r):
    from glinthawk_amd import ops
    rng = np.random.default_rng(s + b)
    return checksum(ops.matmul_scaled(draw(rng, (b, s), 6), draw(rng, (r, s), 6), 0.5))


@pytest.mark.parametrize("shape", FEW_ROWS)
def test_product_of_few_weight_rows(shape):
    assert few_rows_bits(*shape) == FEW_ROWS[shape]


# (heads, kv heads, head sizes), tokens: a work-group for each, rows that end inside a group of threads, padded heads; long rows of many tokens, several a work-group
APPEND = {(32, 32, 128, 128, 521): 3915238599, (40, 8, 128, 64, 700): 3069143961, (25, 5, 104, 72, 900): 2630354648, (60, 20, 52, 36, 611): 3883644428,
          (4, 4, 64, 64, 1000): 1073606430, (32, 32, 128, 128, 1100): 1240766657, (64, 16, 128, 40, 1301): 2555571595}


def append_bits(heads, kv, d, dv, T):
    """q, then what two contexts were appended; the tokens of a third one are passed over."""
    import torch
    from glinthawk_amd import ops
    rng = np.random.default_rng(heads + T)
    a, n = ops.window_attn(heads, kv, d, dv, 1.0, 9, 2, 5), heads * d + kv * (d + dv)
    x, w = (torch.from_numpy(rng.integers(-3, 4, s).astype(np.float32)).cuda().bfloat16() for s in ((3 * T, 16), (n, 16)))     # products below 256: exact
    b, qn, kn = draw(rng, n, 3), draw(rng, heads * d, 2) / 4 + 1, draw(rng, kv * d, 2) / 4 + 1
    region = [torch.zeros((T + 11, ops.window_row_bytes(a, torch.bfloat16) // 2), dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    table, start = ops.row_table([region[0].data_ptr(), 0, region[1].data_ptr()]), torch.tensor([3, 0, 11], dtype=torch.int32, device="cuda")
    return checksum(ops.matmul_window_append(x, w, a, table, start, T, b, qn, kn, 2e-3), *region)


@pytest.mark.parametrize("shape", APPEND)
def test_query_key_norm_and_append(shape):
    assert append_bits(*shape) == APPEND[shape]


# rows, width, dtype, a norm behind the product: a thread for each group of columns with work-groups beyond those in flight, and few rows; more groups a thread
STEP = {(700, 4096, "bfloat16", True): 3824987965, (999, 4096, "bfloat16", False): 2599642962, (33, 4096, "bfloat16", True): 1377173294,
        (1300, 2048, "bfloat16", True): 3409561444, (600, 1024, "float32", True): 706433486, (1100, 4096, "float32", True): 3856038900}


def step_bits(rows, width, dtype, post):
    """The residual stream, then the normed rows."""
    import torch
    from glinthawk_amd import ops
    rng = np.random.default_rng(rows)
    inp, w = (torch.from_numpy(rng.integers(-3, 4, s).astype(np.float32)).cuda().to(getattr(torch, dtype)) for s in ((rows, 16), (width, 16)))
    x, bias, norms = draw(rng, (rows, width), 9, "float32"), draw(rng, width, 3, dtype), [draw(rng, width, 2, dtype) / 4 + 1 for _ in range(2)]
    out = torch.empty((rows, width), dtype=inp.dtype, device="cuda")
    ops.matmul_stream(x, inp, w, 1e-4, bias=bias, post_norm=norms[0] if post else None, next_norm=norms[1], out=out)
    return checksum(x, out)


@pytest.mark.parametrize("shape", STEP)
def test_residual_step(shape):
    assert step_bits(*shape) == STEP[shape]


# heads, head sizes, contexts, dtype: tokens one after the other
MLSTM_STEP = {(4, 16, 512, 300, "bfloat16"): 9421239, (4, 16, 512, 300, "float32"): 2747313704, (2, 24, 1024, 150, "bfloat16"): 2003180597, (3, 16, 40, 500, "float32"): 1522406068}


def mlstm_step_bits(H, d, dv, B, dtype):
    """Three tokens of every context: outputs, then the state."""
    import torch
    from glinthawk_amd import ops
    from glinthawk_amd._lib import GhMlstm
    rng, dt = np.random.default_rng(d + dv), getattr(torch, dtype)
    m, width = GhMlstm(H, d, dv, 15.0, 1e-4), 8
    rows, gate_row = ops.mlstm_weight_rows(m)
    w = rng.integers(-2, 3, (rows, width)) * np.where(np.arange(rows) >= gate_row, 0.5, 1.0)[:, None]
    w, x = torch.from_numpy(w.astype(np.float32)).cuda().to(dt), torch.from_numpy(rng.integers(-1, 2, (3, B, width)).astype(np.float32)).cuda().to(dt)
    bias_i, bias_f, norm = draw(rng, H, 0, dtype), draw(rng, H, 0, dtype) + 3, draw(rng, H * dv, 0, dtype) / 8 + 1
    state = torch.zeros((B, ops.mlstm_state_bytes(m) // 4), device="cuda")
    table = ops.row_table([s.data_ptr() for s in state])
    out = [ops.mlstm_forward(x[t], w, m, bias_i, bias_f, norm, table, torch.full((B,), t, dtype=torch.int32, device="cuda"), 1) for t in range(3)]
    return checksum(*out, state)


@pytest.mark.parametrize("shape", MLSTM_STEP)
def test_mlstm_step(shape):
    assert mlstm_step_bits(*shape) == MLSTM_STEP[shape]


# heads, key heads, tokens of a context, width: columns that overflow whole rounds of tiles by the heads' gates, with a ragged last tile; few rows
PARALLEL = {(32, 32, 4096, 2048): 1705321414, (32, 32, 667, 4096): 3510089885, (28, 4, 8150, 512): 498023561, (5, 5, 40, 256): 483779571}


def parallel_bits(heads, kv, T, width):
    """Queries, gates and what two contexts were appended, the tokens of a third one passed over; products are exact in any order."""
    import torch
    from glinthawk_amd import ops
    rng, d, keys = np.random.default_rng(heads + T), 128, -(-T // 32) * 32
    a = ops.window_attn(heads, kv, d, d, 1.0, values_are_keys=True)
    n, _ = ops.parallel_weight_rows(a, True, 0)
    x, w = (torch.from_numpy(rng.integers(-3, 4, s).astype(np.float32)).cuda().bfloat16() for s in ((3 * T, width), (n, width)))
    at = keys * kv * d * 2
    region = [torch.zeros(at + keys * kv * 4, dtype=torch.uint8, device="cuda") for _ in range(2)]
    start = torch.zeros(3, dtype=torch.int32, device="cuda")
    q, gates = ops.matmul_parallel(x, w / 64, a, ops.row_table([region[0].data_ptr(), 0, region[1].data_ptr()]), start, T, 1e-3, 0.1, 512, True, None, factor_offset=at)
    return checksum(q, gates, *region)


@pytest.mark.parametrize("shape", PARALLEL)
def test_heads_of_a_parallel_layer(shape):
    assert parallel_bits(*shape) == PARALLEL[shape]
