"""Projections fused with their follow-up ops against the same ops issued one by one (bit-exact where
the arithmetic is element-wise, tolerance where a reduction order differs) and against the oracle."""
import ctypes

import numpy as np
import pytest
import torch

import oracle as O
from glinthawk_amd import Shape, _lib, ops, stage as S
from helpers import Arena, assert_close, assert_half_parity, oracle_cfg
from test_gpu_stage import SHAPES, OracleModel, d2h, load_weights, make_weights

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    ops.init(0)


@pytest.mark.parametrize("dt", [torch.float16, torch.float32])
@pytest.mark.parametrize("b,s,r", [(4, 288, 288), (1, 288, 288), (1, 260, 4100), (64, 1024, 512), (5, 768, 1000), (3, 100, 36),
                                   # more than 64 rows: any of the kernels leaves the partial sums
                                   (100, 512, 260), (256, 1024, 512), (300, 4096, 1000),
                                   # enough 256-token tiles: the residual is added in the large tile kernel's epilogue (f16, r % 8 == 0)
                                   (768, 8192, 16384), (2048, 512, 6152), (3000, 1024, 6144), (2300, 512, 8192),
                                   (2048, 512, 6150)])          # r % 8 != 0: fp32 partials and the row kernel
def test_matmul_accum_and_norm(dt, b, s, r, product_route):
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn((b, s), generator=g, device="cuda").to(dt)
    w = (torch.randn((r, s), generator=g, device="cuda") / s ** 0.5).to(dt)
    res = torch.randn((b, r), generator=g, device="cuda").to(dt)
    nw = (1 + 0.1 * torch.randn(r, generator=g, device="cuda")).to(dt)
    # separate ops
    want_res = res.clone()
    ops.accum(want_res, ops.matmul(x, w))
    want_norm = ops.rmsnorm(want_res, nw)
    # fused, without and with the norm
    got_res = res.clone()
    assert ops.matmul_accum(got_res, x, w) is None
    assert torch.equal(got_res, want_res)
    got_res2 = res.clone()
    got_norm = ops.matmul_accum(got_res2, x, w, nw)
    assert torch.equal(got_res2, want_res)
    tol = 2e-3 if dt == torch.float16 else 3e-6
    assert torch.allclose(got_norm.float(), want_norm.float(), rtol=tol, atol=tol)
    # and against the oracle's fp32 path
    o_res = res.float().cpu().numpy()
    O.accum(o_res, O.matmul(x.float().cpu().numpy(), w.float().cpu().numpy()))
    assert_close(got_norm.float().cpu().numpy(), O.rmsnorm(o_res, nw.float().cpu().numpy()), what="fused accum+rmsnorm")
    # the plain product of the separate ops and the product inside each of the two fused calls
    product_route.check(3 if dt == torch.float16 and product_route.wanted(b, s, r) else 0)


@pytest.mark.parametrize("dt", [torch.float16, torch.float32])
@pytest.mark.parametrize("b,s,r", [(4, 288, 288), (3, 100, 37), (70, 512, 1000),
                                   (2048, 512, 6152)])          # f16: enough tiles for the residual add in the tile kernel's epilogue
@pytest.mark.parametrize("at", ["residual", "norm_out", "norm_weight"])
def test_matmul_accum_norm_of_unaligned_rows(dt, b, s, r, at):
    """A buffer that starts one element past a 16-byte boundary gives what aligned ones give, up to the order of the norm's sum."""
    g = torch.Generator(device="cuda").manual_seed(7)
    x = torch.randn((b, s), generator=g, device="cuda").to(dt)
    w = (torch.randn((r, s), generator=g, device="cuda") / s ** 0.5).to(dt)
    res = torch.randn((b, r), generator=g, device="cuda").to(dt)
    nw = (1 + 0.1 * torch.randn(r, generator=g, device="cuda")).to(dt)

    def place(t, shifted):
        buffer = torch.zeros(t.numel() + 1, dtype=dt, device="cuda")
        view = buffer[1:] if shifted else buffer[:-1]
        return view.view(t.shape).copy_(t)

    want_res = res.clone()
    want_norm = ops.matmul_accum(want_res, x, w, nw)
    got_res, got_norm, weight = place(res, at == "residual"), place(torch.zeros_like(res), at == "norm_out"), place(nw, at == "norm_weight")
    _lib.check(_lib.lib().gh_matmul_accum(ops._p(got_res), ops._p(x), ops._p(w), s, r, b, ops._p(got_norm), ops._p(weight), ops._dt(x), ops._stream()))
    tol = 2e-3 if dt == torch.float16 else 3e-6
    assert torch.allclose(got_res.float(), want_res.float(), rtol=tol, atol=tol)
    assert torch.allclose(got_norm.float(), want_norm.float(), rtol=tol, atol=tol)


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("b,s", [(3, 512), (70, 1024), (300, 4096)])
def test_outputs_over_their_activations(dt, b, s):
    """An output buffer that lies over the activations gives what one of its own gives (the order of fp32 sums may differ: a rounding)."""
    if dt != torch.float32 and b == 300:
        b = 2304                                        # enough tiles for the epilogues of the large tile kernel
    g = torch.Generator(device="cuda").manual_seed(b)
    x = torch.randn((b, s), generator=g, device="cuda").to(dt)
    w = (torch.randn((3 * s, s), generator=g, device="cuda") / s ** 0.5).to(dt)
    tol = dict(rtol=1e-5, atol=1e-5) if dt == torch.float32 else dict(rtol=2e-2, atol=2e-2) if dt == torch.bfloat16 else dict(rtol=4e-3, atol=4e-3)
    lib, p, shape, st = _lib.lib(), ops._p, Shape(dim=s, n_layers=1, n_heads=s // 64, n_kv_heads=s // 64, hidden_dim=s, seq_len=8), ops._stream()
    half = w[:s].contiguous()                           # w1 and w3 of half as many rows
    got, spare = x.clone(), torch.empty((b, s // 2), dtype=dt, device="cuda")
    if dt == torch.bfloat16:
        _lib.check(lib.gh_matmul_gate(p(spare), p(x), p(half), None, s, s // 2, b, ops.GH_ACT_SILU, ops._dt(x), st))
        _lib.check(lib.gh_matmul_gate(p(got), p(got), p(half), None, s, s // 2, b, ops.GH_ACT_SILU, ops._dt(x), st))
        assert torch.allclose(got.flatten()[: spare.numel()].float(), spare.flatten().float(), **tol)
        return
    _lib.check(lib.gh_matmul_silu_gate(p(spare), p(x), p(half), s, s // 2, b, ops._dt(x), st))
    _lib.check(lib.gh_matmul_silu_gate(p(got), p(got), p(half), s, s // 2, b, ops._dt(x), st))
    assert torch.allclose(got.flatten()[: spare.numel()].float(), spare.flatten().float(), **tol)
    residual, got = x.clone(), x.clone()
    ops.matmul_accum(residual, x, half)
    _lib.check(lib.gh_matmul_accum(p(got), p(got), p(half), s, s, b, None, None, ops._dt(x), st))
    assert torch.allclose(got.float(), residual.float(), **tol)
    pos = torch.arange(b, dtype=torch.int32, device="cuda") % 8
    re, im = (torch.randn((8, 32), generator=g, device="cuda").to(dt) for _ in range(2))
    cache, over = (torch.zeros((b, 2 * s), dtype=dt, device="cuda") for _ in range(2))
    q, _ = ops.matmul_qkv_rope_append(x, w, pos, re, im, ops.row_table([cache[i].data_ptr() for i in range(b)]), shape)
    got = x.clone()
    _lib.check(lib.gh_matmul_qkv_rope_append(p(got), None, p(got), p(w), s, b, p(pos), p(re), p(im), p(ops.row_table([over[i].data_ptr() for i in range(b)])),
                                             shape.n_kv_heads, shape.gqa_size, shape.head_size, ops._dt(x), st))
    assert torch.allclose(got.float(), q.float(), **tol) and torch.allclose(over.float(), cache.float(), **tol)


@pytest.mark.parametrize("b,s,r", [(2080, 1024, 8192), (3080, 2048, 5120)])
def test_norm_over_activations_of_shorter_rows(b, s, r):
    """The norm's rows in the buffer of the activations, whose rows are shorter, where the product is better run in two parts along the tokens: norms
    of the first must not land on activations of the second.  The parts may sum in another order: a rounding of f16."""
    g = torch.Generator(device="cuda").manual_seed(b)
    x = torch.randn((b, s), generator=g, device="cuda").half()
    w = (torch.randn((r, s), generator=g, device="cuda") / s ** 0.5).half()
    res = torch.randn((b, r), generator=g, device="cuda").half()
    nw = (1 + 0.1 * torch.randn(r, generator=g, device="cuda")).half()
    want_res = res.clone()
    want_norm = ops.matmul_accum(want_res, x, w, nw)
    both = torch.empty((b, r), dtype=torch.float16, device="cuda")
    both.flatten()[: x.numel()] = x.flatten()
    _lib.check(_lib.lib().gh_matmul_accum(ops._p(res), ops._p(both), ops._p(w), s, r, b, ops._p(both), ops._p(nw), ops._dt(x), ops._stream()))
    assert torch.allclose(res.float(), want_res.float(), rtol=4e-3, atol=4e-3)
    assert torch.allclose(both.float(), want_norm.float(), rtol=4e-3, atol=4e-3)


# rows that a wave requests in one go (the norm in the product's launch): one piece and a bit, the most that two and four weight rows a wave leave
# room for, and one element more; s % 4 != 0; f16: two launches
@pytest.mark.parametrize("dt,s", [(torch.float32, 4), (torch.float32, 256), (torch.float32, 288), (torch.float32, 512), (torch.float32, 516), (torch.float32, 1024),
                                  (torch.float32, 1028), (torch.float32, 290), (torch.float16, 288)])
@pytest.mark.parametrize("b", [1, 2, 4, 5, 9, 17, 67])
def test_products_of_normed_rows(dt, s, b):
    """Against 64 bits.  fp32: an element of the normed row is off by some 4 roundings of 2^-24, and the sum of s products by at most s of them, of the sum
    of magnitudes; f16: the rounding of the normed row, 2^-11 of the magnitudes, and of the result."""
    g = torch.Generator(device="cuda").manual_seed(s * 31 + b)
    shape = Shape(dim=48, n_layers=1, n_heads=6, n_kv_heads=2, hidden_dim=s, seq_len=8)
    x = (3 * torch.randn((b, s), generator=g, device="cuda")).to(dt)
    nw = (1 + 0.1 * torch.randn(s, generator=g, device="cuda")).to(dt)
    normed = x.double() / torch.sqrt((x.double() ** 2).mean(-1, keepdim=True) + 1e-5) * nw.double()
    unit = (s + 8) * 2.0 ** -24 if dt == torch.float32 else 2.0 ** -10

    def bound(w):
        return unit * (normed.abs() @ w.double().abs().T) + 2.0 ** (-24 if dt == torch.float32 else -11) * (normed @ w.double().T).abs() + 1e-6

    for r in (1, 37, 4096, 4100):
        w = (torch.randn((r, s), generator=g, device="cuda") / s ** 0.5).to(dt)
        got = ops.rmsnorm_matmul(x, nw, w)
        assert ((got.double() - normed @ w.double().T).abs() <= bound(w)).all()
    for hidden in (3, 768, 2050):
        w = (torch.randn((2 * hidden, s), generator=g, device="cuda") / s ** 0.5).to(dt)
        y = normed @ w.double().T
        y1, y3, slack = y[:, :hidden], y[:, hidden:], bound(w)
        got = ops.rmsnorm_matmul_silu_gate(x, nw, w).double()
        # the gate's slope in y1 is at most 1.1 |y3|; the fast exponential and the rounding of the factors and the result on top
        want = y1 * torch.sigmoid(y1) * y3
        rounding = 2e-6 if dt == torch.float32 else 2.0 ** -9
        assert ((got - want).abs() <= 1.1 * slack[:, :hidden] * y3.abs() + slack[:, hidden:] * y1.abs() + rounding * (1 + want.abs())).all()
    w = (torch.randn((80, s), generator=g, device="cuda") / s ** 0.5).to(dt)
    pos = torch.arange(b, dtype=torch.int32, device="cuda") % 8
    angle = torch.rand((8, 4), generator=g, device="cuda") * 6
    re, im = torch.cos(angle).to(dt), torch.sin(angle).to(dt)
    caches = [torch.full((b, 32), 5.0, dtype=dt, device="cuda") for _ in range(2)]
    rows = [ops.row_table([0 if i == 1 else c[i].data_ptr() for i in range(b)]) for c in caches]
    got = ops.rmsnorm_matmul_qkv_rope_append(x, nw, w, pos, re, im, rows[0], shape)
    want, _ = ops.matmul_qkv_rope_append(ops.rmsnorm(x, nw), w, pos, re, im, rows[1], shape)
    tol = dict(rtol=1e-5, atol=1e-5) if dt == torch.float32 else dict(rtol=4e-3, atol=4e-3)     # another order of the norm's sum; a rotation adds two products
    assert torch.allclose(got.float(), want.float(), **tol) and torch.allclose(caches[0].float(), caches[1].float(), **tol)


def test_norm_over_the_rows_it_reads():
    """An output that lies over the activations, and weights or rows that start off a 16-byte boundary, go through two launches: the same values."""
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn((4, 288), generator=g, device="cuda")
    nw, w = 1 + 0.1 * torch.randn(288, generator=g, device="cuda"), torch.randn((288, 288), generator=g, device="cuda") / 17
    want, lib, p, st = ops.rmsnorm_matmul(x, nw, w), _lib.lib(), ops._p, ops._stream()
    got = x.clone()
    _lib.check(lib.gh_rmsnorm_matmul(p(got), p(got), p(nw), p(w), 288, 288, 4, ops._dt(x), st))
    assert torch.allclose(got, want, rtol=1e-5, atol=1e-5)
    shifted = torch.empty(w.numel() + 1, device="cuda")[1:].view(288, 288).copy_(w)
    _lib.check(lib.gh_rmsnorm_matmul(p(got), p(x), p(nw), p(shifted), 288, 288, 4, ops._dt(x), st))
    assert torch.allclose(got, want, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dt", [torch.float16, torch.float32])
@pytest.mark.parametrize("b,s,hidden", [(4, 288, 768), (1, 288, 768), (1, 260, 2050), (64, 512, 1536), (3, 100, 50), (130, 512, 1536), (512, 8192, 12544),
                                        # enough row tiles for one launch without a K split: both factors in one kernel
                                        (64, 512, 16384), (5, 256, 16404), (33, 1024, 28672),
                                        (5, 256, 16386)])     # rows not a multiple of 4: the two-kernel route
def test_matmul_silu_gate(dt, b, s, hidden, product_route):
    check_matmul_silu_gate(dt, b, s, hidden, product_route)


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("b,s,hidden", [(64, 512, 16384), (5, 256, 16404), (33, 1024, 28672), (64, 8192, 3584), (17, 768, 16500)])
def test_matmul_silu_gate_one_launch_with_four_and_eight_waves(waves, b, s, hidden, product_route):
    """The one-launch form (w1 and w3 rows of the same outputs in one work-group, gate in the epilogue) with work-groups of four
    and of eight waves, whichever the library would pick for the shape: row counts that leave the last work-group and the last
    wave partly empty, few and many columns."""
    _lib.check(_lib.lib().gh_gemm_set_gate_waves(waves))
    try:
        check_matmul_silu_gate(torch.float16, b, s, hidden, product_route)
    finally:
        _lib.check(_lib.lib().gh_gemm_set_gate_waves(0))


@pytest.mark.parametrize("b,s,hidden", [(65, 1024, 2816), (77, 2048, 5632), (96, 3072, 8192), (77, 4096, 11008), (65, 6656, 17920), (224, 1024, 2816)])
def test_silu_gate_stays_in_the_product_where_that_is_faster(b, s, hidden):
    """Shapes at which the ring kernel with the gate was timed 7 to 25 % faster than a K split with the gate behind it: the default gives the ring
    kernel's bits, which a K range summed in parts would not."""
    g = torch.Generator(device="cuda").manual_seed(b)
    x = torch.randn((b, s), generator=g, device="cuda").half()
    w13 = (torch.randn((2 * hidden, s), generator=g, device="cuda") / s ** 0.5).half()
    got = ops.matmul_silu_gate(x, w13)
    _lib.check(_lib.lib().gh_gemm_set_tuning(5, 0, 0))
    try:
        assert torch.equal(got, ops.matmul_silu_gate(x, w13))
    finally:
        _lib.check(_lib.lib().gh_gemm_set_tuning(0, 0, 0))


def check_matmul_silu_gate(dt, b, s, hidden, product_route):
    g = torch.Generator(device="cuda").manual_seed(2)
    x = torch.randn((b, s), generator=g, device="cuda").to(dt)
    w13 = (torch.randn((2 * hidden, s), generator=g, device="cuda") / s ** 0.5).to(dt)
    hb = ops.matmul(x, w13[:hidden].contiguous())
    hb2 = ops.matmul(x, w13[hidden:].contiguous())
    ops.silu(hb, hb2)
    got = ops.matmul_silu_gate(x, w13)
    # the fused call multiplies one (2*hidden, s) matrix and may split K differently from the two
    # separate calls, so the fp32 sums can differ in the last bit before rounding
    tol = 2e-3 if dt == torch.float16 else 2e-6
    assert torch.allclose(got.float(), hb.float(), rtol=tol, atol=tol)
    if b * hidden * s <= 64 * 512 * 16384:
        xh, wh = x.float().cpu().numpy(), w13.float().cpu().numpy()
        want = O.matmul(xh, np.ascontiguousarray(wh[:hidden]))
        O.silu(want, O.matmul(xh, np.ascontiguousarray(wh[hidden:])))
        assert_close(got.float().cpu().numpy(), want, what="fused w1, w3, silu")
    # some hundred rows and a wide [w1; w3]: one product of the vendor library, then the gate over the two halves of each row
    wide = dt == torch.float16 and 128 <= b < product_route.ROWS and 2 * hidden >= 16384 and s % 8 == 0 and hidden % 8 == 0
    plain = 2 if dt == torch.float16 and product_route.wanted(b, s, hidden) else 0        # the two separate products above
    product_route.check(plain + (1 if wide else 0))


# the gate in the product's own epilogue: whole 256 x 256 tiles that leave whole and ragged, walked and not, an odd number of steps, a rest
# of tokens on the ring kernel, and the ring kernel alone with ragged rows and columns
@pytest.mark.parametrize("activation", [ops.GH_ACT_SILU, ops.GH_ACT_GELU_TANH])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("b,s,hidden", [(4096, 256, 8192), (2300, 576, 4104), (2100, 640, 6152), (300, 4096, 12544), (77, 520, 2052), (200, 512, 16404), (5, 4096, 11008)])
def test_matmul_gate_in_epilogue(b, s, hidden, bias, activation):
    """Against 64 bits, bf16.  The gate works on the fp32 sums: one rounding, off by 2^-8 of the result, and 1e-4 for the sums and the fast
    exponential.  From 192 rows on the tanh gate and biases are a kernel of their own over rounded factors: off by 2^-8 of the plain product
    each, which reaches the output times the other factor (and times the activation's slope, at most 1.13), 1 % for the second order."""
    g = torch.Generator(device="cuda").manual_seed(b + hidden)
    x = torch.randn((b, s), generator=g, device="cuda").bfloat16()
    w = (torch.randn((2 * hidden, s), generator=g, device="cuda") / s ** 0.5).bfloat16()
    add = torch.randn(2 * hidden, generator=g, device="cuda").bfloat16() if bias else None
    got = ops.matmul_gate(x, w, add, activation).double()
    raw = x.double() @ w.double().t()
    y = raw + (add.double() if bias else 0.0)
    a, u = y[:, :hidden], y[:, hidden:]
    act = a * torch.sigmoid(a) if activation == ops.GH_ACT_SILU else torch.nn.functional.gelu(a, approximate="tanh")
    bound = 2.0 ** -8 * (act * u).abs() + 1e-4
    if b >= 192 and (bias or activation != ops.GH_ACT_SILU):
        bound = 1.01 * (bound + 2.0 ** -8 * (1.13 * (raw[:, :hidden] * u).abs() + (act * raw[:, hidden:]).abs())) + 1e-3
    assert ((got - act * u).abs() <= bound).all()


# tiles that walk over row tiles and token tiles, whole and ragged; a work-group each; an odd number of steps
@pytest.mark.parametrize("activation", [ops.GH_ACT_SILU, ops.GH_ACT_GELU_TANH])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("b,s,hidden", [(4096, 256, 8192), (4100, 256, 8200), (2304, 640, 8192), (2300, 576, 8200), (512, 128, 16384)])
def test_matmul_gate_of_whole_tiles(b, s, hidden, bias, activation):
    """The gate with tanh or biases in the tiles' epilogue, against 64 bits: on the fp32 sums, one rounding to bf16, off by 2^-8 of the result, and 1e-4 for the
    sums and the fast exponential.  Each bias once in a thousand is far off the rest, so that a wrong row's would show."""
    if activation == ops.GH_ACT_SILU and not bias:
        pytest.skip("the plain gate")
    g = torch.Generator(device="cuda").manual_seed(b + hidden)
    x = torch.randn((b, s), generator=g, device="cuda").bfloat16()
    w = (torch.randn((2 * hidden, s), generator=g, device="cuda") / s ** 0.5).bfloat16()
    add = torch.randn(2 * hidden, generator=g, device="cuda") if bias else None
    if bias:
        add[::997] += 20.0
        add = add.bfloat16()
    lib = _lib.lib()
    _lib.check(lib.gh_gemm_set_tuning(4, 0, 0))
    try:
        got = ops.matmul_gate(x, w, add, activation).double()
    finally:
        _lib.check(lib.gh_gemm_set_tuning(0, 0, 0))
    y = x.double() @ w.double().t() + (add.double() if bias else 0.0)
    a, u = y[:, :hidden], y[:, hidden:]
    want = (a * torch.sigmoid(a) if activation == ops.GH_ACT_SILU else torch.nn.functional.gelu(a, approximate="tanh")) * u
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4 * (1.0 + want.abs().sqrt())).all()


# 512 rows: the tiles' epilogues whole and with a ragged last tile; 16: the ring kernel
@pytest.mark.parametrize("b,hidden", [(512, 16384), (500, 16280), (16, 16384)])
@pytest.mark.parametrize("dt,activation,bias", [(torch.float16, ops.GH_ACT_SILU, False), (torch.bfloat16, ops.GH_ACT_SILU, False), (torch.bfloat16, ops.GH_ACT_SILU, True),
                                                (torch.bfloat16, ops.GH_ACT_GELU_TANH, False)])
def test_gate_of_large_and_small_factors(dt, activation, bias, b, hidden):
    """Factors that are one weight each, so that the sums are exact: over the range of the exponential, signed zeros, the type's smallest and largest,
    infinities and NaN, against 64 bits.  One rounding to the type, and the exponent's own, 2^-23 of its 127 at most; below 2^-119 (f16: its smallest) nothing is asked
    but the size: from a divisor of 2^126 on, at factors of -87.3 and less, the reciprocal may be 0, and the quotient is at most 88.8 * 2^-126."""
    lim = torch.finfo(dt)
    a = torch.cat([torch.linspace(-130.0, 130.0, 521), torch.tensor([0.0, -0.0, lim.tiny, -lim.tiny, lim.max, lim.min, float("inf"), -float("inf"), float("nan")]),
                   torch.logspace(-6, 4, 101), -torch.logspace(-6, 4, 101)]).to(dt).cuda()
    u = torch.tensor([1.0, -0.75, 1.5e-3], device="cuda").to(dt)
    w = torch.zeros((2 * hidden, 128), device="cuda", dtype=dt)
    n = torch.arange(hidden, device="cuda")
    w[:hidden, 0], w[hidden:, 0] = a[n % len(a)], u[n // len(a) % len(u)]
    x = torch.zeros((b, 128), device="cuda", dtype=dt)
    x[:, 0] = 1.0
    lib = _lib.lib()
    _lib.check(lib.gh_gemm_set_tuning(4 if b > 16 else 5, 0, 0))
    try:
        if dt == torch.float16:
            got = ops.matmul_silu_gate(x, w).double()
        else:
            got = ops.matmul_gate(x, w, torch.zeros(2 * hidden, device="cuda", dtype=dt) if bias else None, activation).double()
    finally:
        _lib.check(lib.gh_gemm_set_tuning(0, 0, 0))
    y, f = w[:hidden, 0].double(), w[hidden:, 0].double()
    z = y if activation == ops.GH_ACT_SILU else 2 * 0.7978845608028654 * (y + 0.044715 * y ** 3)
    exact = y / (1.0 + torch.exp(-z)) * f
    for row in (got[0], got[-1]):
        finite = exact.isfinite() & (exact.abs() <= lim.max)
        assert torch.equal(row.isnan(), exact.isnan())
        assert torch.equal(row[exact.isinf()], exact[exact.isinf()])
        eps = (2.0 ** -11 if dt == torch.float16 else 2.0 ** -8) + 127 * 2.0 ** -23 + (3 * 2.0 ** -23 * z.abs().clamp(max=130.0))
        small = lim.tiny * 2.0 ** -10 if dt == torch.float16 else 2.0 ** -119
        assert ((row - exact).abs() <= eps * exact.abs() + small)[finite].all()


# whole tiles and a ragged last one; the ring kernel
@pytest.mark.parametrize("b,hidden,kernel", [(512, 16384, 4), (500, 16280, 4), (16, 16384, 5)])
def test_gate_of_vanishing_factors(b, hidden, kernel):
    """bf16, factors between -128 ln 2, where the divisor overflows, and -126 ln 2, from where on it has no normal reciprocal: against 64 bits, one rounding to the type
    and the exponent's own."""
    w, x = torch.zeros((2 * hidden, 128), device="cuda", dtype=torch.bfloat16), torch.zeros((b, 128), device="cuda", dtype=torch.bfloat16)
    y, f = torch.tensor([-87.0, -87.5, -88.0, -88.5], device="cuda"), torch.tensor([1.0, -0.75, 4.0], device="cuda")
    n = torch.arange(hidden, device="cuda")
    w[:hidden, 0], w[hidden:, 0], x[:, 0] = y[n % 4].bfloat16(), f[n // 4 % 3].bfloat16(), 1.0
    lib = _lib.lib()
    _lib.check(lib.gh_gemm_set_tuning(kernel, 0, 0))
    try:
        got = ops.matmul_gate(x, w, None, ops.GH_ACT_SILU).double()
    finally:
        _lib.check(lib.gh_gemm_set_tuning(0, 0, 0))
    y, f = w[:hidden, 0].double(), w[hidden:, 0].double()
    want = y / (1.0 + torch.exp(-y)) * f
    assert ((got - want).abs() <= (2.0 ** -8 + 2.0 ** -14) * want.abs()).all()


@pytest.mark.parametrize("b,hidden", [(512, 16384), (500, 16280)])
def test_gate_of_tiles_and_of_stored_factors(b, hidden):
    """f16: the product of gate and factor is rounded as every other route rounds it, to the bit.  A sum is one product of two values here, so the factors are known.  Of
    these outputs 6.4e-5 are not the correctly rounded ones, with v_fma_mixlo_f16 in the place of a multiplication and a conversion 8.4e-5."""
    g = torch.Generator(device="cuda").manual_seed(b)
    w, x = torch.zeros((2 * hidden, 128), device="cuda", dtype=torch.float16), torch.zeros((b, 128), device="cuda", dtype=torch.float16)
    w[:, 0], x[:, 0] = torch.randn(2 * hidden, generator=g, device="cuda").half(), torch.randn(b, generator=g, device="cuda").half() * 2
    factors = (x[:, :1].float() * w[:, 0].float()).half()
    want = factors[:, :hidden].contiguous()
    ops.silu(want, factors[:, hidden:].contiguous())
    lib = _lib.lib()
    _lib.check(lib.gh_gemm_set_tuning(4, 0, 0))
    try:
        got = ops.matmul_silu_gate(x, w)
    finally:
        _lib.check(lib.gh_gemm_set_tuning(0, 0, 0))
    assert torch.equal(got, want)


@pytest.mark.parametrize("dt", [torch.float16, torch.float32])
@pytest.mark.parametrize("shape", [Shape(dim=32, n_layers=1, n_heads=4, n_kv_heads=2, hidden_dim=48, seq_len=16),
                                   Shape(dim=288, n_layers=1, n_heads=6, n_kv_heads=6, hidden_dim=768, seq_len=256),
                                   Shape(dim=1024, n_layers=1, n_heads=8, n_kv_heads=2, hidden_dim=64, seq_len=320)],
                         ids=["tiny", "stories15m", "gqa4"])
def test_matmul_qkv_rope_append(dt, shape):
    batch = 5
    arena_a = Arena(shape, batch, dt, seed=3)
    arena_b = Arena(shape, batch, dt, seed=3)
    g = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randn((batch, shape.dim), generator=g, device="cuda").to(dt)
    wqkv = (torch.randn((shape.dim + 2 * shape.kv_dim, shape.dim), generator=g, device="cuda") / shape.dim ** 0.5).to(dt)
    re32, im32 = O.rope_tables(shape.seq_len, shape.head_size)
    re, im = torch.from_numpy(re32).cuda().to(dt), torch.from_numpy(im32).cuda().to(dt)
    pos = [0, 3, shape.seq_len - 1, 7, 1]
    present = [True, True, True, False, True]
    dpos = torch.tensor(pos, dtype=torch.int32, device="cuda")
    rows_a = ops.row_table([arena_a.row_ptr(i, pos[i]) if present[i] else 0 for i in range(batch)])
    rows_b = ops.row_table([arena_b.row_ptr(i, pos[i]) if present[i] else 0 for i in range(batch)])
    # separate ops: matmul q, matmul kv, append, rope
    q = ops.matmul(x, wqkv[: shape.dim].contiguous())
    kv = ops.matmul(x, wqkv[shape.dim:].contiguous())
    ops.kv_append(rows_a, kv, shape.kv_dim)
    ops.rope(dpos, re, im, q, rows_a, shape)
    # fused
    q2, kv2 = ops.matmul_qkv_rope_append(x, wqkv, dpos, re, im, rows_b, shape, want_kv=True)
    # one (dim + 2 kv_dim, dim) product vs two separate ones: K may be split differently, so equality
    # holds to the last bit of the fp32 sums only
    tol = 2e-3 if dt == torch.float16 else 2e-6
    assert torch.allclose(q2.float(), q.float(), rtol=tol, atol=tol)
    assert torch.allclose(kv2.float(), kv.float(), rtol=tol, atol=tol)
    assert torch.allclose(arena_b.dev.float(), arena_a.dev.float(), rtol=tol, atol=tol)
    for i in range(batch):
        if present[i]:
            # the appended V half is exactly the (unrotated) matmul result the call reports
            assert torch.equal(arena_b.dev[i, pos[i], shape.kv_dim:], kv2[i, shape.kv_dim:])
        else:
            assert torch.equal(q2[i], kv2.new_tensor(q2[i]))      # finite, untouched by RoPE (checked via the oracle below)
    # rows other than the appended ones are untouched bit for bit
    before = torch.from_numpy(arena_b.host).cuda()
    mask = torch.ones(before.shape[:2], dtype=torch.bool, device="cuda")
    for i in range(batch):
        if present[i]:
            mask[i, pos[i]] = False
    assert torch.equal(arena_b.dev[mask], before[mask])


# tokens that end on a tile, behind one, with a rest that is a product of its own; steps that are walked (even) and not; heads of 128 to 8
@pytest.mark.parametrize("s,kv_heads,gqa,head_size,b", [(1024, 4, 2, 128, 7168), (2048, 4, 4, 128, 3328), (2048, 4, 4, 128, 4100), (1024, 8, 4, 64, 5000), (576, 2, 8, 128, 7000),
                                                        (640, 16, 2, 32, 9000), (512, 32, 4, 16, 9000), (576, 32, 4, 8, 9100),
                                                        (8192, 8, 8, 128, 3328)])
def test_many_rows_of_qkv_rotated_and_appended(s, kv_heads, gqa, head_size, b):
    """Against product, append and rotation one by one.  The product may sum in another order (a rounding of f16), and a rotation adds two products.  Empty
    contexts keep their query unrotated; the rows around an appended one stay as they are; cache rows off a 16-byte boundary."""
    dim, kv_dim = kv_heads * gqa * head_size, kv_heads * head_size
    assert _lib.lib().gh_matmul_qkv_fuses_many_rows(s, kv_heads, gqa, head_size, b, 0) == 1
    shape = Shape(dim=dim, n_layers=1, n_heads=kv_heads * gqa, n_kv_heads=kv_heads, hidden_dim=64, seq_len=64)
    g = torch.Generator(device="cuda").manual_seed(b)
    x = torch.randn((b, s), generator=g, device="cuda").half()
    w = (torch.randn((dim + 2 * kv_dim, s), generator=g, device="cuda") / s ** 0.5).half()
    pos = torch.randint(0, 64, (b,), generator=g, device="cuda", dtype=torch.int32)
    angle = torch.rand((64, head_size // 2), generator=g, device="cuda") * 6
    re, im = torch.cos(angle).half(), torch.sin(angle).half()
    for shift in (0, 4):
        flat = [torch.full((2 * b * 2 * kv_dim + 8,), 5.0, dtype=torch.float16, device="cuda") for _ in range(2)]
        caches = [f[shift: shift + 2 * b * 2 * kv_dim].view(b, 2, 2 * kv_dim) for f in flat]         # a row is appended, the next stays
        rows = [ops.row_table([0 if i % 97 == 5 else c[i].data_ptr() for i in range(b)]) for c in caches]
        q = ops.matmul(x, w[:dim].contiguous())
        ops.kv_append(rows[0], ops.matmul(x, w[dim:].contiguous()), kv_dim)
        ops.rope(pos, re, im, q, rows[0], shape)
        got, _ = ops.matmul_qkv_rope_append(x, w, pos, re, im, rows[1], shape)
        assert torch.allclose(got.float(), q.float(), rtol=4e-3, atol=4e-3)
        assert torch.allclose(flat[1].float(), flat[0].float(), rtol=4e-3, atol=4e-3)
        assert (caches[1][:, 1] == 5.0).all() and (caches[1][5] == 5.0).all()


@pytest.mark.parametrize("name,dtype", [("test-gqa4", "f16"), ("stories15m", "f32"), ("test-tiny", "f32")])
def test_stage_with_and_without_fused_projections(name, dtype):
    cfg = SHAPES[name]
    np_dt = np.float16 if dtype == "f16" else np.float32
    wcls = name != "stories15m"
    layers, base = make_weights(cfg, np_dt, seed=31, wcls=wcls)
    batch = 4
    a = S.Stage(name, dtype, 0, cfg.n_layers, batch, batch, with_cls=True, fused_projections=True)
    b = S.Stage(name, dtype, 0, cfg.n_layers, batch, batch, with_cls=True, fused_projections=False)
    ref = OracleModel(cfg, layers, base)
    ref16 = OracleModel(cfg, layers, base, np.float16) if dtype == "f16" else None
    for st in (a, b):
        load_weights(st, cfg, layers, base, wcls)
        st.new_state(batch)
        for i in range(batch):
            st.set_prompt(i, i, 3 + i, 0)
    tokens = [3 + i for i in range(batch)]
    for step in range(8):
        want = ref.step(tokens, list(range(batch)), [step] * batch)
        assert a.forward() and b.forward()
        la = d2h(a.scratch_ptr("logits"), (batch, cfg.vocab_size), np_dt).astype(np.float32)
        lb = d2h(b.scratch_ptr("logits"), (batch, cfg.vocab_size), np_dt).astype(np.float32)
        # the two differ in reduction order only: the rmsnorm sum, and the K split of a concatenated
        # projection against the split of its parts (an fp16 rounding can flip and travel through the layers)
        tol = 8e-3 if dtype == "f16" else 2e-5
        np.testing.assert_allclose(la, lb, rtol=tol, atol=tol)
        if dtype == "f16":
            want16 = ref16.step(tokens, list(range(batch)), [step] * batch)
            assert_half_parity(la, want16, want, what=f"{name} fused-projection logits step {step}")
            assert_half_parity(lb, want16, want, what=f"{name} separate-projection logits step {step}")
        else:
            assert_close(la, want, mean_rel=1e-3, what=f"{name} fused-projection logits step {step}")
        tokens = [a.row(i)["token"] for i in range(batch)]
        for i in range(batch):                         # keep both stages on the same token stream
            b.set_prompt(i, i, tokens[i], step + 1)
            a.set_prompt(i, i, tokens[i], step + 1)
    a.close()
    b.close()


# every width of the activation tile and the row it ends on; shares of 32 to 64 rows of the CUs, work-groups with a part of a share; K that ends inside a step, that is
# shorter than the ring, one step; heads of 8
@pytest.mark.parametrize("s,kv_heads,gqa,head_size,b", [(4096, 32, 1, 128, 1), (4096, 32, 1, 128, 32), (1024, 16, 4, 128, 33), (1024, 32, 2, 64, 64), (520, 32, 2, 128, 48),
                                                        (1000, 16, 4, 128, 20), (1096, 32, 1, 128, 63), (128, 32, 2, 64, 5), (64, 512, 1, 8, 17),
                                                        (8, 200, 1, 20, 3), (5120, 40, 1, 128, 31), (8192, 8, 8, 128, 16)])
def test_few_rows_of_qkv_rotated_and_appended(s, kv_heads, gqa, head_size, b):
    """Against 64 bits: two roundings of f16 and fp32 sums of s products.  Empty contexts keep their query unrotated; cache rows on and off an 8-byte boundary, the rows around them."""
    dim, kv_dim = kv_heads * gqa * head_size, kv_heads * head_size
    shape = Shape(dim=dim, n_layers=1, n_heads=kv_heads * gqa, n_kv_heads=kv_heads, hidden_dim=64, seq_len=64)
    g = torch.Generator(device="cuda").manual_seed(b)
    x = torch.randn((b, s), generator=g, device="cuda").half()
    w = (torch.randn((dim + 2 * kv_dim, s), generator=g, device="cuda") / s ** 0.5).half()
    pos = torch.randint(0, 64, (b,), generator=g, device="cuda", dtype=torch.int32)
    angle = torch.rand((64, head_size // 2), generator=g, device="cuda") * 6
    re, im = torch.cos(angle).half(), torch.sin(angle).half()
    assert _lib.lib().gh_matmul_qkv_fuses_few_rows(s, kv_heads, gqa, head_size, b, _lib.GH_F16) == 1
    y = (x.double() @ w.double().t()).half().double()
    missing = [i for i in range(b) if i % 7 == 5]
    turn = torch.ones((b, 1, 1), dtype=torch.bool, device="cuda")
    turn[missing] = False
    a, c = re[pos.long()].double()[:, None], im[pos.long()].double()[:, None]

    def turned(v):
        v = v.view(b, -1, head_size // 2, 2)
        out = torch.stack([v[..., 0] * a - v[..., 1] * c, v[..., 0] * c + v[..., 1] * a], -1).view(b, -1, head_size)
        return torch.where(turn, out, v.reshape(b, -1, head_size)).reshape(b, -1)

    want_q, want_row = turned(y[:, :dim].contiguous()), torch.cat([turned(y[:, dim: dim + kv_dim].contiguous()), y[:, dim + kv_dim:]], 1)
    for shift in (0, 1):
        flat = torch.full((2 * b * 2 * kv_dim + 8,), 5.0, dtype=torch.float16, device="cuda")
        cache = flat[shift: shift + 2 * b * 2 * kv_dim].view(b, 2, 2 * kv_dim)
        rows = ops.row_table([0 if i in missing else cache[i].data_ptr() for i in range(b)])
        got, _ = ops.matmul_qkv_rope_append(x, w, pos, re, im, rows, shape)
        # a product's sum may round to either side of a tie: one unit of f16 (2^-10) of each of a pair, and the rotation's own rounding
        assert torch.allclose(got.double(), want_q, rtol=4e-3, atol=4e-3)
        for i in range(b):
            assert (cache[i] == 5.0).all() if i in missing else torch.allclose(cache[i, 0].double(), want_row[i], rtol=4e-3, atol=4e-3) and (cache[i, 1] == 5.0).all()


# widths and heads of the smallest and the largest the launch takes, groups of query heads, heads that leave rows of lanes idle; more keys than one turn
@pytest.mark.parametrize("kv_heads,gqa,head_size,batch", [(6, 1, 48, 4), (2, 2, 8, 7), (5, 1, 64, 3), (2, 4, 40, 6), (1, 1, 4, 8), (4, 1, 20, 64), (3, 2, 44, 8)])
def test_attention_in_the_launch_of_its_projections(kv_heads, gqa, head_size, batch):
    """Against 64 bits: rounding is that of fp32 sums of up to 320 products and 600 weights, some 1e-6; a wrong key, row or rotation is far beyond.  Cache rows on
    and off a 16-byte boundary, an empty context, a key whose scores are infinite, rows around the appended one."""
    shape = Shape(dim=kv_heads * gqa * head_size, n_layers=1, n_heads=kv_heads * gqa, n_kv_heads=kv_heads, hidden_dim=64, seq_len=600)
    dim, kv_dim = shape.dim, shape.kv_dim
    g = torch.Generator(device="cuda").manual_seed(head_size)
    x, nw = torch.randn((batch, dim), generator=g, device="cuda"), torch.randn((dim,), generator=g, device="cuda")
    w = torch.randn((dim + 2 * kv_dim, dim), generator=g, device="cuda") / dim ** 0.5
    angle = torch.rand((600, head_size // 2), generator=g, device="cuda") * 6
    re, im = torch.cos(angle), torch.sin(angle)
    pos = ([0, 1, 255, 256, 599, 31, 257, 300] * 8)[:batch]
    dpos = torch.tensor(pos, dtype=torch.int32, device="cuda")
    assert _lib.lib().gh_rmsnorm_qkv_attn_rides(batch, ctypes.byref(shape.c()), _lib.GH_F32) == 1
    for shift in (0, 1):
        flat = torch.randn((batch * 600 * 2 * kv_dim + 1,), generator=g, device="cuda")
        cache = flat[shift: shift + batch * 600 * 2 * kv_dim].view(batch, 600, 2 * kv_dim)
        cache[2, 7, 0] = -float("inf")
        before = cache.clone()
        rows = ops.row_table([0 if i == 1 and batch > 4 else cache[i].data_ptr() for i in range(batch)])
        ends = ops.row_table([0 if i == 1 and batch > 4 else cache[i, pos[i]].data_ptr() for i in range(batch)])
        got = ops.rmsnorm_qkv_attn(x, nw, w, dpos, re, im, rows, ends, shape)
        xd = x.double()
        y = (xd / torch.sqrt((xd * xd).mean(1, keepdim=True) + 1e-5) * nw.double()) @ w.double().t()
        for i in range(batch):
            if i == 1 and batch > 4:
                assert (got[i] == 0).all() and torch.equal(cache[i], before[i])
                continue
            p = pos[i]
            a, b = re[p].double(), im[p].double()

            def turned(v):
                v = v.view(-1, head_size // 2, 2)
                return torch.stack([v[..., 0] * a - v[..., 1] * b, v[..., 0] * b + v[..., 1] * a], -1).view(-1, head_size)

            q, k, v = turned(y[i, :dim]), turned(y[i, dim: dim + kv_dim]), y[i, dim + kv_dim:].view(-1, head_size)
            old = before[i, :p].double().view(p, 2, kv_heads, head_size)
            keys, values = torch.cat([old[:, 0], k[None]]), torch.cat([old[:, 1], v[None]])
            want = torch.empty((gqa * kv_heads, head_size), dtype=torch.float64, device="cuda")
            for h in range(gqa * kv_heads):
                want[h] = torch.softmax(keys[:, h // gqa].contiguous() @ q[h] * head_size ** -0.5, 0) @ values[:, h // gqa].contiguous()
            for have, should in ((got[i], want.view(-1)), (cache[i, p], torch.cat([k.view(-1), v.view(-1)]))):
                fine = ~should.isnan()
                assert torch.equal(have.isnan(), ~fine)
                assert (have.double() - should)[fine].norm() <= 5e-6 * should[fine].norm() + 1e-12
            keep = torch.arange(600, device="cuda") != p
            assert torch.equal(cache[i][keep], before[i][keep])
