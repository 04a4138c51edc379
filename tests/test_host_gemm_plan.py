"""The GEMM kernels' plans are host logic: properties every plan must have, and the plans of the shapes the benchmark configurations use
(256 compute units, the value the library assumes before a device is initialised).  gh_gemm_ring_plan is of the kernel that products of up
to some hundred rows run on, gh_gemm_stream_plan of the one that runs on request."""
import ctypes as C
import threading

import numpy as np
import pytest

from glinthawk_amd import _lib


def plan(s, r, b):
    splits, kps, rows = C.c_uint32(0), C.c_uint32(0), C.c_uint32(0)
    _lib.check(_lib.lib().gh_gemm_stream_plan(s, r, b, C.byref(splits), C.byref(kps), C.byref(rows)))
    return splits.value, kps.value, rows.value


def test_every_plan_covers_k_exactly_once():
    rng = np.random.default_rng(5)
    shapes = [(256, 4, 1), (256, 100000, 64), (1 << 16, 128, 3)]
    shapes += [(256 * int(rng.integers(1, 200)), 4 * int(rng.integers(1, 20000)), int(rng.integers(1, 300))) for _ in range(300)]
    for s, r, b in shapes:
        splits, kps, rows = plan(s, r, b)
        assert splits >= 1 and kps % 256 == 0 and kps >= 256
        assert (splits - 1) * kps < s <= splits * kps, (s, r, b, splits, kps)      # no empty range, nothing left over
        assert rows in (96, 112, 128)
        if splits > 1:
            assert rows == 128 and kps >= 512, (s, r, b, splits, kps, rows)          # small tiles only without a split; at least two slabs per range
        assert splits <= 16


@pytest.mark.parametrize("name,s,r,b,want", [
    ("70B wo", 8192, 8192, 64, (4, 2048, 128)),                 # 64 row blocks x 4 = one work-group per CU
    ("70B wq+wkv", 8192, 10240, 64, (3, 2816, 128)),            # 80 x 3 = 240, not 320
    ("70B w2", 28672, 8192, 64, (8, 3584, 128)),                # two work-groups per CU
    ("70B w1+w3", 8192, 57344, 64, (1, 8192, 112)),             # 512 work-groups of 112 rows instead of 448 of 128
    ("7B wo", 4096, 4096, 32, (8, 512, 128)),
    ("13B w1+w3", 5120, 27648, 8, (2, 2560, 128)),
])
def test_plans_of_the_benchmark_shapes(name, s, r, b, want):
    assert plan(s, r, b) == want, name


def test_rejects_what_the_kernel_does_not_take():
    splits, kps, rows = C.c_uint32(0), C.c_uint32(0), C.c_uint32(0)
    rc = _lib.lib().gh_gemm_stream_plan(100, 64, 1, C.byref(splits), C.byref(kps), C.byref(rows))
    assert rc != 0 and b"256" in _lib.lib().gh_last_error()


def ring_plan(s, r, b, gated=False):
    out = (C.c_uint32 * 6)()
    _lib.check(_lib.lib().gh_gemm_ring_plan(s, r, b, int(gated), out))
    return tuple(out)


def some_shapes(n, seed):
    rng = np.random.default_rng(seed)
    size = lambda lo, hi: int(np.exp(rng.uniform(np.log(lo), np.log(hi))))
    return [(8 * size(1, 4000), 4 * size(1, 20000), size(1, 3000 if i % 3 else 70), bool(i % 2)) for i in range(n)]


def test_every_ring_plan_covers_the_product_once():
    for s, r, b, gated in [(8, 1, 1, False), (8, 4, 1, True), (1 << 21, 128, 3, False), (288, 32000, 7000, False)] + some_shapes(500, 6):
        w, x, rows, cols, splits, steps = ring_plan(s, r, b, gated)
        assert (w, x) in [(128, 32), (256, 32), (128, 64), (256, 64), (128, 96), (256, 96), (128, 128), (256, 128), (128, 192), (128, 256)]
        assert rows % 4 == 0 and 16 <= rows <= (w // 2 if gated else w) and 1 <= cols <= x and (b > 256 or x >= b)
        total = -(-s // 64)
        assert 1 <= splits <= 16 and steps * (splits - 1) < total <= steps * splits      # no empty range, nothing left over
        assert splits == 1 or (steps >= 4 and not gated)
        assert -(-b // cols) * cols >= b and (cols % 16 == 0 or cols >= b)


@pytest.mark.parametrize("name,s,r,b,gated,want", [
    ("70B wo", 8192, 8192, 64, False, (128, 64, 128, 64, 4, 32)),
    ("70B w2", 28672, 8192, 64, False, (256, 64, 256, 64, 8, 56)),
    ("70B w1 and w3", 8192, 28672, 64, True, (256, 64, 112, 64, 1, 128)),
    ("7B wq and wkv", 4096, 12288, 32, False, (128, 32, 96, 32, 2, 32)),
    ("7B w1 and w3, a prompt", 4096, 11008, 77, True, (128, 96, 44, 80, 1, 64)),
])
def test_ring_plans_of_the_benchmark_shapes(name, s, r, b, gated, want):
    assert ring_plan(s, r, b, gated) == want, name


def test_a_kept_ring_plan_is_that_of_its_product():
    """More shapes than a thread keeps plans of, asked for again and again, from several threads, and with the units to balance for changed in
    between: every answer is the first one's."""
    shapes = some_shapes(400, 7)
    first = [ring_plan(*c) for c in shapes]
    wrong = []

    def ask():
        for _ in range(3):
            wrong.extend(c for c, want in zip(shapes, first) if ring_plan(*c) != want)

    threads = [threading.Thread(target=ask) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    try:
        _lib.check(_lib.lib().gh_gemm_set_tuning(0, 64, 0))
        assert sum(ring_plan(*c) != want for c, want in zip(shapes, first)) > 100
    finally:
        _lib.check(_lib.lib().gh_gemm_set_tuning(0, 256, 0))
    assert [ring_plan(*c) for c in shapes] == first


def test_ring_plan_rejects_what_the_kernel_does_not_take():
    out = (C.c_uint32 * 6)()
    for s, r, b, gated in [(100, 64, 1, 0), ((1 << 21) + 8, 64, 1, 0), (64, 0, 1, 0), (64, 64, 0, 0), (64, 66, 1, 1)]:
        assert _lib.lib().gh_gemm_ring_plan(s, r, b, gated, out) != 0 and b"ring" in _lib.lib().gh_last_error()


def test_q_k_v_of_few_rows_leave_their_own_kernel_to_a_forced_one():
    """The fused product has a kernel of its own for 32 to 64 weight rows a compute unit: a forced kernel goes before it, and the units that plans are balanced for are its."""
    lib = _lib.lib()
    shapes = [(4096, 32, 1, 128, 32), (8192, 8, 8, 128, 1), (5120, 40, 1, 128, 16)]

    def takes(shape):
        return lib.gh_matmul_qkv_fuses_few_rows(*shape, _lib.GH_F16)

    assert [takes(c) for c in shapes] == [1, 1, 1]
    try:
        for kernel in (1, 2, 3, 4, 5):
            _lib.check(lib.gh_gemm_set_tuning(kernel, 0, 0))
            assert [takes(c) for c in shapes] == [0, 0, 0], kernel
        _lib.check(lib.gh_gemm_set_tuning(0, 64, 0))              # 160 to 240 rows a unit
        assert [takes(c) for c in shapes] == [0, 0, 0]
    finally:
        _lib.check(lib.gh_gemm_set_tuning(0, 256, 0))
    assert [takes(c) for c in shapes] == [1, 1, 1]
