"""Operator parity on the device: each ernie_hip op against the oracle and the
reference's own known-answer tests (ported in kat.py)."""
import math

import numpy as np
import pytest

import ernie_amd as E
import kat
import oracle as O
from gpu_util import ALL_DT, NAMES, dev, empty, host, stored

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ALL_DT, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("width", [128, 3072, 4096])
@pytest.mark.parametrize("scale", [1.0, 512.0])
def test_rmsnorm_probe_kat(ctx, dt, width, scale):
    # probes/rmsnorm_probe.cpp: inputs and weights exact in every storage type.
    x, gamma, expected = kat.rmsnorm_kat_case(width, scale)
    xd, out = dev(x, dt), empty(x.shape, dt)
    ctx.rmsnorm(xd, dt, dev(gamma), x.shape[0], width, out, dt)
    err = np.max(np.abs(host(out) - expected))
    assert err <= kat.RMSNORM_LIMITS[NAMES[dt]], err


@pytest.mark.parametrize("scale", [1.0, 1024.0])
def test_layernorm_probe_kat(ctx, scale):
    x, _, expected = kat.rmsnorm_kat_case(4096, scale, centered=True)
    zeros = dev(np.zeros(4096, np.float32))
    out = empty(x.shape)
    ctx.layernorm_modulate(dev(x), zeros, zeros, x.shape[0], 4096, out, E.FP32)
    assert np.max(np.abs(host(out) - expected)) <= kat.RMSNORM_LIMITS["fp32"]


@pytest.mark.parametrize("dt", ALL_DT, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("shape", [0, 1])
def test_gelu_probe_kat(ctx, dt, shape):
    x = kat.gelu_kat_input(shape)
    xd = dev(x, dt)
    ctx.gelu(xd, dt, x.size)
    err = np.max(np.abs(host(xd) - kat.gelu_expected(x)))
    assert err <= kat.GELU_LIMITS[NAMES[dt]], err


@pytest.mark.parametrize("dt", ALL_DT, ids=lambda d: NAMES[d])
def test_residual_contract(ctx, dt):
    # tests/test_residual_contract.cpp: |a| >= 70000 adds exactly in FP32, and the
    # low-storage normalized projection of the sum stays within .001 / .004.
    a, b = kat.residual_case()
    out = empty(a.shape)
    ctx.residual_add(dev(a), E.FP32, dev(b, dt), dt, out, a.size)
    s = host(out)
    np.testing.assert_array_equal(s, (a + b).astype(np.float32))
    norm = empty(a.shape, dt)
    ctx.rmsnorm(out, E.FP32, dev(np.ones(4096, np.float32)), 4, 4096, norm, dt)
    sd = s.astype(np.float64)
    expected = sd / np.sqrt((sd * sd).mean(axis=1, keepdims=True) + 1e-6)
    limit = {E.FP32: 1e-6, E.FP16: 0.001, E.BF16: 0.004}[dt]
    assert np.max(np.abs(host(norm) - expected)) <= limit


@pytest.mark.parametrize("dt", ALL_DT, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("name,m,n,k,bias", kat.GEMM_KAT_SHAPES)
def test_gemm_exact_products_kat(ctx, dt, name, m, n, k, bias):
    # tests/test_bf16_gemm.cpp: multiples of 1/8, exact FP32 products and sums;
    # the low-precision result must equal round-to-nearest-even of the FP64 sum.
    a, w, b = kat.gemm_kat_case(m, n, k)
    ref = a.astype(np.float64) @ w.astype(np.float64).T + (b.astype(np.float64) if bias else 0.0)
    ad, wd = dev(a, dt), dev(w, dt)
    bd = dev(b) if bias else None
    c32 = empty((m, n))
    ctx.gemm(ad, k, wd, k, c32, n, m, n, k, dt, E.FP32, bias=bd)
    np.testing.assert_array_equal(host(c32).astype(np.float64), ref)
    if dt != E.FP32:
        c16 = empty((m, n), dt)
        ctx.gemm(ad, k, wd, k, c16, n, m, n, k, dt, dt, bias=bd)
        np.testing.assert_array_equal(host(c16), stored(ref.astype(np.float32), dt))


@pytest.mark.parametrize("dt", ALL_DT, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("m,n,k", [(300, 520, 256), (4160, 256, 512), (33, 4096, 128), (1056, 96, 4096),
                                   (4160, 4096, 256), (4120, 4096, 256)])
def test_gemm_random_against_oracle(ctx, dt, m, n, k):
    # 4160 / 4120 x 4096: 256 full tiles and a 64- or 24-row tail row; the 16-bit kernel
    # computes the tail in 16-row chunks inside full tiles (light tiles), one per
    # workgroup at most.
    a = O.normal((m, k), 1)
    w = O.normal((n, k), 2, std=0.02)
    a_s, w_s = stored(a, dt), stored(w, dt)
    ref = O.gemm_nt(a_s, w_s).astype(np.float64)
    c = empty((m, n))
    ctx.gemm(dev(a, dt), k, dev(w, dt), k, c, n, m, n, k, dt, E.FP32)
    g = kat.gate(host(c), ref, 0, 1e-5, 1e-5)
    assert g["passed"], g


@pytest.mark.parametrize("dt", [E.FP16, E.BF16], ids=lambda d: NAMES[d])
@pytest.mark.parametrize("m,n,k", [(193, 256, 96), (255, 520, 128), (481, 384, 256)])
def test_gemm_last_rows_of_a_nearly_full_tile(ctx, dt, m, n, k):
    # 193 to 255 rows past a multiple of 256: the last tile needs its whole height.
    a, w = O.normal((m, k), 3), O.normal((n, k), 4, std=0.02)
    ref = O.gemm_nt(stored(a, dt), stored(w, dt)).astype(np.float64)
    c = empty((m, n)).fill_(float("nan"))
    ctx.gemm(dev(a, dt), k, dev(w, dt), k, c, n, m, n, k, dt, E.FP32)
    g = kat.gate(host(c), ref, 0, 1e-5, 1e-5)
    assert g["passed"], g


@pytest.mark.parametrize("m,n,k,ldc", [(1, 5, 16, 7), (260, 260, 16, 260), (127, 132, 48, 132), (129, 128, 80, 128),
                                       (260, 260, 1040, 261)])
def test_gemm_fp32_split_products(ctx, m, n, k, ldc):
    # Tile edges, K steps of 16 past a multiple of 32, unaligned output rows (K = 16: on the
    # FP32 matrix cores, without a split). The three
    # parts are exact and the products left out below 2^-24 of a product, so the error is
    # that of k FP32 roundings: k 2^-24 of sum |a| |w|. In the 2-norm 2e-8 to 2e-7 of the
    # result were measured; without one of the six partial products it is 1.8e-6 and more.
    a, w = O.normal((m, k), 3) * np.float32(1000), O.normal((n, k), 4, std=0.02)
    a64, w64 = a.astype(np.float64), w.astype(np.float64)
    c = empty((m, ldc)).fill_(float("nan"))
    ctx.gemm(dev(a), k, dev(w), k, c, ldc, m, n, k, E.FP32, E.FP32)
    ref = a64 @ w64.T
    assert np.all(np.abs(host(c)[:, :n] - ref) <= (k + 1) * 2.0**-24 * (np.abs(a64) @ np.abs(w64).T))
    assert np.linalg.norm(host(c)[:, :n] - ref) <= 5e-7 * np.linalg.norm(ref)


@pytest.mark.parametrize("m,n,k", [(130, 140, 48), (33, 260, 4096)])
@pytest.mark.parametrize("sa,sw", [(1e-36, 1.0), (1.0, 1e-37), (1e-37, 1e30), (1e-42, 1e20), (1e-20, 1e-15)])
def test_gemm_fp32_small_magnitudes(ctx, m, n, k, sa, sw):
    # Values down to FP32 subnormals keep all their bits. Error of a sum of k products
    # in FP32: at most k 2^-24 of sum |a| |w|, about sqrt(k) 2^-24 of it in the 2-norm, where
    # |result| is about sum |a| |w| / sqrt(k): k 2^-24 at the very most, and about 2e-7
    # measured; lost low bits of a value of 1e-36 alone give 2.6e-5.
    a, w = O.normal((m, k), 3) * np.float32(sa), O.normal((n, k), 4) * np.float32(sw)
    ref = a.astype(np.float64) @ w.astype(np.float64).T
    c = empty((m, n)).fill_(float("nan"))
    ctx.gemm(dev(a), k, dev(w), k, c, n, m, n, k, E.FP32, E.FP32)
    assert np.linalg.norm(host(c) - ref) <= 1e-6 * np.linalg.norm(ref)


def test_gemm_fp32_identity_returns_every_value(ctx):
    # Values of all exponents with random significands, subnormals included, times the
    # identity: the parts of each value add up to it exactly.
    m, k = 4096, 32
    rng = np.random.default_rng(11)
    bits = (np.arange(m * k, dtype=np.uint32) % 255) << 23 | rng.integers(0, 1 << 23, m * k, dtype=np.uint32)
    a = (bits | rng.integers(0, 2, m * k, dtype=np.uint32) << 31).view(np.float32).reshape(m, k)
    c = empty((m, k))
    ctx.gemm(dev(a), k, dev(np.eye(k, dtype=np.float32)), k, c, k, m, k, k, E.FP32, E.FP32)
    assert np.array_equal(host(c), a)


@pytest.mark.parametrize("k", [48, 4096])
def test_gemm_fp32_infinities_and_the_largest_values(ctx, k):
    # Infinities stay infinities (no infinity times a zero part), NaN stays in its row,
    # and a value that rounds to a BF16 infinity is still a finite FP32 one. K = 4096: the
    # same in tiles that are split along K.
    m, n = 130, 140
    a, w = O.normal((m, k), 5), np.abs(O.normal((n, k), 6)) + np.float32(0.5)
    a[3, 7], a[70, 1], a[129, 47] = np.inf, np.nan, -np.inf
    big = np.finfo(np.float32).max
    a[40], w[2] = 0, 0
    a[40, 33], w[2, 33] = big, 1
    c = empty((m, n))
    ctx.gemm(dev(a), k, dev(w), k, c, n, m, n, k, E.FP32, E.FP32)
    got = host(c)
    rest = np.delete(np.arange(n), 2)
    assert np.all(np.isposinf(got[3][rest])) and np.all(np.isneginf(got[129][rest])) and np.all(np.isnan(got[70]))
    assert got[40, 2] == big
    ok = np.delete(np.arange(m), (3, 40, 70, 129))
    ref = a[ok].astype(np.float64) @ w.astype(np.float64).T
    assert np.all(np.abs(got[ok] - ref) <= (k + 1) * 2.0**-24 * (np.abs(a[ok]).astype(np.float64) @ np.abs(w).T))


@pytest.mark.parametrize("dt", [E.FP16, E.BF16], ids=lambda d: NAMES[d])
@pytest.mark.parametrize("m,n,k", [(1, 17, 32), (15, 520, 96), (16, 8200, 544), (17, 300, 2048), (128, 300, 2048),
                                   (129, 300, 2048)])
def test_gemm_few_rows(ctx, dt, m, n, k):
    # Up to 16 rows: 16 or (past 8192 columns) 32 columns per workgroup, K steps that do
    # not divide among its waves. More rows: every tile split along K; the same calls in
    # a captured graph, which takes no scratch: up to 128 rows 16 columns per workgroup.
    import torch
    a, w, bias = O.normal((m, k), 3), O.normal((n, k), 4, std=0.02), O.normal((n,), 5)
    ref = O.gemm_nt(stored(a, dt), stored(w, dt)).astype(np.float64) + bias
    ad, wd, bd, c = dev(a, dt), dev(w, dt), dev(bias), empty((m, n)).fill_(float("nan"))
    ctx.gemm(ad, k, wd, k, c, n, m, n, k, dt, E.FP32, bias=bd)
    g = kat.gate(host(c), ref, 0, 1e-5, 1e-5)
    assert g["passed"], g
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    c.fill_(float("nan"))
    torch.cuda.synchronize()
    try:
        ctx.call("set_stream", E.c_vp(stream.cuda_stream))
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="relaxed"):
            ctx.gemm(ad, k, wd, k, c, n, m, n, k, dt, E.FP32, bias=bd)
    finally:
        ctx.call("set_stream", E.c_vp(torch.cuda.current_stream().cuda_stream))
    for _ in range(2):
        graph.replay()
        torch.cuda.synchronize()
        g = kat.gate(host(c), ref, 0, 1e-5, 1e-5)
        assert g["passed"], g
        c.fill_(float("nan"))
        torch.cuda.synchronize()


@pytest.mark.parametrize("dt", [E.FP16, E.BF16], ids=lambda d: NAMES[d])
@pytest.mark.parametrize("m,n,k", [(257, 300, 2048), (320, 520, 1056), (575, 300, 2080), (576, 96, 4096), (832, 300, 2048),
                                   (257, 16900, 4096), (1030, 12032, 64)])
def test_gemm_tail_rows_below_few_tiles(ctx, dt, m, n, k):
    # 1 to 64 rows below one to three rows of tiles, every tile split along K. 257 x 16900: 134
    # tiles are too many for that, so the 67 of one row are 320 rows tall. 1030 x 12032
    # and K = 64: 188 full tiles and 47 of the tail in one round, none split.
    a, w = O.normal((m, k), 3), O.normal((n, k), 4, std=0.02)
    ref = O.gemm_nt(stored(a, dt), stored(w, dt)).astype(np.float64)
    c = empty((m, n)).fill_(float("nan"))
    ctx.gemm(dev(a, dt), k, dev(w, dt), k, c, n, m, n, k, dt, E.FP32)
    g = kat.gate(host(c), ref, 0, 1e-5, 1e-5)
    assert g["passed"], g


@pytest.mark.parametrize("dt", [E.FP16, E.BF16], ids=lambda d: NAMES[d])
@pytest.mark.parametrize("out", [E.FP32, None], ids=["fp32-out", "16-bit-out"])
@pytest.mark.parametrize("m,n,k", [(1344, 12288, 64), (1313, 12285, 96), (1282, 24576, 32), (1330, 24570, 32)])
def test_gemm_light_tiles_on_a_partial_round(ctx, dt, out, m, n, k):
    # Five rows of 48 or 96 full tiles, 15/16 of one or two rounds, and a tail of 2 to 64 rows
    # whose tiles would begin another round: the tail goes into the full tiles as one to
    # four chunks of 16 rows (ragged columns: stored element by element).
    a, w, bias = O.normal((m, k), 3), O.normal((n, k), 4, std=0.02), O.normal((n,), 5)
    ref = O.gemm_nt(stored(a, dt), stored(w, dt)).astype(np.float64) + bias
    c = empty((m, n), out or dt).fill_(float("nan"))
    ctx.gemm(dev(a, dt), k, dev(w, dt), k, c, n, m, n, k, dt, out or dt, bias=dev(bias))
    # One rounding to the output type: half a unit in the last place, at most 2^-11 or 2^-8 of a value.
    eps = 1e-5 if out else 2.0**-11 + 1e-5 if dt == E.FP16 else 2.0**-8 + 1e-5
    assert np.all(np.abs(host(c) - ref) <= eps * (np.abs(ref) + 1e-2))


def test_gemm_scratch_is_allocated_when_used():
    # A context takes no scratch until a matrix product of its own can use it.
    import torch
    before = torch.cuda.mem_get_info()[0]
    c = E.Context(0)
    assert before - torch.cuda.mem_get_info()[0] < 64 << 20
    c.close()


def test_gemm_scratch_beside_a_capture(ctx):
    # Calls on the null stream, then on another one while a third stream is captured in the
    # strictest mode: the capture stays valid, and both calls have their results.
    import torch
    m, n, k = 300, 256, 4096
    a, w = O.normal((m, k), 3), O.normal((n, k), 4, std=0.02)
    ref = O.gemm_nt(stored(a, E.FP16), stored(w, E.FP16)).astype(np.float64)
    ad, wd, outs = dev(a, E.FP16), dev(w, E.FP16), [empty((m, n)).fill_(float("nan")) for _ in range(2)]
    side, captured, graph = torch.cuda.Stream(), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    x = empty((4096,)).fill_(0)
    torch.cuda.synchronize()
    try:
        ctx.call("set_stream", None)
        ctx.gemm(ad, k, wd, k, outs[0], n, m, n, k, E.FP16, E.FP32)
        ctx.call("set_stream", E.c_vp(side.cuda_stream))
        with torch.cuda.graph(graph, stream=captured, capture_error_mode="global"):
            x.add_(1)
            ctx.gemm(ad, k, wd, k, outs[1], n, m, n, k, E.FP16, E.FP32)
    finally:
        ctx.call("set_stream", E.c_vp(torch.cuda.current_stream().cuda_stream))
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
    assert np.all(host(x) == 3)
    for out in outs:
        g = kat.gate(host(out), ref, 0, 1e-5, 1e-5)
        assert g["passed"], g


def captured_gemm(ctx, *args):
    """The call recorded into a graph, which takes no scratch, and replayed."""
    import torch
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    try:
        ctx.call("set_stream", E.c_vp(stream.cuda_stream))
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="relaxed"):
            ctx.gemm(*args)
    finally:
        ctx.call("set_stream", E.c_vp(torch.cuda.current_stream().cuda_stream))
    graph.replay()
    torch.cuda.synchronize()


@pytest.mark.parametrize("m,n,k,split", [(320, 16384, 1024, False), (2090, 4096, 1024, False), (400, 24576, 1024, False),
                                         (1152, 8192, 1024, False), (1568, 12288, 1024, False), (1056, 12288, 1024, False),
                                         (100, 1024, 4096, True), (320, 1024, 4096, True), (512, 1024, 4096, True),
                                         (2368, 8192, 4096, True), (1152, 16384, 4096, True)])
def test_gemm_split_where_it_pays(ctx, m, n, k, split):
    # Enough tiles or few K steps: no split (nor light tiles), so the bits of a captured call,
    # which has no scratch to split with. Few tiles and many K steps: parts of K summed
    # in another order. Both against the products of the stored values.
    import torch
    a, w = dev(O.normal((m, k), 3), E.FP16), dev(O.normal((n, k), 4, std=0.02), E.FP16)
    c, whole = empty((m, n)).fill_(float("nan")), empty((m, n)).fill_(float("nan"))
    ctx.gemm(a, k, w, k, c, n, m, n, k, E.FP16, E.FP32)
    captured_gemm(ctx, a, k, w, k, whole, n, m, n, k, E.FP16, E.FP32)
    assert torch.equal(c, whole) == (not split)
    ref = a.double() @ w.double().T
    for x in (c, whole):
        # k FP32 roundings of sums that grow to the result: sqrt(k) 2^-24 of it at most.
        assert float((x - ref).norm() / ref.norm()) < math.sqrt(k) * 2**-24


@pytest.mark.parametrize("m,n,k,few", [(100, 32768, 512, False), (64, 32768, 512, False), (16, 65536, 512, False),
                                       (32, 3072, 3072, True), (128, 3072, 3072, True), (40, 8224, 1024, True),
                                       (100, 8224, 3072, True)])
def test_gemm_few_rows_where_they_pay(ctx, m, n, k, few):
    # A captured call of few rows: past the columns where every workgroup's reading of A costs
    # more than tiles over all of K, the bits of the first rows of a call with more rows
    # (whole tiles); below, the few-row kernel's, which adds its waves' parts of K.
    import torch
    rows = 260
    a, w = dev(O.normal((rows, k), 3), E.BF16), dev(O.normal((n, k), 4, std=0.02), E.BF16)
    c, more = empty((m, n)).fill_(float("nan")), empty((rows, n)).fill_(float("nan"))
    captured_gemm(ctx, a, k, w, k, c, n, m, n, k, E.BF16, E.FP32)
    captured_gemm(ctx, a, k, w, k, more, n, rows, n, k, E.BF16, E.FP32)
    assert torch.equal(c, more[:m]) == (not few)
    ref = a.double() @ w.double().T
    for x in (c, more):
        # k FP32 roundings of sums that grow to the result: sqrt(k) 2^-24 of it at most.
        assert float((x - ref[:len(x)]).norm() / ref[:len(x)].norm()) < math.sqrt(k) * 2**-24


def test_gemm_rejects_unsupported_shapes(ctx):
    a, c = empty((4, 40), E.FP16), empty((4, 8))
    with pytest.raises(E.ErnieError):
        ctx.gemm(a, 40, a, 40, c, 8, 4, 8, 40, E.FP16, E.FP32)  # K % 32 != 0


@pytest.mark.parametrize("dt", ALL_DT, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("mask_heads", [1, 2])
@pytest.mark.parametrize("queries,keys,width", [(3, 17, 128), (257, 65, 128), (3, 17, 124)])
def test_attention_mask_kat(ctx, dt, queries, keys, width, mask_heads):
    # tests/test_attention_mask.cpp: row mask == dense mask bitwise, repeated
    # runs identical, FP32 against FP64 with the mask as a visible-key count.
    heads = 2
    for shift in (0, 3):
        q, k, v, row, dense = kat.attention_mask_case(queries, keys, mask_heads, width, shift)
        qd, kd, vd = dev(q, dt), dev(k, dt), dev(v, dt)
        strides = (queries * width, width, keys * width, width, keys * width, width, queries * width, width)
        outs = []
        for rep, mask in enumerate((dense, row, row)):
            o = empty((heads, queries, width), dt)
            ctx.sdpa(qd, kd, vd, o, dt, heads, 1, queries, keys, width, strides, mask=dev(mask),
                     mask_heads=mask_heads, mask_rows=mask.shape[1])
            outs.append(host(o))
        np.testing.assert_array_equal(outs[0], outs[1])
        np.testing.assert_array_equal(outs[1], outs[2])
        expected = kat.attention_mask_expected(stored(q, dt), stored(k, dt), stored(v, dt), keys, mask_heads, shift)
        limit = {E.FP32: 3e-6, E.FP16: 4e-3, E.BF16: 3e-2}[dt]
        assert np.max(np.abs(outs[1] - expected)) < limit


def test_attention_accuracy_probe(ctx):
    # probes/attention_accuracy_probe.cpp: 4160 keys (4128 visible); a constant V
    # column must stay 1 within 5e-7; max error 3e-6 and nrmse 5e-7 vs FP64.
    q, k, v, mask, expected, _ = kat.attention_accuracy_case()
    H, Sq, d = q.shape
    Sk = k.shape[1]
    o = empty(q.shape)
    strides = (Sq * d, d, Sk * d, d, Sk * d, d, Sq * d, d)
    ctx.sdpa(dev(q), dev(k), dev(v), o, E.FP32, H, H, Sq, Sk, d, strides, mask=dev(mask), mask_heads=1,
             mask_rows=Sq)
    g = kat.attention_accuracy_gate(host(o), expected)
    assert g["passed"], g


@pytest.mark.parametrize("dt", [E.FP32, E.FP16, E.BF16], ids=lambda d: NAMES[d])
def test_sdpa_full_size_rows_against_oracle(ctx, dt):
    # SDPA alone at S=4160, 32 heads x 128, last 24 text keys padded; token-major
    # [S][4096] layout as the block uses it. Rows checked: the first query tile,
    # a middle one and the partial last tile, all heads.
    S, H, d, valid = 4160, 32, 128, 4136
    q = O.normal((S, H * d), 2)
    k = O.normal((S, H * d), 3)
    v = O.normal((S, H * d), 4)
    qd, kd, vd = dev(q, dt), dev(k, dt), dev(v, dt)
    o = empty((S, H * d), dt)
    strides = (d, H * d, d, H * d, d, H * d, d, H * d)
    ctx.sdpa(qd, kd, vd, o, dt, H, H, S, S, d, strides, valid_keys=valid)
    out = host(o).reshape(S, H, d).transpose(1, 0, 2)
    qs, ks, vs = (stored(t, dt).reshape(S, H, d).transpose(1, 0, 2).copy() for t in (q, k, v))
    mask = np.zeros(S, np.float32)
    mask[valid:] = -1e30
    # Rows 2240..2303 are the last two waves of their 128-query workgroup.
    for r0, r1 in ((0, 64), (2048, 2112), (2240, 2304), (4096, 4160)):
        ref = O.sdpa(qs, ks, vs, mask=mask, q_range=(r0, r1))[:, r0:r1]
        got = out[:, r0:r1]
        if dt == E.FP32:
            m = kat.fp32_block_rule(got, ref)
            assert m["passed"] and m["nrmse"] < 1e-6, m
        else:
            g = kat.gate(got, ref, *kat.BLOCK_GATES[NAMES[dt]])
            assert g["passed"], g


@pytest.mark.parametrize("dt", [E.FP16, E.BF16], ids=lambda d: NAMES[d])
@pytest.mark.parametrize("S,H,valid", [(256, 2, 256), (512, 3, 500), (1280, 2, 1270), (456, 2, 456), (300, 1, 290),
                                         (1088, 2, 1060)])
def test_sdpa_full_tiles_and_remainder(ctx, dt, S, H, valid):
    # Unmasked attention at lengths around the kernel's workgroup tiles: whole
    # 256-query tiles (the 8-wave form: 256, 512, 1280), 128-query tiles with a partial
    # last tile of 72 / 44 / 64 queries (split along the keys into parts that a second
    # launch merges; its waves past the last query only load and keep the barriers),
    # and valid-key counts that are not multiples of 64. Every row of every head is
    # compared with the oracle.
    d = 128
    q = O.normal((S, H * d), 21)
    k = O.normal((S, H * d), 22)
    v = O.normal((S, H * d), 23)
    o = empty((S, H * d), dt)
    strides = (d, H * d, d, H * d, d, H * d, d, H * d)
    ctx.sdpa(dev(q, dt), dev(k, dt), dev(v, dt), o, dt, H, H, S, S, d, strides, valid_keys=valid)
    out = host(o).reshape(S, H, d).transpose(1, 0, 2)
    qs, ks, vs = (stored(t, dt).reshape(S, H, d).transpose(1, 0, 2).copy() for t in (q, k, v))
    mask = np.zeros(S, np.float32)
    mask[valid:] = -1e30
    ref = O.sdpa(qs, ks, vs, mask=mask)
    g = kat.gate(out, ref, *kat.BLOCK_GATES[NAMES[dt]])
    assert g["passed"], g


@pytest.mark.parametrize("dt", ALL_DT, ids=lambda d: NAMES[d])
def test_qk_norm_rope_against_oracle(ctx, dt):
    S, H = 70, 3
    x = O.normal((S, 3 * H * 128), 5)
    gamma = O.normal((128,), 6, mean=1.0, std=0.1)
    ang = O.normal((S, 128), 7)
    cos, sin = np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)
    xd = dev(x, dt)
    ctx.qk_norm_rope(xd, dt, S, H, 3 * H * 128, dev(gamma), dev(cos), dev(sin))
    got = host(xd)
    xs = stored(x, dt)
    ref = xs.copy()
    for h in range(H):
        sl = xs[:, h * 128:(h + 1) * 128]
        ref[:, h * 128:(h + 1) * 128] = O.rope_rows(O.rmsnorm(sl, gamma), cos, sin)
    tol = {E.FP32: 2e-6, E.FP16: 4e-3, E.BF16: 3e-2}[dt]
    assert np.max(np.abs(got - ref)) <= tol * max(1.0, float(np.abs(ref).max()))
    # Columns outside the first H heads (the V block) are untouched.
    np.testing.assert_array_equal(got[:, H * 128:], xs[:, H * 128:])


@pytest.mark.slow
@pytest.mark.parametrize("dt", [E.FP32, E.FP16, E.BF16], ids=lambda d: NAMES[d])
def test_sdpa_config1_every_row_against_oracle(ctx, dt):
    # The standalone SDPA workload at full size: 32 heads x 128, S = 4160 (4096 image
    # tokens + a 64-token text bucket whose last 24 keys are padding), Q/K/V ~ N(0,1), scale
    # 1/sqrt(128), head-major [32][S][128]. Every query row of every head is compared with
    # the oracle (FP64 sums), so the full query tiles, both rounds of them and the key-split
    # partial last tile are all covered.
    S, H, d, valid = 4160, 32, 128, 4136
    q = O.normal((H, S, d), 2)
    k = O.normal((H, S, d), 3)
    v = O.normal((H, S, d), 4)
    o = empty((H, S, d), dt)
    strides = (S * d, d, S * d, d, S * d, d, S * d, d)
    ctx.sdpa(dev(q, dt), dev(k, dt), dev(v, dt), o, dt, H, H, S, S, d, strides, valid_keys=valid)
    got = host(o)
    mask = np.zeros(S, np.float32)
    mask[valid:] = -1e30
    ref = O.sdpa(stored(q, dt), stored(k, dt), stored(v, dt), mask=mask)
    if dt == E.FP32:
        m = kat.fp32_block_rule(got, ref)
        assert m["passed"] and m["nrmse"] < 1e-6, m
    else:
        g = kat.gate(got, ref, *kat.BLOCK_GATES[NAMES[dt]])
        assert g["passed"], g
        # Per-row error bound as well (the gate's atol + rtol max|ref|), so that a few wrong
        # rows cannot hide in the norm.
        atol, rtol, _ = kat.BLOCK_GATES[NAMES[dt]]
        row_err = np.abs(got - ref).max(axis=2)
        assert float(row_err.max()) <= atol + rtol * float(np.abs(ref).max()), float(row_err.max())


def test_euler_and_finite_contracts(ctx):
    # src/latent_ops.cpp:72-92 and tests/test_latent_contract.cpp.
    x = O.normal((128, 5, 3), 9)
    v = O.normal((128, 5, 3), 10)
    xd, vd, out = dev(x), dev(v), empty(x.shape)
    # Each delta of the 8-step turbo schedule (none a power of two): x + (delta * v) rounded
    # twice, bitwise the oracle's -ffp-contract=off product and sum. A fused multiply-add
    # (one rounding) gives different bits for some elements at these deltas, so the test
    # sees a contraction.
    sig, _ = O.flow_schedule_turbo(8)
    contraction_visible = False
    for i in range(8):
        delta = np.float32(sig[i + 1] - sig[i])
        ctx.euler_step(xd, vd, float(delta), x.size, out)
        ref = O.euler_step(x, v, delta)
        np.testing.assert_array_equal(host(out), ref)
        fused = (x.astype(np.float64) + np.float64(delta) * v.astype(np.float64)).astype(np.float32)
        contraction_visible |= bool(np.any(fused != ref))
    assert contraction_visible
    ctx.euler_step(xd, vd, -0.0625, x.size, out)
    np.testing.assert_array_equal(host(out), O.euler_step(x, v, -0.0625))
    for bad in (0.0, 0.5, -1.5, float("nan")):
        with pytest.raises(E.ErnieError):
            ctx.euler_step(xd, vd, bad, x.size, out)
    ones = dev(np.ones((128, 15), np.float32))
    ctx.euler_step(ones, ones, -1.0, 128 * 15, ones)  # aliased consume-and-replace
    assert np.all(host(ones) == 0.0)
    assert ctx.finite(xd, x.size)
    for bad in (float("inf"), float("nan")):
        y = x.copy()
        y[42, 2, 1] = bad
        assert not ctx.finite(dev(y), y.size)


def test_query_rows_compatibility(ctx):
    for rows in (128, 64, 32, 16):
        ctx.call("set_attention_query_rows", rows)
    with pytest.raises(E.ErnieError):
        ctx.call("set_attention_query_rows", 48)
    assert ctx.L.ernie_hip_attention_internal_submissions(ctx.ctx) == 0


@pytest.mark.parametrize("d,sq,sk", [(128, 130, 65), (40, 33, 129), (127, 1, 64)])
def test_sdpa_fp32_split_products_and_infinities(ctx, d, sq, sk):
    # Tile edges of queries and keys, odd head sizes. Each score is a sum of d products and
    # each output of sk, in FP32 or better; scores lie within 8, so exp2 passes at most 8
    # times their error on. In the 2-norm 2e-7 to 3e-7 of the result were measured; without
    # one of the six partial products it is 1.9e-6 and more. With an infinite value in one
    # column of V the others keep theirs. (Not in the last key: the keys that fill up the
    # last tile repeat it with probability zero, and zero times infinity is NaN, in the
    # FP32 products too.)
    q, k, v = O.normal((2, sq, d), 7), O.normal((2, sk, d), 8), O.normal((2, sk, d), 9)
    strides = (sq * d, d, sk * d, d, sk * d, d, sq * d, d)

    def run(v):
        out = empty((2, sq, d)).fill_(float("nan"))
        ctx.sdpa(dev(q), dev(k), dev(v), out, E.FP32, 2, 2, sq, sk, d, strides)
        return host(out)

    ref = sdpa_reference(q, k, v)
    bound = 8 * (d + sk) * 2.0**-24 * np.abs(v).max()
    got = run(v)
    assert np.abs(got - ref).max() <= bound
    assert np.linalg.norm(got - ref) <= 1e-6 * np.linalg.norm(ref)
    v = v.copy()
    v[1, sk - 2, d - 1] = np.inf
    got = run(v)
    assert np.all(np.isposinf(got[1, :, d - 1]))
    got[1, :, d - 1] = ref[1, :, d - 1]
    assert np.abs(got - ref).max() <= bound


def sdpa_reference(q, k, v):
    s = np.einsum("hqd,hkd->hqk", q.astype(np.float64), k.astype(np.float64)) / np.sqrt(q.shape[-1])
    p = np.exp(s - s.max(-1, keepdims=True))
    return np.einsum("hqk,hkd->hqd", p / p.sum(-1, keepdims=True), v.astype(np.float64))


@pytest.mark.parametrize("sq,sk,sv,scale", [(1e-36, 1e36, 1.0, 1.0), (1e36, 1e-36, 1e-36, 1.0), (1.0, 1.0, 1e-37, 1.0),
                                            (1e-20, 1e20, 1e25, 1.0), (1e15, 1e15, 1.0, 1e-30)])
def test_sdpa_fp32_small_magnitudes(ctx, sq, sk, sv, scale):
    # Queries, keys, values and a scale near the ends of FP32: the relative error is that of
    # values near 1 (4e-7 measured), where parts of BF16 subnormals would give 2.6e-5 and more.
    n, d = 130, 128
    q, k, v = (O.normal((2, n, d), i) * np.float32(x) for i, x in ((7, sq), (8, sk), (9, sv)))
    out = empty((2, n, d)).fill_(float("nan"))
    st = (n * d, d) * 4
    ctx.sdpa(dev(q), dev(k), dev(v), out, E.FP32, 2, 2, n, n, d, st, scale=scale / math.sqrt(d))
    ref = sdpa_reference(q.astype(np.float64) * scale, k, v)
    assert np.linalg.norm(host(out) - ref) <= 2e-6 * np.linalg.norm(ref)


def test_sdpa_fp32_small_probabilities(ctx):
    # A first key with all the weight and no value, others with probabilities of about 1e-37
    # and values of 1e30. A score near -120 in log2 units is rounded to 2^-18 of a unit
    # and scaled and subtracted once each: 1e-5 of a probability at most; parts that end at
    # 2^-133 would lose 2^-134 / 2^-123, 5e-4 of it.
    n, d = 70, 64
    q, k, v = np.zeros((1, 5, d), np.float32), np.zeros((1, n, d), np.float32), np.zeros((1, n, d), np.float32)
    q[:, :, 0] = 1
    k[0, 1:, 0] = -8 * np.linspace(84.5, 86.5, n - 1)
    v[0, 1:] = np.abs(O.normal((n - 1, d), 9)) * np.float32(1e30)
    out = empty((1, 5, d)).fill_(float("nan"))
    ctx.sdpa(dev(q), dev(k), dev(v), out, E.FP32, 1, 1, 5, n, d, (5 * d, d, n * d, d, n * d, d, 5 * d, d))
    ref = sdpa_reference(q, k, v)
    assert np.abs(host(out) - ref).max() <= 2e-5 * np.abs(ref).max()


def test_sdpa_fp32_fully_masked_row(ctx):
    # A query with every key masked out has no result (0 / 0), and does not send the 127
    # others of its workgroup to the FP32 matrix cores: their bits stay the same.
    n, d = 130, 128
    q, k, v = (dev(O.normal((1, n, d), i)) for i in (7, 8, 9))
    mask = O.normal((n, n), 10)
    outs = []
    for _ in range(2):
        out = empty((1, n, d)).fill_(0)
        ctx.sdpa(q, k, v, out, E.FP32, 1, 1, n, n, d, (n * d, d) * 4, mask=dev(mask), mask_heads=1, mask_rows=n)
        outs.append(host(out))
        mask[5] = -np.inf
    assert np.all(np.isnan(outs[1][0, 5]))
    rest = np.delete(np.arange(n), 5)
    assert np.array_equal(outs[0][0, rest], outs[1][0, rest])
