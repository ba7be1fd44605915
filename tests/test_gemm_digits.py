"""The digit-row projections (csrc/gemm_digits.hip): the digits themselves, and every
tile and epilogue at its edges, against 64-bit evaluations.

Bounds: a digit row is x to 2^-30 of its largest element, and the dot products are exact;
what is left are at most ten fp32 roundings of sums of the digits' size, so an output is
within 10 * 2^-24 of sum |w| |x| * scale plus that fixed-point step, 2^-30 max |x| sum |w| *
scale. Rows marked wide are sums of exact products in fp32, as the general W8A32 projection's
are: its error against 64 bits, on the same inputs, is their yardstick."""
from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _digits(x, dev):
    from qwenasr_amd import kernels as K

    rows, cols = x.shape
    dg = torch.empty(4 * rows * cols, dtype=torch.int8, device=dev)
    ex = torch.empty(rows, dtype=torch.int32, device=dev)
    K.digit_rows(dg, ex, x.reshape(-1), rows, cols)
    return dg, ex


def _weight(n, k, dev, seed):
    from qwenasr_amd import kernels as K

    g = torch.Generator(device=dev).manual_seed(seed)
    w = torch.randint(-128, 128, (n * k,), generator=g, device=dev, dtype=torch.int32).to(torch.int8)
    return K.QuantWeight(w, torch.rand(n, generator=g, device=dev) + 0.5, n, k)


def _product(x, w):
    q = w.data.view(w.out_dim, w.in_dim).double().cpu()
    s = w.scales.double().cpu()
    x = x.double().cpu()
    step = 2.0 ** -30 * x.abs().amax(-1, keepdim=True) * q.abs().sum(-1)
    return (x @ q.t()) * s, ((x.abs() @ q.abs().t()) * (10 * 2.0 ** -24) + step) * s + 1e-30


def _near(got, ref, bound):
    assert ((got.double().cpu() - ref).abs() <= bound).all()


@pytest.mark.parametrize("cols", [4, 1000, 1024, 1028, 3072, 5000, 8192])
def test_digit_rows_give_the_row_back(dev, cols):
    r = np.random.default_rng([91, cols])
    x = r.standard_normal((9, cols)).astype(np.float32)
    x[1] *= 1e30
    x[2] *= 1e-42          # subnormal
    x[3] = 0.0
    x[4, 0], x[5, -1], x[6, cols // 2] = np.inf, -np.inf, np.nan
    x[7] = np.round(x[7] * 1000) * np.float32(2.0 ** 20)  # exact multiples of a power of two
    x[8, 0] = 1e6          # an outlier
    dg, ex = (t.cpu().numpy() for t in _digits(torch.from_numpy(x).to(dev), dev))
    value = (dg.reshape(4, 9, cols).astype(np.float64) * 256.0 ** np.arange(4)[:, None, None]).sum(0)
    for i in (0, 1, 2, 3, 7, 8):
        got = np.ldexp(value[i], ex[i])
        step = np.abs(x[i]).max().astype(np.float64) * 2.0 ** -29
        assert np.abs(got - x[i]).max() <= step / 2
    np.testing.assert_array_equal(np.ldexp(value[7], ex[7]), x[7])
    assert (ex[4:7] == -0x40000000).all() and not dg.reshape(4, 9, cols)[:, 4:7].any()


@pytest.mark.parametrize("T,K_,N", [(1, 256, 4), (2, 1024, 1024), (31, 512, 36), (32, 1024, 132), (33, 2048, 1000),
                                    (65, 1024, 4096), (70, 512, 33028), (300, 1024, 12292), (1000, 3072, 1028)])
def test_linear_digits(dev, T, K_, N):
    from qwenasr_amd import kernels as K

    x = torch.randn(T, K_, device=dev, generator=torch.Generator(device=dev).manual_seed(T + N))
    x[:, 3] *= 100.0
    x[T // 2] *= 1e-20
    w = _weight(N, K_, dev, N)
    dg, ex = _digits(x, dev)
    y = torch.full((T * N,), 9.0, device=dev)
    K.linear_digits_int8([y], [w], dg, ex, T, K_)
    ref, bound = _product(x, w)
    _near(y.view(T, N), ref, bound)
    for parts in (2, 3, 4):
        if K_ % (256 * parts) == 0:
            p = torch.full((parts * T * N,), 9.0, device=dev)
            K.linear_digits_int8([p], [w], dg, ex, T, K_, parts=parts)
            _near(p.view(parts, T, N).double().sum(0), ref, bound)
    z = torch.ones(T * N, device=dev)
    K.linear_digits_int8([z], [w], dg, ex, T, K_, residual=True)
    assert torch.equal(z, y + 1.0)


def test_three_matrices_and_a_bad_row(dev):
    from qwenasr_amd import kernels as K

    T, K_, dims = 40, 1024, (2048, 1024, 1028)
    x = torch.randn(T, K_, device=dev)
    x[5, 17], x[39, 0] = float("inf"), float("nan")
    ws = [_weight(n, K_, dev, n) for n in dims]
    dg, ex = _digits(x, dev)
    ys = [torch.empty(T * n, device=dev) for n in dims]
    K.linear_digits_int8(ys, ws, dg, ex, T, K_)
    good = [i for i in range(T) if i not in (5, 39)]
    for y, w in zip(ys, ws):
        got = y.view(T, -1)
        assert got[[5, 39]].isnan().all()
        ref, bound = _product(x[good], w)
        _near(got[good], ref, bound)


@pytest.mark.parametrize("T,H,inter", [(3, 1024, 3072), (40, 256, 18), (70, 1024, 8200), (600, 2048, 6144)])
def test_gate_up_swiglu_digits(dev, T, H, inter):
    from qwenasr_amd import kernels as K

    w = _weight(2 * inter, H, dev, inter)
    w.scales.mul_(2e-4)
    x = torch.randn(T, H, device=dev)
    dg, ex = _digits(x, dev)
    gu = torch.empty(T * 2 * inter, device=dev)
    K.linear_digits_int8([gu], [w], dg, ex, T, H)
    out, ref = (torch.full((T * inter,), 9.0, device=dev) for _ in range(2))
    K.gate_up_swiglu_digits_int8(out, w, dg, ex, T, H, inter, prefill=True)
    K.swiglu_multiply(ref, gu, T, inter)  # the tiles' K groups may differ: a last bit of the gates and ups
    torch.testing.assert_close(out, ref, rtol=1e-6, atol=1e-6)
    K.gate_up_swiglu_digits_int8(out, w, dg, ex, T, H, inter)
    g, u = gu.view(T, inter, 2).double().unbind(-1)
    torch.testing.assert_close(out.view(T, inter).double(), g / (1 + (-g).exp()) * u, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("T,start,rows", [(5, 0, 5), (33, 7, 64), (40, 24, 64), (200, 100, 300)])
def test_qkv_heads_digits_equals_the_two_launches(dev, T, start, rows):
    """The projections followed by head_rms_norm_rope_kv (their tiles may add K in another
    number of parts); rows that do not fit the cache are refused."""
    from qwenasr_amd import kernels as K

    H, nq, nk, hd = 1024, 16, 8, 128
    ws = [_weight(n * hd, H, dev, n + i) for i, n in enumerate((nq, nk, nk))]
    for w in ws:
        w.scales.mul_(1e-3)
    dg, ex = _digits(torch.randn(T, H, device=dev), dev)
    qw, kw = torch.rand(hd, device=dev) + 0.5, torch.rand(hd, device=dev) + 0.5
    rope = K.RopeCache(dev)
    rope.ensure(start + T, hd, 1e6)
    q1, k1, v1 = (torch.empty(T * n * hd, device=dev) for n in (nq, nk, nk))
    caches = [torch.full((rows * nk * hd,), 5.0, device=dev) for _ in range(4)]
    q2 = torch.empty_like(q1)
    K.qkv_heads_digits_int8(q2, caches[2], caches[3], rows, *ws, dg, ex, T, H, nq, nk, hd, qw, kw, rope, start, 1e-6)
    with pytest.raises(K.QasrError):
        K.qkv_heads_digits_int8(q2, caches[2], caches[3], start + T - 1, *ws, dg, ex, T, H, nq, nk, hd, qw, kw, rope,
                                start, 1e-6)
    K.linear_digits_int8([q1, k1, v1], ws, dg, ex, T, H)
    K.head_rms_norm_rope_kv(q1, k1, v1, qw, kw, rope, None, start, T, nq, nk, hd, 1e-6, caches[0], caches[1], rows)
    for a, b in ((q1, q2), (caches[0], caches[2]), (caches[1], caches[3])):
        torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-5)


def test_add_rms_norm_digits(dev):
    from qwenasr_amd import kernels as K

    for rows, cols in ((1, 1024), (7, 2048), (3, 1500), (2, 8192)):
        x, d = torch.randn(rows * cols, device=dev), torch.randn(rows * cols, device=dev)
        g = torch.rand(cols, device=dev) + 0.5
        for delta in (None, d):
            a, b = x.clone(), x.clone()
            xn, ref = torch.empty_like(x), torch.empty_like(x)
            dg = torch.empty(4 * rows * cols, dtype=torch.int8, device=dev)
            ex = torch.empty(rows, dtype=torch.int32, device=dev)
            K.add_rms_norm_digits(a, delta, g, xn, dg, ex, rows, cols, 1e-6)
            if delta is None:
                K.rms_norm(ref, b, g, rows, cols, 1e-6)
            else:
                K.add_rms_norm(b, delta, g, ref, rows, cols, 1e-6)
            assert torch.equal(a, b)
            if delta is not None:  # slices that add up to delta exactly
                c, dg3, ex3 = x.clone(), torch.empty_like(dg), torch.empty_like(ex)
                half = torch.cat([delta * 0.5, delta * 0.25, delta * 0.25])
                K.add_rms_norm_digits(c, half, g, None, dg3, ex3, rows, cols, 1e-6, 3)
                assert torch.equal(a, c) and torch.equal(dg, dg3) and torch.equal(ex, ex3)
            # each sums the squares through at most 42 additions (half of that in the row) and rounds 3 times
            torch.testing.assert_close(xn, ref, rtol=2 * 24 * 2.0 ** -24, atol=0)
            dg2, ex2 = _digits(xn.view(rows, cols), dev)
            assert torch.equal(dg, dg2) and torch.equal(ex, ex2)


@pytest.mark.parametrize("rows,K_,vocab", [(2, 1024, 4000), (7, 2048, 3004), (32, 1024, 33000), (40, 2048, 1000)])
def test_lm_head_rows_from_digits(dev, rows, K_, vocab):
    """Several rows with a workspace that holds their digits (the last one's does not, and
    takes the general projection): logits against 64 bits, the first largest wins."""
    from qwenasr_amd import kernels as K

    x = torch.randn(rows, K_, device=dev)
    w = _weight(vocab, K_, dev, rows)
    ws = torch.empty(8 * 37984 if vocab > 1000 else 4096, dtype=torch.uint8, device=dev)
    logits, idx = torch.empty(rows * vocab, device=dev), torch.empty(rows, dtype=torch.int32, device=dev)
    K.lm_head_int8_argmax(idx, logits, x.view(-1), w, rows, K_, vocab, ws)
    got = logits.view(rows, vocab)
    ref, bound = _product(x, w)
    _near(got, ref, bound if vocab > 1000 else 1e-5 * bound / (10 * 2.0 ** -24))
    assert torch.equal(idx.long(), got.argmax(-1))


OUTLIERS = (7, 100, 200)  # columns whose weights are 0 in the tests of wide rows


def _wide_case(T, K_, N, dev):
    """Rows that range too far for the digits (one or three elements far above the rest) among
    ordinary ones and ones just inside the line; the weights are 0 at those elements, so the
    outputs are sums of the small ones. Last rows: an infinity and a NaN."""
    x = torch.randn(T, K_, device=dev, generator=torch.Generator(device=dev).manual_seed(T + K_))
    x[1::5, 7] = 1e4
    x[2::5, 100] = -1e6
    x[3::5, 7], x[3::5, 100], x[3::5, 200] = 1e5, 1e5, -1e5
    x[4::5, 200] = 60.0  # at most 100 times the mean magnitude
    x[T - 2, 17], x[T - 1, 18] = float("-inf"), float("nan")
    w = _weight(N, K_, dev, N)
    w.data.view(N, K_)[:, list(OUTLIERS)] = 0
    mean = x.double().abs().mean(-1)
    wide = ~((x.double().abs().amax(-1) <= 128 * mean) & ~mean.isinf()) & ~mean.isnan()
    return x, w, wide


def _digits_wide(x, dev):
    from qwenasr_amd import kernels as K

    rows, cols = x.shape
    dg = torch.empty(4 * rows * cols, dtype=torch.int8, device=dev)
    ex = torch.empty(rows, dtype=torch.int32, device=dev)
    K.digit_rows(dg, ex, x.reshape(-1), rows, cols, wide=True)
    return dg, ex


def _error(got, ref):  # of each row, against 64 bits
    return (got.double() - ref).norm(dim=-1) / ref.norm(dim=-1)


def test_which_rows_are_marked(dev):
    x = torch.randn(7, 1024, device=dev)
    x[1] = 3e38                    # the sum of magnitudes overflows: marked
    x[2] = 0.0
    x[3, 1:] = 0.0                 # one element: 1024 times the mean
    x[4] *= 1e-42                  # subnormal, no outlier
    x[5] = 1.0
    x[5, 9] = 128 * 1023 / 896.0   # 128 times the mean, to rounding
    x[5, 9] *= 1.001
    x[6] = 1.0
    x[6, 9] = 128 * 1023 / 896.0 * 0.999
    _, ex = _digits_wide(x, dev)
    assert (ex == -0x40000001).tolist() == [False, True, False, True, False, True, False]


# one shape per tile (32 x 32, 64 x 32, 128 x 32, 256 x 64), ragged in rows and tokens, and a long sum
@pytest.mark.parametrize("T,K_,N", [(9, 512, 1028), (65, 1024, 4096), (70, 512, 33028), (300, 1024, 12292),
                                    (12, 6144, 2048)])
def test_wide_rows_keep_fp32_precision(dev, T, K_, N):
    from qwenasr_amd import kernels as K

    x, w, wide = _wide_case(T, K_, N, dev)
    dg, ex = _digits_wide(x, dev)
    assert ((ex == -0x40000001) == wide).all() and wide[1:T - 1:5].all() and not wide[4:T - 2:5].any()
    flat = x.reshape(-1)
    y, old = (torch.full((T * N,), 9.0, device=dev) for _ in range(2))
    K.linear_digits_int8([y], [w], dg, ex, T, K_, x=flat)
    K.linear_nobias_int8(old, flat, w.data, w.scales, T, K_, N)
    ref = (x.double() @ w.data.view(N, K_).double().t().contiguous()) * w.scales.double()
    fin = slice(0, T - 2)
    limit = 1.25 * _error(old.view(T, N)[fin], ref[fin])  # a quarter for another order of the sums
    assert (_error(y.view(T, N)[fin], ref[fin]) <= limit).all()
    for parts in (2, 3, 4):
        if K_ % (256 * parts) == 0:
            p = torch.full((parts * T * N,), 9.0, device=dev)
            K.linear_digits_int8([p], [w], dg, ex, T, K_, parts=parts, x=flat)
            assert (_error(p.view(parts, T, N).double().sum(0)[fin], ref[fin]) <= limit).all()
    z = torch.ones(T * N, device=dev)
    K.linear_digits_int8([z], [w], dg, ex, T, K_, residual=True, x=flat)
    assert torch.equal(z.view(T, N)[fin], (y + 1.0).view(T, N)[fin])
    # an infinity and a NaN travel as in fp32: NaN only where a weight of 0 meets the infinity
    got = y.view(T, N)[T - 2:]
    assert torch.equal(got.isnan(), ref[T - 2:].isnan()) and torch.equal(got[0].isinf(), ref[T - 2].isinf())
    keep = ~got[0].isnan()
    assert torch.equal(got[0][keep].double(), ref[T - 2][keep]) and got[1].isnan().all()
    # a NaN needs no floats; without them a marked row gives NaN
    assert int(ex[T - 1]) == -0x40000000
    wide[T - 1] = True
    K.linear_digits_int8([y], [w], dg, ex, T, K_)
    assert torch.equal(y.view(T, N).isnan().all(-1), wide) and torch.equal(y.view(T, N).isnan().any(-1), wide)


def test_wide_rows_in_the_other_epilogues(dev):
    """gate/up + SwiGLU and q/k/v + heads, whose marked rows equal the plain projection's followed
    by the separate launches (their tiles may add K in another number of parts)."""
    from qwenasr_amd import kernels as K

    T, H, inter, nq, nk, hd = 45, 1024, 3072, 16, 8, 128
    x, w, _ = _wide_case(T, H, 2 * inter, dev)
    x = x[:T - 2].contiguous()
    T -= 2
    flat = x.view(-1)
    w.scales.mul_(2e-4)
    dg, ex = _digits_wide(x, dev)
    gu, out, ref = (torch.empty(T * n, device=dev) for n in (2 * inter, inter, inter))
    K.linear_digits_int8([gu], [w], dg, ex, T, H, x=flat)
    K.swiglu_multiply(ref, gu, T, inter)
    K.gate_up_swiglu_digits_int8(out, w, dg, ex, T, H, inter, prefill=True, x=flat)
    torch.testing.assert_close(out, ref, rtol=1e-6, atol=1e-6)
    K.gate_up_swiglu_digits_int8(out, w, dg, ex, T, H, inter, x=flat)
    g, u = gu.view(T, inter, 2).double().unbind(-1)
    torch.testing.assert_close(out.view(T, inter).double(), g / (1 + (-g).exp()) * u, rtol=1e-6, atol=1e-6)
    ws = [_weight(n * hd, H, dev, n + i) for i, n in enumerate((nq, nk, nk))]
    for m in ws:
        m.scales.mul_(1e-3)
        m.data.view(-1, H)[:, list(OUTLIERS)] = 0
    qw, kw = torch.rand(hd, device=dev) + 0.5, torch.rand(hd, device=dev) + 0.5
    rope = K.RopeCache(dev)
    rope.ensure(T, hd, 1e6)
    q1, k1, v1 = (torch.empty(T * n * hd, device=dev) for n in (nq, nk, nk))
    caches = [torch.full((T * nk * hd,), 5.0, device=dev) for _ in range(4)]
    q2 = torch.empty_like(q1)
    K.qkv_heads_digits_int8(q2, caches[2], caches[3], T, *ws, dg, ex, T, H, nq, nk, hd, qw, kw, rope, 0, 1e-6, flat)
    K.linear_digits_int8([q1, k1, v1], ws, dg, ex, T, H, x=flat)
    K.head_rms_norm_rope_kv(q1, k1, v1, qw, kw, rope, None, 0, T, nq, nk, hd, 1e-6, caches[0], caches[1], T)
    for a, b in ((q1, q2), (caches[0], caches[2]), (caches[1], caches[3])):
        torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-5)


def test_add_rms_norm_digits_marks_wide_rows(dev):
    from qwenasr_amd import kernels as K

    for rows, cols in ((7, 1024), (6, 8192)):
        x = torch.randn(rows, cols, device=dev)
        x[2, 5], x[4, 1], x[5, 9] = 1e6, float("inf"), 30.0
        g = torch.rand(cols, device=dev) + 0.5
        a, b, c = (x.reshape(-1).clone() for _ in range(3))
        xn, own, plain = torch.empty_like(a), torch.full_like(a, 7.0), torch.empty_like(a)
        dg, dg2 = (torch.empty(4 * rows * cols, dtype=torch.int8, device=dev) for _ in range(2))
        ex, ex2, ex3 = (torch.empty(rows, dtype=torch.int32, device=dev) for _ in range(3))
        K.add_rms_norm_digits(a, None, g, plain, dg, ex, rows, cols, 1e-6)
        K.add_rms_norm_digits(b, None, g, xn, dg2, ex2, rows, cols, 1e-6, wide=True)
        K.add_rms_norm_digits(c, None, g, own, dg2, ex3, rows, cols, 1e-6, wide=True, all_rows=False)
        marked = [2]  # an infinity's row is normalised to NaN
        rest = [i for i in range(rows) if i not in marked]
        assert (ex2[marked] == -0x40000001).all() and int(ex2[4]) == -0x40000000
        assert torch.equal(ex2, ex3) and torch.equal(ex[rest], ex2[rest])
        assert torch.equal(dg.view(4, rows, cols)[:, rest], dg2.view(4, rows, cols)[:, rest])
        torch.testing.assert_close(xn, plain, rtol=0, atol=0, equal_nan=True)
        own = own.view(rows, cols)
        torch.testing.assert_close(own[marked], plain.view(rows, cols)[marked], rtol=0, atol=0, equal_nan=True)
        assert (own[rest] == 7.0).all()


@pytest.mark.parametrize("outlier", [1e4, 1e6])
def test_lm_head_rows_keep_fp32_precision_beside_an_outlier(dev, outlier):
    """With a workspace (digit rows) the logits are no further from 64 bits than without."""
    from qwenasr_amd import kernels as K

    rows, K_, vocab = 9, 2048, 4000
    x = torch.randn(rows, K_, device=dev, generator=torch.Generator(device=dev).manual_seed(5))
    x[::2, 7] = outlier
    w = _weight(vocab, K_, dev, 3)
    w.data.view(vocab, K_)[:, 7] = 0
    ref = (x.double() @ w.data.view(vocab, K_).double().t().contiguous()) * w.scales.double()
    idx, errors = torch.empty(rows, dtype=torch.int32, device=dev), []
    for ws in (torch.empty(1 << 20, dtype=torch.uint8, device=dev), None):
        logits = torch.empty(rows * vocab, device=dev)
        K.lm_head_int8_argmax(idx, logits, x.view(-1), w, rows, K_, vocab, ws)
        errors.append(_error(logits.view(rows, vocab), ref))
    assert (errors[0] <= 1.25 * errors[1]).all()


@pytest.mark.parametrize("rows", [2, 7])
def test_lm_head_row_with_an_infinity(dev, rows):
    """2 to 7 rows: an infinity gives infinite logits and the first positive one wins, as in fp32."""
    from qwenasr_amd import kernels as K

    K_, vocab = 1024, 3000
    x = torch.randn(rows, K_, device=dev)
    x[1, 3] = float("inf")
    w = _weight(vocab, K_, dev, 8)
    col = w.data.view(vocab, K_)[:, 3]
    col[col == 0] = -1
    idx, logits = torch.empty(rows, dtype=torch.int32, device=dev), torch.empty(rows * vocab, device=dev)
    ws = torch.empty(1 << 20, dtype=torch.uint8, device=dev)
    K.lm_head_int8_argmax(idx, logits, x.view(-1), w, rows, K_, vocab, ws)
    assert torch.equal(logits.view(rows, vocab)[1], torch.where(col > 0, float("inf"), float("-inf")))
    assert int(idx[1]) == int((col > 0).nonzero()[0])


@pytest.mark.parametrize("rows", [7, 8, 38])
def test_lm_head_workspace_for_rows(dev, rows):
    """A workspace asked for with the rows holds their digits (38 rows of 2048 do not fit the
    one-row workspace of this vocabulary): the digit projection's logits, bit for bit; one
    made for a row less gives the general projection's."""
    from qwenasr_amd import kernels as K

    K_, vocab = 2048, 4000
    x = torch.randn(rows, K_, device=dev)
    w = _weight(vocab, K_, dev, rows)
    dg, ex = _digits_wide(x, dev)
    digits, plain, logits = (torch.empty(rows * vocab, device=dev) for _ in range(3))
    idx = torch.empty(rows, dtype=torch.int32, device=dev)
    K.linear_digits_int8([digits], [w], dg, ex, rows, K_, x=x.view(-1))
    K.linear_nobias_int8(plain, x.view(-1), w.data, w.scales, rows, K_, vocab)
    assert not torch.equal(digits, plain)
    for have, want in ((rows, digits), (rows - 1, plain)):
        ws = K.lm_head_workspace(vocab, dev, have, K_)
        K.lm_head_int8_argmax(idx, logits, x.view(-1), w, rows, K_, vocab, ws)
        assert torch.equal(logits, want)
        assert torch.equal(idx.long(), logits.view(rows, vocab).argmax(-1))


def test_parts_worth_taking(dev):
    from qwenasr_amd import kernels as K

    assert K.linear_digits_parts(11, 2048, 1024) == 4 and K.linear_digits_parts(11, 3072, 1024) == 4
    assert K.linear_digits_parts(64, 6144, 2048) == 2 and K.linear_digits_parts(65, 2048, 2048) == 1
    assert K.linear_digits_parts(2, 512, 256) == 1 and K.linear_digits_parts(2, 1024, 256) == 2


def test_refusals(dev):
    from qwenasr_amd import _lib, kernels as K

    x = torch.zeros(4 * 512, device=dev)
    dg, ex = torch.zeros(4 * 4 * 512, dtype=torch.int8, device=dev), torch.zeros(4, dtype=torch.int32, device=dev)
    w = _weight(8, 512, dev, 1)
    y = torch.zeros(64, device=dev)
    for call in (lambda: K.linear_digits_int8([y], [w], dg, ex, 4, 384),               # in_dim not a multiple of 256
                 lambda: K.linear_digits_int8([y], [K.QuantWeight(w.data, w.scales, 6, 512)], dg, ex, 4, 512),
                 lambda: K.linear_digits_int8([y], [w], dg, ex, 1, 512, parts=4),
                 lambda: K.digit_rows(dg, ex, x, 4, 510),
                 lambda: K.digit_rows(dg[1:], ex, x, 1, 512)):
        with pytest.raises(K.QasrError) as e:
            call()
        assert e.value.code == _lib.QASR_ERR_UNSUPPORTED
    with pytest.raises(IndexError):
        K.linear_digits_int8([y[:31]], [w], dg, ex, 4, 512)
