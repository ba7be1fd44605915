"""How the decode attentions cut their keys: one token's 64-key splits at every
edge of a tile, and a small batch's shorter chunks (a larger workspace), against
the oracle at the fp32 tolerance of the other attention tests."""
from __future__ import annotations

import numpy as np
import pytest

import oracle

torch = pytest.importorskip("torch")

NQ, NK, HD = 16, 8, 128
KV = NK * HD


@pytest.mark.gpu
@pytest.mark.parametrize("pos", [0, 1, 15, 16, 62, 63, 64, 65, 127, 128, 191, 403, 4095])
def test_one_token_split_edges(dev, pos):
    from qwenasr_amd import kernels as K

    r = np.random.default_rng([81, pos])
    q = r.standard_normal(NQ * HD).astype(np.float32)
    k, v = (r.standard_normal((pos + 1) * KV).astype(np.float32) for _ in range(2))
    d = lambda a: torch.from_numpy(a).to(dev)  # noqa: E731
    out = torch.full((NQ * HD,), 9.0, device=dev)
    K.causal_attention_split(out, d(q), d(k), d(v), 1, pos + 1, NQ, NK, HD, HD ** -0.5, pos,
                             K.attention_workspace(1, NQ, HD, dev))
    ref = oracle.causal_attention(q, k, v, 1, pos + 1, NQ, NK, HD, HD ** -0.5, pos)
    np.testing.assert_allclose(out.cpu().numpy(), ref, rtol=1e-5, atol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("nq,nk,hd", [(8, 1, 128), (8, 8, 128), (16, 4, 128), (4, 4, 64), (8, 1, 64), (8, 2, 64)])
def test_one_token_split_other_heads(dev, nq, nk, hd):
    from qwenasr_amd import kernels as K

    kv = nk * hd
    for pos in (0, 5, 63, 64, 130, 255):
        r = np.random.default_rng([85, pos, nq])
        q = r.standard_normal(nq * hd).astype(np.float32)
        k, v = (r.standard_normal((pos + 1) * kv).astype(np.float32) for _ in range(2))
        d = lambda a: torch.from_numpy(a).to(dev)  # noqa: E731
        out = torch.full((nq * hd,), 9.0, device=dev)
        K.causal_attention_split(out, d(q), d(k), d(v), 1, pos + 1, nq, nk, hd, hd ** -0.5, pos,
                                 K.attention_workspace(1, nq, hd, dev))
        ref = oracle.causal_attention(q, k, v, 1, pos + 1, nq, nk, hd, hd ** -0.5, pos)
        np.testing.assert_allclose(out.cpu().numpy(), ref, rtol=1e-5, atol=1e-5, err_msg=f"pos {pos}")


@pytest.mark.gpu
@pytest.mark.parametrize("T,start,nq,nk", [(77, 610, 16, 8), (128, 385, 16, 8), (16, 1000, 16, 8), (9, 3000, 16, 8),
                                           (33, 400, 8, 8), (40, 2000, 16, 4), (20, 4200, 16, 2), (77, 179, 16, 8)])
def test_prefill_key_splits(dev, T, start, nq, nk):
    """A chunk over a cache in key splits (a last one with fewer tiles, rows whose causal
    range ends before it) against the unsplit kernel; a workspace too small for them
    gives the unsplit kernel's result bit for bit."""
    from qwenasr_amd import kernels as K

    n, kv = T + start, nk * HD
    r = np.random.default_rng([83, T, start])
    q = torch.from_numpy(r.standard_normal(T * nq * HD).astype(np.float32)).to(dev)
    k, v = (torch.from_numpy(r.standard_normal(n * kv).astype(np.float32)).to(dev) for _ in range(2))
    whole, out = torch.empty_like(q), torch.full_like(q, 9.0)
    K.causal_attention(whole, q, k, v, T, n, nq, nk, HD, HD ** -0.5, start)
    ws = torch.full((512 * 16 * (HD + 2),), float("nan"), device=dev)
    K.causal_attention_split(out, q, k, v, T, n, nq, nk, HD, HD ** -0.5, start, ws)
    torch.testing.assert_close(out, whole, rtol=1e-5, atol=1e-5)
    K.causal_attention_split(out, q, k, v, T, n, nq, nk, HD, HD ** -0.5, start, ws[:64])
    assert torch.equal(out, whole)
    rows = [0, T // 2, T - 1]
    for i in rows:
        ref = oracle.causal_attention(q.view(T, -1)[i].cpu().numpy(), k.cpu().numpy()[:(start + i + 1) * kv],
                                      v.cpu().numpy()[:(start + i + 1) * kv], 1, start + i + 1, nq, nk, HD, HD ** -0.5,
                                      start + i)
        np.testing.assert_allclose(whole.view(T, -1)[i].cpu().numpy(), ref, rtol=1e-5, atol=1e-5)


def test_split_workspace_sizes():
    from qwenasr_amd import _lib

    split = _lib.lib().qasr_batched_decode_attention_split_workspace_floats
    whole = _lib.lib().qasr_batched_decode_attention_workspace_floats
    assert split(11, 16, 128, 768) == 11 * 16 * 12 * 130   # chunks of 64 keys
    assert split(30, 16, 128, 1500) == 30 * 16 * 8 * 130   # of 192
    assert split(1, 16, 128, 64) == 0                      # one chunk
    assert split(1, 16, 128, 10000) == 16 * 53 * 130       # of 192: at most 64 chunks
    for b, h, rows in ((64, 16, 1024), (256, 16, 2048), (1 << 40, 16, 2048), (3, 1 << 62, 100), (1, 16, 40000),
                       (2, 16, 0), (2, 16, 1 << 31)):
        assert split(b, h, 128, rows) == whole(b, h, 128, rows)
    for b in (1, 2, 7, 20, 63, 64, 200):
        for rows in (1, 65, 300, 513, 2048, 32768, 32769):
            assert split(b, 16, 128, rows) >= whole(b, 16, 128, rows)


@pytest.mark.gpu
@pytest.mark.parametrize("nq,nk,hd,rows", [(16, 8, 128, 130), (16, 8, 128, 768), (8, 8, 128, 300), (16, 4, 64, 500)])
def test_short_chunks(dev, nq, nk, hd, rows):
    from qwenasr_amd import _lib, kernels as K

    kv, pos = nk * hd, [0, 63, 64, rows - 1, rows // 2, rows]
    B = len(pos)
    r = np.random.default_rng([82, nq, rows])
    q = r.standard_normal((B, nq * hd)).astype(np.float32)
    k, v = (r.standard_normal((B, rows, kv)).astype(np.float32) for _ in range(2))
    d = lambda a: torch.from_numpy(a).to(dev).reshape(-1)  # noqa: E731
    p = d(np.array(pos, np.int32))
    ws = K.batched_decode_split_workspace(B, nq, hd, rows, dev)
    assert ws.numel() > _lib.lib().qasr_batched_decode_attention_workspace_floats(B, nq, hd, rows)
    order = torch.empty(2 * B, dtype=torch.int32, device=dev)
    K.batched_decode_order(order, p, B, rows)
    out, oq = torch.full((B * nq * hd,), 9.0, device=dev), torch.empty(B * nq * hd, dtype=torch.int8, device=dev)
    osc = torch.empty(B, device=dev)
    dq, dk, dv = d(q), d(k), d(v)
    for quant in (False, True):
        ws.fill_(7.0)
        K.batched_decode_attention(out, dq, dk, dv, rows, p, B, nq, nk, hd, hd ** -0.5, ws, oq if quant else None,
                                   osc if quant else None, order)
        got = out.view(B, -1).cpu().numpy()
        assert np.isnan(got[-1]).all()  # a position outside the cache
        for m in range(B - 1):
            n = pos[m] + 1
            ref = oracle.causal_attention(q[m], k[m, :n].ravel(), v[m, :n].ravel(), 1, n, nq, nk, hd, hd ** -0.5, n - 1)
            np.testing.assert_allclose(got[m], ref, rtol=1e-5, atol=1e-5, err_msg=f"stream {m}")
    rq, rs = torch.empty_like(oq), torch.empty_like(osc)
    K.quantize_rows_i8(rq, rs, out, B, nq * hd)
    assert torch.equal(oq, rq) and torch.equal(osc, rs)


@pytest.mark.gpu
@pytest.mark.parametrize("pos,nq,nk,hd,out_dim", [(0, 16, 8, 128, 1024), (63, 16, 8, 128, 2048), (64, 16, 8, 128, 1000),
                                                  (403, 16, 8, 128, 1024), (511, 16, 8, 128, 8192),
                                                  (512, 16, 8, 128, 1024), (300, 8, 8, 128, 4100), (300, 4, 4, 64, 100)])
def test_decode_attention_linear_equals_the_two_calls(dev, pos, nq, nk, hd, out_dim):
    """Bit for bit decode_attention and the o projection: 1 to 8 splits merged by the
    projection, 9 (a merge launch), another head size (the two calls); rows past a
    multiple of a workgroup's."""
    from qwenasr_amd import kernels as K

    r = np.random.default_rng([84, pos, nq])
    d = lambda *s: torch.from_numpy(r.standard_normal(s).astype(np.float32).ravel()).to(dev)  # noqa: E731
    kv, qd, rows = nk * hd, nq * hd, pos + 3
    q, k, v, kc, vc = d(qd), d(kv), d(kv), d(rows * kv), d(rows * kv)
    qw, kw = d(hd), d(hd)
    w = K.QuantWeight(torch.from_numpy(r.integers(-127, 128, out_dim * qd).astype(np.int8)).to(dev), d(out_dim), out_dim,
                      qd)
    rope = K.RopeCache(dev)
    rope.ensure(pos + 1, hd, 1e6)
    got = []
    for fused in (True, False):
        out, y = torch.full((qd,), 9.0, device=dev), torch.full((out_dim,), 9.0, device=dev)
        ws = K.attention_workspace(1, nq, hd, dev).fill_(float("nan"))
        caches = kc.clone(), vc.clone()
        args = (q.clone(), k, v, qw, kw, rope, pos, nq, nk, hd, 1e-6, hd ** -0.5, *caches, rows, ws)
        if fused:
            K.decode_attention_linear_int8(y, out, *args, w, out_dim)
        else:
            K.decode_attention(out, *args)
            K.linear_nobias_int8(y, out, w.data, w.scales, 1, qd, out_dim)
        got.append((y, *caches))
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("pos", [0, 70, 511, 600])
def test_decode_attention_linear_takes_weights_of_any_alignment(dev, pos):
    """The o projection's weights and scales as views off 16-byte alignment: decode_attention
    followed by linear_nobias_int8, bit for bit; the decode step runs with them."""
    from qwenasr_amd import kernels as K

    nq, nk, hd, H, rows = 16, 8, 128, 1024, 640
    g = torch.Generator(device=dev).manual_seed(pos)
    r = lambda n: torch.randn(n, generator=g, device=dev)  # noqa: E731
    q, k, v, qw, kw = r(nq * hd), r(nk * hd), r(nk * hd), r(hd), r(hd)
    kc, vc = r(rows * nk * hd), r(rows * nk * hd)
    rope = K.RopeCache(dev)
    rope.ensure(rows, hd, 1e6)
    ws = K.attention_workspace(1, nq, hd, dev)
    data = torch.randint(-128, 128, (H * nq * hd + 1,), generator=g, device=dev, dtype=torch.int32).to(torch.int8)[1:]
    w = K.QuantWeight(data, (r(H + 1).abs() + 0.1)[1:], H, nq * hd)
    a, b, y, z = (torch.full((n,), 9.0, device=dev) for n in (nq * hd, nq * hd, H, H))
    K.decode_attention(a, q.clone(), k, v, qw, kw, rope, pos, nq, nk, hd, 1e-6, 0.1, kc.clone(), vc.clone(), rows, ws)
    K.linear_nobias_int8(y, a, w.data, w.scales, 1, nq * hd, H)
    K.decode_attention_linear_int8(z, b, q.clone(), k, v, qw, kw, rope, pos, nq, nk, hd, 1e-6, 0.1, kc, vc, rows, ws,
                                   w, H)
    assert torch.equal(y, z)


@pytest.mark.gpu
@pytest.mark.parametrize("nq,out_dim", [(8, 500), (8, 2500), (8, 8200), (16, 300), (16, 4100)])
def test_every_row_count_of_the_projection_has_a_merging_kernel(dev, nq, out_dim):
    """1, 2, 4 and 8 rows a wave at 1024 inputs, 1, 2 and 4 at 2048: the merging launch runs for
    each (a size without one raises instead of leaving y as it was)."""
    test_decode_attention_linear_equals_the_two_calls(dev, 130, nq, 8, 128, out_dim)
