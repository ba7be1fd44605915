"""How the decode attentions cut their keys, against the oracle at the fp32
tolerance of the other attention tests."""
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
