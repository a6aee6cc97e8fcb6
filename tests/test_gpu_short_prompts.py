"""Prompt kernels on both sides of their small-call rules: the attention's
workgroup form for batches of short prompts, and the Q/K/V kernel's units per
wave (one up to 3,072 units of 8 head rows, two beyond)."""

from __future__ import annotations

import pytest
import torch

from conftest import O, assert_bits_exact, bits, gen, normal

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs an MI355X")]

from starter_amd.kernels.prefill import prefill_attention, prefill_qkv  # noqa: E402

DEV = "cuda"


# 33 x 8 pairs: at least one wide workgroup per CU; 48 | 49 positions: 4-wave form | 8-wave form
@pytest.mark.parametrize("length", [1, 5, 16, 17, 48, 49, 64])
def test_attention_of_many_short_prompts(length):
    g = gen(800 + length)
    batch, hq, hk, capacity = 33, 32, 8, length + 3
    q, k, v = (normal((batch, n, t, 128), g=g) for n, t in ((length, hq), (hk, capacity), (hk, capacity)))
    k[:, :, length:], v[:, :, length:] = float("nan"), float("nan")  # slots past the prompt are never read
    got = prefill_attention(q.to(DEV), k.to(DEV), v.to(DEV), length, 128 ** -0.5).float().cpu()
    kf, vf = (t[:, :, :length].float().repeat_interleave(hq // hk, 1) for t in (k, v))
    s = (q.float().transpose(1, 2) @ kf.transpose(2, 3).contiguous()) * 128 ** -0.5
    s.masked_fill_(torch.ones(length, length).triu(1).bool(), float("-inf"))
    want = (torch.softmax(s, -1) @ vf).transpose(1, 2)
    # the bar of the reference's attention tests: bf16 probabilities and output
    torch.testing.assert_close(got, want, rtol=0.02, atol=0.004 * 4)
    assert float((got - want).norm() / want.norm()) < 0.01


@pytest.mark.parametrize("batch,length,nq,nk", [(1, 1, 32, 8), (3, 5, 16, 8), (1, 512, 32, 8), (1, 513, 32, 8),
                                                (7, 110, 16, 8), (1, 1100, 8, 8)])
def test_qkv_units_per_wave(batch, length, nq, nk):
    g = gen(820 + length)
    capacity = length + 2
    qkv = normal((batch * length, (nq + 2 * nk) * 128), g=g)
    qw, kw = normal((128,), 1.0, 0.1, g), normal((128,), 1.0, 0.1, g)
    cos, sin = normal((capacity, 128), g=g), normal((capacity, 128), g=g)
    cache = torch.full((batch, nk, capacity, 128), 33.0, dtype=torch.bfloat16)
    keys, values = cache.to(DEV), cache.to(DEV)
    q = prefill_qkv(qkv.to(DEV), qw.to(DEV), kw.to(DEV), 1e-6, 1e-6, cos.to(DEV), sin.to(DEV), keys, values, length)
    rq, rk, rv = O.prefill_qkv(bits(qkv), bits(qw), bits(kw), 1e-6, 1e-6, bits(cos), bits(sin), bits(cache),
                               bits(cache), length)
    assert_bits_exact(q, rq, what="q")
    assert_bits_exact(keys, rk, what="keys")
    assert_bits_exact(values, rv, what="values")
