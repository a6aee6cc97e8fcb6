"""Prompt kernels on both sides of their dispatch rules: the attention's
workgroup forms, and the Q/K/V kernel's units per wave (one up to 3,072 units of
8 head rows, two beyond, in workgroups of one wave or four)."""

from __future__ import annotations

import pytest
import torch

from conftest import O, assert_bits_exact, bits, gen, normal

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs an MI355X")]

from starter_amd.kernels.prefill import prefill_attention, prefill_qkv  # noqa: E402

DEV = "cuda"


def check_attention(batch, length, hq, hk):
    g = torch.Generator(device=DEV).manual_seed(800 + length + hq)
    capacity = length + 3
    q, k, v = (torch.randn(batch, n, t, 128, generator=g, device=DEV).bfloat16()
               for n, t in ((length, hq), (hk, capacity), (hk, capacity)))
    k[:, :, length:], v[:, :, length:] = float("nan"), float("nan")  # slots past the prompt are never read
    got = prefill_attention(q, k, v, length, 128 ** -0.5).float()
    hide = torch.ones(length, length, device=DEV).triu(1).bool()
    for b in range(0, batch, max(1, batch // 5)):
        kf, vf = (t[b, :, :length].float().repeat_interleave(hq // hk, 0) for t in (k, v))
        s = (q[b].float().transpose(0, 1) @ kf.transpose(1, 2).contiguous()) * 128 ** -0.5
        want = (torch.softmax(s.masked_fill(hide, float("-inf")), -1) @ vf).transpose(0, 1)
        # bf16 probabilities (2^-9 of a sum of up to 4 x |v|) and output (2^-8)
        torch.testing.assert_close(got[b], want, rtol=0.02, atol=0.016)
        assert float((got[b] - want).norm() / want.norm()) < 0.01


# at least one wide workgroup per CU: 16 | 17 positions, one to four wide blocks, a fifth and a sixth
# at most and over half full, seven
@pytest.mark.parametrize("batch,length", [(33, 1), (33, 5), (33, 16), (33, 17), (33, 48), (33, 64), (33, 65), (9, 255),
                                          (9, 256), (9, 257), (9, 288), (9, 289), (9, 352), (9, 353), (9, 385)])
def test_attention_forms_at_four_heads_per_kv_head(batch, length):
    check_attention(batch, length, 32, 8)


# 1,023 | 1,024 wide workgroups: the narrow form | the 8-wave form
@pytest.mark.parametrize("batch,length,hk", [(1, 1, 8), (3, 97, 8), (341, 64, 3), (256, 33, 4), (128, 64, 8), (64, 65, 8)])
def test_attention_forms_at_two_heads_per_kv_head(batch, length, hk):
    check_attention(batch, length, 2 * hk, hk)


# under | at one wide workgroup per CU; up to four wide blocks of 32, a fifth half full and fuller
@pytest.mark.parametrize("batch,length", [(1, 1), (5, 130), (128, 3), (128, 33), (64, 127), (64, 128), (64, 144), (64, 145)])
def test_attention_forms_at_eight_heads_per_kv_head(batch, length):
    check_attention(batch, length, 16, 2)


# at 32 over 8 heads: 16 | 17 positions; exactly one wide workgroup per CU and more; six blocks up to 9/8 of
# that and beyond; over six.  16 over 8: four per CU.  16 over 2: 32 positions a block
@pytest.mark.parametrize("batch,length,hq,hk", [(33, 16, 32, 8), (33, 17, 32, 8), (8, 250, 32, 8), (9, 250, 32, 8), (8, 257, 32, 8),
                                                (6, 352, 32, 8), (7, 352, 32, 8), (9, 353, 32, 8), (9, 400, 32, 8),
                                                (32, 200, 16, 8), (64, 127, 16, 2), (64, 144, 16, 2), (64, 145, 16, 2)])
def test_attention_forms_give_the_same_bits(batch, length, hq, hk):
    """A sequence alone runs the narrow form, in a batch the one its grid asks for."""
    g = torch.Generator(device=DEV).manual_seed(810 + length)
    q, k, v = (torch.randn(1, *shape, 128, generator=g, device=DEV).bfloat16()
               for shape in ((length, hq), (hk, length), (hk, length)))
    alone = prefill_attention(q, k, v, length, 128 ** -0.5)
    many = prefill_attention(*(t.expand(batch, -1, -1, -1).contiguous() for t in (q, k, v)), length, 128 ** -0.5)
    assert torch.equal(many, alone.expand_as(many))


@pytest.mark.parametrize("batch,length,nq,nk", [(1, 1, 32, 8), (3, 5, 16, 8), (1, 512, 32, 8), (1, 513, 32, 8),
                                                (7, 110, 16, 8), (1, 1100, 8, 8), (1, 700, 24, 8), (3, 300, 40, 8)])
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
