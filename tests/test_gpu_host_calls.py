"""The wrappers' native path against their Python path on the same operands: the
same bits, shapes, strides and dtypes where both take a call, the same errors
where the native one leaves it (strided, wrong-shaped, subclassed operands).
"""

from __future__ import annotations

import pytest
import torch

from conftest import gen, normal

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs an MI355X")]

from starter_amd.kernels import _lib  # noqa: E402
from starter_amd.kernels.decode_fused import add_rms_norm, qkv_norm_rope_cache, silu_mul  # noqa: E402
from starter_amd.kernels.embedding import embedding  # noqa: E402
from starter_amd.kernels.lm_head import lm_head_argmax  # noqa: E402
from starter_amd.kernels.prefill import prefill_attention, prefill_qkv  # noqa: E402
from starter_amd.kernels.rmsnorm import rms_norm  # noqa: E402
from starter_amd.kernels.skinny_gemm import linear_partials, linear_silu_mul  # noqa: E402
from starter_amd.kernels.small_query_attention import SmallQueryAttention  # noqa: E402

EPS = 1e-6


class Tagged(torch.Tensor):
    """A tensor subclass: left to the Python path."""


def calls():
    """(name, native, call): call() on operands made anew each time from one seed, and whether the
    native path is to take it."""
    def t(*shape, std=1.0, seed=5):
        return normal(shape, 0.0, std, gen(seed)).cuda()

    def attend(splits, batch=3, capacity=70, cache_dtype=torch.bfloat16):
        qkv = (torch.randn(splits, batch, 1536, generator=gen(6)).cuda() if splits else t(batch, 1536))
        keys, values = t(batch, 2, capacity, 128).to(cache_dtype), t(batch, 2, capacity, 128, seed=7)
        return (qkv, t(128), t(128), EPS, EPS, t(capacity, 128), t(capacity, 128),
                torch.tensor([capacity - 2], device="cuda"), keys, values)

    def run_qkv(splits, **kw):
        operands = attend(splits, **kw)
        attention = SmallQueryAttention(3, 8, 2, 70, "cuda", key_align=16)
        used = torch.full((6,), 69, dtype=torch.int32, device="cuda")
        return (attention.run_qkv(*operands, used, 0.09), *operands[8:])

    def rope_cache(splits):
        operands = attend(splits)
        return (qkv_norm_rope_cache(*operands), *operands[8:])

    def prompt(length):
        keys, values = t(2, 2, 40, 128), t(2, 2, 40, 128)
        q = prefill_qkv(t(2 * length, 1536), t(128), t(128), EPS, EPS, t(40, 128), t(40, 128), keys, values, length)
        return q, prefill_attention(q, keys, values, length, 0.09), keys, values

    ids = torch.tensor([[3, 99], [-1, 0]], device="cuda")
    return [
        ("rms_norm", True, lambda: rms_norm(t(2, 3, 256), t(256), EPS)),
        ("rms_norm 1d", True, lambda: rms_norm(t(256), t(256), EPS)),
        ("rms_norm integer eps", True, lambda: rms_norm(t(1, 256), t(256), 1)),
        ("rms_norm strided", False, lambda: rms_norm(t(3, 2, 256).transpose(0, 1), t(256), EPS)),
        ("rms_norm strided gain", False, lambda: rms_norm(t(3, 256), t(512)[::2], EPS)),
        ("rms_norm empty", False, lambda: rms_norm(t(0, 256), t(256), EPS)),
        ("rms_norm subclass", False, lambda: rms_norm(t(3, 256).as_subclass(Tagged), t(256), EPS)),
        ("rms_norm float32", False, lambda: rms_norm(t(3, 256).float(), t(256), EPS)),
        ("rms_norm too wide", False, lambda: rms_norm(t(3, 8256), t(8256), EPS)),
        ("add_rms_norm", True, lambda: add_rms_norm(t(5, 320), t(5, 320, seed=8), t(320), EPS)),
        ("add_rms_norm partials", True, lambda: add_rms_norm(t(5, 320), t(3, 5, 320, seed=8).float(), t(320), EPS)),
        ("add_rms_norm shape", False, lambda: add_rms_norm(t(5, 320), t(4, 320), t(320), EPS)),
        ("add_rms_norm parts shape", False, lambda: add_rms_norm(t(5, 320), t(3, 5, 64).float(), t(320), EPS)),
        ("add_rms_norm strided", False, lambda: add_rms_norm(t(5, 640)[:, ::2], t(5, 320), t(320), EPS)),
        ("silu_mul", True, lambda: silu_mul(t(7, 514))),
        ("silu_mul odd", False, lambda: silu_mul(t(7, 513))),
        ("silu_mul block", False, lambda: silu_mul(t(7, 512), 0)),
        ("embedding", True, lambda: embedding(ids, t(100, 264))),
        ("embedding strided ids", False, lambda: embedding(ids.T, t(100, 264))),
        ("embedding int32", False, lambda: embedding(ids.int(), t(100, 264))),
        ("linear_partials", True, lambda: linear_partials(t(20, 256), t(96, 256))),
        ("linear_partials rows", False, lambda: linear_partials(t(65, 256), t(96, 256))),
        ("linear_partials columns", False, lambda: linear_partials(t(5, 256), t(80, 256))),
        ("linear_partials unaligned", False, lambda: linear_partials(t(256 * 5 + 1)[1:].view(5, 256), t(96, 256))),
        ("linear_silu_mul", True, lambda: linear_silu_mul(t(20, 256), t(128, 256, std=0.1))),
        ("linear_silu_mul pairs", False, lambda: linear_silu_mul(t(20, 256), t(96, 256))),
        ("lm_head", True, lambda: lm_head_argmax(t(20, 256), t(112, 256))),
        ("lm_head logits", True, lambda: lm_head_argmax(t(20, 256), t(112, 256), logits=True)),
        ("lm_head into", False, lambda: lm_head_argmax(t(2, 256), t(112, 256),
                                                       tokens=torch.empty(2, dtype=torch.int64, device="cuda"))),
        ("rope_cache", True, lambda: rope_cache(0)),
        ("rope_cache partials", True, lambda: rope_cache(4)),
        ("run_qkv", True, lambda: run_qkv(0)),
        ("run_qkv partials", True, lambda: run_qkv(4)),
        ("run_qkv batch", False, lambda: run_qkv(0, batch=2)),
        ("run_qkv cache type", False, lambda: run_qkv(0, cache_dtype=torch.float16)),
        ("prompt", True, lambda: prompt(33)),
        ("prompt too long", False, lambda: prompt(41)),
    ]


def outcome(call):
    try:
        out = call()
    except (ValueError, RuntimeError) as error:
        return type(error), str(error)
    return [(o.shape, o.stride(), o.dtype, type(o), o) for o in (out if isinstance(out, tuple) else (out,))]


@pytest.mark.parametrize("index", range(len(calls()) if torch.cuda.is_available() else 0))
@torch.no_grad()
def test_native_and_python_paths_agree(index, monkeypatch):
    name, native, call = calls()[index]
    taken = []

    class Watched:
        def __getattr__(self, function):
            def run(*args):
                out = getattr(module, function)(*args)
                taken.append(out is not NotImplemented)
                return out
            return run

    module = _lib.host()
    assert not isinstance(module, _lib._NoHostCalls)
    monkeypatch.setattr(_lib, "_host", Watched())
    got = outcome(call)
    # a refused chain may have had a native first call
    assert all(taken) if native else not (taken and taken[-1]), (name, taken)
    monkeypatch.setattr(_lib, "_host", _lib._NoHostCalls())
    want = outcome(call)
    if isinstance(want, tuple):
        assert got == want, name
        return
    for g, w in zip(got, want, strict=True):
        assert g[:4] == w[:4], name
        assert torch.equal(g[4].view(torch.uint8) if g[4].dtype == torch.bfloat16 else g[4],
                           w[4].view(torch.uint8) if w[4].dtype == torch.bfloat16 else w[4]), name


def test_grad_mode_and_dispatch_modes_take_the_python_path():
    from torch.utils._python_dispatch import TorchDispatchMode

    class Seen(TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.ops = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.ops.append(func)
            return func(*args, **(kwargs or {}))

    x, w = torch.ones(2, 256, dtype=torch.bfloat16, device="cuda"), torch.ones(256, dtype=torch.bfloat16, device="cuda")
    with Seen() as seen:
        assert _lib.host().rms_norm(x, w, EPS) is NotImplemented
        rms_norm(x, w, EPS)
    assert seen.ops  # the allocation is still the mode's to see
    with torch.enable_grad():  # refused by the attention, as before
        kind, text = outcome(next(call for name, _, call in calls() if name == "run_qkv"))
    assert kind is ValueError and "expected packed" in text
