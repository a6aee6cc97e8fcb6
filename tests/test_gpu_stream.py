"""The one-workgroup-per-CU weight streams (partials beyond 16 rows, gate/up and
LM head from 5) at the edges of their plans: fewer tiles than CUs, one tile
more than an even share, several column blocks per workgroup, and K ranges of
one chunk, an odd number of chunks and fewer chunks than the ring holds.

Integer inputs: every partial sum is a whole number below 2^24, so the result
is exact in any order and compared bit for bit with a float64 product.
"""

from __future__ import annotations

import pytest
import torch

from conftest import O, assert_bits_exact, bits, gen

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs an MI355X")]

from starter_amd import modules  # noqa: E402
from starter_amd.kernels import _lib, skinny_gemm as sk  # noqa: E402
from starter_amd.kernels.lm_head import lm_head_argmax  # noqa: E402

DEV = "cuda"


def ints(shape, lo, hi, g):
    return torch.randint(lo, hi + 1, shape, generator=g).to(torch.bfloat16)


@pytest.mark.parametrize("m", [17, 32, 33, 48, 64])
# 2 tiles | 258 for 256 workgroups | 2 a workgroup | 2 or 3, K of 1, 3, 2 and 5 chunks a split
@pytest.mark.parametrize("n,k,splits", [(32, 64, 1), (32, 192, 3), (4128, 192, 1), (6144, 128, 1),
                                        (2048, 320, 5), (416, 640, 2)])
def test_partials(m, n, k, splits):
    g = gen(700 + m + n)
    x, w = ints((m, k), -4, 4, g), ints((n, k), -3, 3, g)
    xd, wd = x.to(DEV), w.to(DEV)
    got = torch.full((splits, m, n), float("nan"), device=DEV)
    _lib.call("qf_linear_partials", xd.data_ptr(), m, k, wd.data_ptr(), n, splits, got.data_ptr(),
              _lib.stream(xd.device))
    per = k // splits
    want = torch.stack([x.double()[:, s * per:(s + 1) * per] @ w.double()[:, s * per:(s + 1) * per].T
                        for s in range(splits)]).float()
    assert torch.equal(got.cpu(), want)


@pytest.mark.parametrize("m", [5, 16, 17, 33, 64])
# 4 half tiles | 260 for 256 workgroups | 20 a workgroup (two blocks)
@pytest.mark.parametrize("n,k", [(32, 64), (2080, 192), (40960, 64), (96, 1024)])
def test_silu_mul(m, n, k):
    g = gen(720 + m + n)
    x, w = ints((m, k), -2, 2, g), ints((2 * n, k), -1, 1, g)
    got = sk.linear_silu_mul(x.to(DEV), w.to(DEV))
    proj = (x.double() @ w.double().T).float().to(torch.bfloat16)
    assert_bits_exact(got, O.silu_mul(bits(proj)), what=f"silu m={m} n={n} k={k}")


@pytest.mark.parametrize("m", [5, 16, 17, 33, 64])
# 1 tile | 257 tiles for 256 workgroups | 39 a workgroup (three blocks)
@pytest.mark.parametrize("vocab,k", [(16, 64), (4112, 192), (159760, 64)])
def test_lm_head(m, vocab, k):
    g = gen(740 + m + vocab)
    x, w = ints((m, k), -1, 1, g), ints((vocab, k), -1, 1, g)
    tokens, logits = lm_head_argmax(x.to(DEV), w.to(DEV), logits=True)
    want = (x.double() @ w.double().T).float().to(torch.bfloat16)
    assert torch.equal(logits.cpu(), want)
    assert torch.equal(tokens.cpu(), want.float().argmax(-1))  # full of ties: the first maximum


def device_ints(shape, most, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randint(-most, most + 1, shape, generator=g, device=DEV, dtype=torch.int8).bfloat16()


@pytest.mark.parametrize("m", [17, 32, 33, 48, 64])
# tiles a workgroup (as blocks, on the kernel for): 4 | 6 | 7 (8) | 9 (10) | 11 (13) | 15 (16) | 17 (19) | 20 (2 x 10) |
# 12 splits x 23 (2 x 12 on 13), the last group shorter | 130 splits x 38 (2 x 19)
@pytest.mark.parametrize("n,k,splits", [(16384, 320, 1), (24576, 448, 1), (28672, 320, 1), (36864, 320, 1), (45056, 448, 1),
                                        (61440, 320, 1), (69632, 320, 1), (81920, 320, 1), (7456, 5376, 12),
                                        (608, 41600, 130),
                                        # small workgroups: one chunk a split, two, four, columns past the last tile
                                        (2560, 5056, 79), (608, 8896, 139), (640, 12800, 100), (352, 33024, 129),
                                        # and at 8 chunks: blocks of 8 tiles up to 48 rows, of 13 up to 32
                                        (2560, 6144, 12), (2592, 6144, 12), (2560, 9728, 19)])
def test_partials_of_several_tiles_and_blocks(m, n, k, splits):
    x, w = device_ints((m, k), 4, 780 + m), device_ints((n, k), 3, 781 + n)
    got = torch.full((splits, m, n), float("nan"), device=DEV)
    _lib.call("qf_linear_partials", x.data_ptr(), m, k, w.data_ptr(), n, splits, got.data_ptr(), _lib.stream(x.device))
    for s in range(splits):
        part = slice(s * (k // splits), (s + 1) * (k // splits))
        assert torch.equal(got[s].double(), x[:, part].double() @ w[:, part].double().T), s


@pytest.mark.parametrize("k,n", [(64, 32), (320, 96), (1024, 2080), (2112, 4096), (2048, 8224)])
def test_gate_up_rows_up_to_16_share_their_bits(k, n):
    """Below the stream's widths a row's result does not depend on the rows beside it."""
    g = torch.Generator(device=DEV).manual_seed(785 + n)
    x, w = (torch.randn(rows, k, generator=g, device=DEV).bfloat16() for rows in (16, 2 * n))
    whole = sk.linear_silu_mul(x, w)
    for m in (1, 4, 5, 8, 9, 12, 13):
        assert torch.equal(sk.linear_silu_mul(x[:m].contiguous(), w), whole[:m]), m


@pytest.mark.parametrize("m", [5, 9, 12, 13, 16])
# one tile a stream workgroup | two, and three | three, and four, at the K on both sides of the rule
@pytest.mark.parametrize("n,k", [(96, 2112), (4096, 2112), (4128, 2112), (6144, 2112), (6176, 2112), (4128, 3072), (6176, 2048)])
def test_gate_up_on_both_sides_of_the_streams_rule(m, n, k):
    x, w = device_ints((m, k), 2, 786 + m), device_ints((2 * n, k), 1, 787 + n)
    got = sk.linear_silu_mul(x, w)
    proj = (x.double() @ w.double().T).float().to(torch.bfloat16)
    assert_bits_exact(got, O.silu_mul(bits(proj)), what=f"silu m={m} n={n} k={k}")


@pytest.mark.parametrize("m", [17, 33, 64])
# K in order: 3 ragged stages of 128 or 5 of 64 | in quarters: 8 of 128 or 16 of 64
@pytest.mark.parametrize("k", [320, 1024])
# 5 tiles a workgroup | 11 (13) | 18 (19; in quarters beyond 32 rows 2 x 9) | 20 (2 x 10), its last group shorter
@pytest.mark.parametrize("n", [10240, 22528, 36864, 40928])
def test_silu_mul_of_several_tiles_and_blocks(m, k, n):
    x, w = device_ints((m, k), 2, 790 + m), device_ints((2 * n, k), 1, 791 + n)
    got = sk.linear_silu_mul(x, w)
    proj = (x.double() @ w.double().T).float().to(torch.bfloat16)
    assert_bits_exact(got, O.silu_mul(bits(proj)), what=f"silu m={m} n={n} k={k}")


@pytest.mark.parametrize("m", [5, 17, 33, 64])
@pytest.mark.parametrize("k", [320, 1024])
# 14 tiles a workgroup (16) | 39 (3 x 13)
@pytest.mark.parametrize("vocab", [57344, 159760])
def test_lm_head_of_several_tiles_and_blocks(m, k, vocab):
    x, w = device_ints((m, k), 1, 795 + m), device_ints((vocab, k), 1, 796 + vocab)
    tokens, logits = lm_head_argmax(x, w, logits=True)
    want = (x.double() @ w.double().T).float().to(torch.bfloat16)
    assert torch.equal(logits, want)
    assert torch.equal(tokens.cpu(), want.float().cpu().argmax(-1))  # full of ties: the first maximum


@pytest.mark.parametrize("m", [5, 33, 64])
@pytest.mark.parametrize("fill", ["nan", "-inf"])
def test_lm_head_order_across_workgroups(m, fill):
    """NaN above everything and the first of several; a row of nothing but -inf picks column 0."""
    vocab, k = 4112, 64
    g = gen(750 + m)
    x, w = torch.ones(m, k).bfloat16(), ints((vocab, k), -1, 1, g)
    if fill == "nan":
        w[[4111, 2049, 3000]] = float("nan")
        w[17] = float("inf")
    else:
        w[:] = float("-inf")
    tokens, _ = lm_head_argmax(x.to(DEV), w.to(DEV), logits=True)
    assert tokens.tolist() == [2049 if fill == "nan" else 0] * m


@pytest.mark.parametrize("m", [5, 17, 33, 64])
# in order (an odd number of chunks, 64 and 128 k per stage) | in quarters
@pytest.mark.parametrize("k", [320, 2560, 1024, 4096])
def test_column_bits_do_not_depend_on_their_place(m, k):
    """Equal weight rows give equal bits wherever they stand, in a call of any width: the order of
    additions is a function of K alone, so a column shard equals its part of the whole."""
    g = gen(770 + m + k)
    base, x = torch.randn(64, k, generator=g).bfloat16().to(DEV), torch.randn(m, k, generator=g).bfloat16().to(DEV)
    few, many = base.repeat(5, 1), base.repeat(513, 1)  # 64 and 128 k per stage, one to three blocks
    _, narrow = lm_head_argmax(x, few, logits=True)
    _, wide = lm_head_argmax(x, many, logits=True)
    assert torch.equal(wide.view(m, -1, 64), narrow[:, None, :64].expand(m, 513, 64))
    assert torch.equal(narrow.view(m, -1, 64), narrow[:, None, :64].expand(m, 5, 64))
    if m > 16:  # up to there gate/up and partials choose their kernel by width
        narrow, wide = (sk.linear_silu_mul(x, torch.cat([w, -w])) for w in (few, many))
        assert torch.equal(wide.view(m, -1, 64), narrow[:, None, :64].expand(m, 513, 64))
        narrow, wide = (sk.linear_partials(x, w) for w in (few, many))
        assert torch.equal(wide.view(*narrow.shape[:2], -1, 64), narrow[:, :, None, :64].expand(-1, m, 513, 64))


class _MLP(torch.nn.Module):
    def __init__(self, hidden, inner, g):
        super().__init__()
        self.gate_proj, self.up_proj = (torch.nn.Linear(hidden, inner, bias=False) for _ in range(2))
        self.down_proj, self.act_fn = torch.nn.Linear(inner, hidden, bias=False), torch.nn.SiLU()
        for p in self.parameters():
            p.data = torch.randn(p.shape, generator=g) * 0.1


@pytest.mark.parametrize("shape", [(1, 256), (2, 3, 256), (64, 256), (65, 256), (1, 0, 256)])
@pytest.mark.parametrize("inner", [320, 96, 80])  # 80: not whole column pairs, the library's product
@pytest.mark.parametrize("form", ["plain", "strided", "autocast"])
@torch.no_grad()
def test_packed_mlp_on_both_sides_of_its_row_rule(shape, inner, form, monkeypatch):
    """The module on decode-sized inputs against the projections and activation in sequence: within
    the f32 accumulation of a projection, which moves single bf16 values by one rounding."""
    g = gen(760 + inner)
    module = modules.PackedMLP(_MLP(256, inner, g).cuda().bfloat16())
    x = torch.randn(shape, generator=g).cuda().bfloat16()
    if form == "strided":
        x = torch.stack([x, x], -1)[..., 0]
    taken = []
    monkeypatch.setattr(modules, "linear_silu_mul", lambda *args: taken.append(args) or sk.linear_silu_mul(*args))
    with torch.autocast("cuda", dtype=torch.float16, enabled=form == "autocast"):
        got = module(x)
        assert len(taken) == (1 <= x.shape[:-1].numel() <= 64 and inner != 80 and form == "plain")
        projected = torch.nn.functional.linear(x, module.gate_up_weight)
        gate, up = projected.chunk(2, -1)
        want = module.down_proj(torch.nn.functional.silu(gate) * up)
    assert got.shape == want.shape and got.dtype == want.dtype
    torch.testing.assert_close(got.float(), want.float(), rtol=0.02, atol=0.02 * float(want.float().abs().max()) if want.numel() else 0)


class _Scaled(torch.Tensor):
    """A weight without memory of its own, as quantised ones are: bf16(values * 0.5) when a product asks."""

    @staticmethod
    def __new__(cls, values):
        return torch.Tensor._make_wrapper_subclass(cls, values.shape, dtype=torch.bfloat16, device=values.device)

    def __init__(self, values):
        self.values = values

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        if func is torch.ops.aten.detach.default:
            return cls(args[0].values)
        return func(*[a.values * 0.5 if isinstance(a, _Scaled) else a for a in args], **(kwargs or {}))


@torch.no_grad()
def test_packed_mlp_leaves_subclassed_weights_and_watched_calls_to_torch():
    from torch.utils._python_dispatch import TorchDispatchMode

    class Seen(TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.ops = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.ops.append(str(func))
            return func(*args, **(kwargs or {}))

    g = gen(765)
    module = modules.PackedMLP(_MLP(256, 320, g).cuda().bfloat16())
    x = torch.randn(3, 256, generator=g).cuda().bfloat16()
    with Seen() as seen:
        module(x)
    assert sum("mm" in op or "linear" in op for op in seen.ops) == 2, seen.ops  # both products
    weight = module.gate_up_weight
    halved = torch.nn.Parameter(weight * 0.5, requires_grad=False)
    module.gate_up_weight = halved
    want = module(x)
    module.gate_up_weight = torch.nn.Parameter(_Scaled(weight.data), requires_grad=False)
    torch.testing.assert_close(module(x).float(), want.float(), rtol=0.02, atol=0.02 * float(want.float().abs().max()))
