"""Products of many rows on the tile kernel: edges of its tiles against float64, and the calls that stay with the library."""

import pytest
import torch
import torch.nn.functional as F

from kllms_amd import ops

DEV = "cuda:0"
gpu = pytest.mark.gpu


def _operands(M, N, K, gated, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn((2 if gated else 1) * N, K, generator=g, device=DEV) * K ** -0.5).bfloat16()
    return x, w


def _near(got, ref, sums):
    # half a bf16 step of the result, and fp32 sums of K terms in any order: 2^-24 of the sum of their sizes a step
    return ((got.double() - ref).abs() <= 2 ** -8 * ref.abs() + sums).all()


# one row, one column unit, odd rows behind a tile, a last column tile of 8, one stage and odd numbers of them; at 17 stages
# two shares, at 33 and 65 four, where the rule's tiles leave units idle
SIZES = [(1, 8, 64), (33, 264, 128), (129, 520, 1088), (257, 256, 2112), (1031, 1288, 192),
         (70, 2056, 4160)]


@gpu
@pytest.mark.parametrize("mj", range(2, 9))
@pytest.mark.parametrize("share", [False, True])
@pytest.mark.parametrize("M,N,K", SIZES)
def test_tiles_against_float64(M, N, K, share, mj):
    C = ops._hip_or_raise()
    x, w = _operands(M, N, K, False)
    bias = torch.randn(N, device=DEV).bfloat16()
    ref = x.double() @ w.double().t()
    slack = K * 2 ** -24 * (x.double().abs() @ w.double().abs().t())
    assert _near(C.linear_tiles(x, w, bias[:0], 0, mj, share, 0.0, 0.0), ref, slack)
    assert _near(C.linear_tiles(x, w, bias, 0, mj, share, 0.0, 0.0), ref + bias.double(), slack + 1e-6)
    x, w = _operands(M, N, K, True, 1)
    g, u = (x.double() @ w.double().t()).chunk(2, -1)
    slack = K * 2 ** -24 * (x.double().abs() @ w.double().abs().t())
    # the activations' slopes are below 1.1 (silu) and 1.1 * alpha, their values below the other factor
    slack = 3 * (slack[:, :N] * (u.abs() + 1) + slack[:, N:] * (g.abs() + 1)) + 1e-5
    assert _near(C.linear_tiles(x, w, bias[:0], 1, mj, share, 0.0, 0.0), F.silu(g) * u, slack)
    c, d = g.clamp(max=1.5), u.clamp(-1.5, 1.5)
    assert _near(C.linear_tiles(x, w, bias[:0], 2, mj, share, 1.5, 1.702), c * torch.sigmoid(1.702 * c) * (d + 1), slack)


def _shares(M, N, K, mj):
    """Shares of the last round's tiles on each XCD, and whole rounds before it: (tiles, 256 x 32 mj) dealt to 8 x 32 units."""
    tiles, stages = -(-M // (32 * mj)) * -(-N // 256), K // 64
    out = set()
    for xcd in range(8):
        n = tiles * (xcd + 1) // 8 - tiles * xcd // 8
        out.add((max(1, min(32 // (n % 32), 4, stages // 8)) if n % 32 else 1, n // 32))
    return out


# 9 of an XCD's 32 units in three shares; the same behind a whole round; odd numbers of stages in two, three and four shares
SHARED = [(576, 2048, 1536, 2), (2624, 2048, 1536, 2), (2600, 2040, 2624, 2), (1100, 2048, 1600, 3), (450, 1032, 4160, 4),
          (3400, 1536, 1088, 8), (2200, 2048, 2112, 2)]


@gpu
@pytest.mark.parametrize("M,N,K,mj", SHARED)
def test_shares_against_float64(M, N, K, mj):
    test_tiles_against_float64(M, N, K, True, mj)


def test_shares_of_every_kind_are_tested():
    kinds = set().union(*(_shares(*c) for c in SHARED), *(_shares(*c, 8) for c in SIZES))
    assert {s for s, _ in kinds} == {1, 2, 3, 4}
    assert {s for s, rounds in kinds if rounds} >= {3, 4}


@gpu
@pytest.mark.parametrize("M,N,K,act", [(1300, 3216, 2048, 0), (1170, 6144, 4096, 0), (700, 2048, 8192, 0), (777, 8192, 2048, 1), (400, 8192, 2048, 2)])
def test_entry_points_against_float64(M, N, K, act):
    x, w = _operands(M, N, K, act > 0, 2)
    y = x.double() @ w.double().t()
    if act == 0:
        got, ref = ops.linear(x, w), y
    elif act == 1:
        got, ref = ops.linear_silu(x, w), F.silu(y[:, :N]) * y[:, N:]
    else:
        c, d = y[:, :N].clamp(max=7.0), y[:, N:].clamp(-7.0, 7.0)
        got, ref = ops.linear_clamped_glu(x, w, 7.0, 1.702), c * torch.sigmoid(1.702 * c) * (d + 1)
    # one rounding to bf16 of values of a normal shape is 0.0017 of them in the 2-norm
    assert (got.double() - ref).norm() <= 0.002 * ref.norm()


@gpu
def test_extreme_sums_of_the_clamped_form():
    x, w = _operands(256, 128, 64, True, 3)
    got = ops._hip_or_raise().linear_tiles((x * 1000).contiguous(), w, x[:0, 0], 2, 2, False, 7.0, 1.702)
    y = (x * 1000).double() @ w.double().t()
    c, d = y[:, :128].clamp(max=7.0), y[:, 128:].clamp(-7.0, 7.0)
    assert torch.isfinite(got).all()
    # factors of at most 8 beside slopes below 1.1, as above
    slack = 64 * 2 ** -24 * ((x.double() * 1000).abs() @ w.double().abs().t())
    assert _near(got, c * torch.sigmoid(1.702 * c) * (d + 1), 9 * (slack[:, :128] + slack[:, 128:]) + 1e-5)


@gpu
def test_gates_without_a_limit():
    """Sums behind fp32's range and close to it, with no limit: the gate's sigmoid ends at 0 and 1."""
    x = torch.ones(8, 64, device=DEV).bfloat16()
    w = torch.full((16, 64), 0.25, device=DEV).bfloat16()
    w[:4] = torch.tensor([3e38, 5e36, -5e36, 1e-30], device=DEV).unsqueeze(1)      # inf, 3.2e38, -3.2e38, 6.4e-29
    got = ops._hip_or_raise().linear_tiles(x, w, x[:0, 0], 2, 2, False, float("inf"), 1.702)
    g, u = (x.float() @ w.float().t()).chunk(2, -1)
    ref = g * torch.sigmoid(1.702 * g) * (u + 1)
    assert torch.isinf(ref[:, 0]).all() and torch.equal(got.isnan(), ref.isnan())
    assert torch.equal(got.isinf(), ref.bfloat16().isinf())
    ok = ref.bfloat16().isfinite()
    assert torch.allclose(got.float()[ok], ref[ok], rtol=2 ** -7)


@gpu
def test_calls_that_stay_with_the_library():
    pick = lambda x, w, bias=None: ops._hip_or_raise().linear_tiles_pick(x, w, bias, 0)  # noqa: E731
    x, w = _operands(2048, 2048, 1024, False)
    assert pick(x, w) and pick(x, torch.nn.Parameter(w, requires_grad=False))
    assert not pick(x[:128], w) and not pick(x.float(), w.float())
    assert not pick(x[:, ::2], w[:, ::2]) and not pick(x[:, :1000].contiguous(), w[:, :1000].contiguous())
    assert not pick(x.t().contiguous().t(), w) and not pick(x.view(2, 1024, 1024), w)
    off = torch.empty(x.numel() + 1, device=DEV, dtype=x.dtype)[1:].view_as(x).copy_(x)
    assert not pick(off, w) and torch.allclose(ops.linear(off, w).float(), ops.linear(x, w).float(), atol=0.05)
    assert not pick(x, w, torch.zeros(2048, device=DEV))
    xg = x.clone().requires_grad_()
    ops.linear(xg, w).sum().backward()
    assert xg.grad is not None
    with torch.no_grad():
        assert pick(xg, w)
    got = torch.func.vmap(lambda t: ops.linear(t, w))(x.view(2, 1024, 1024))
    assert torch.allclose(got.view(2048, -1).float(), ops.linear(x, w).float(), atol=0.05)
    _, tangent = torch.func.jvp(lambda t: ops.linear(t, w), (x,), (x,))
    assert torch.allclose(tangent.float(), ops.linear(x, w).float(), atol=0.05)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, x)
        assert not pick(dual, w)
    traced = torch.jit.trace(lambda t: ops.linear(t, w), (x,), check_trace=False)
    assert torch.allclose(traced(x * 2).float(), ops.linear(x * 2, w).float(), atol=0.05)


@gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_autocast_decides_the_type_at_every_row_count(dtype):
    x, w = _operands(2304, 2048, 1024, False)
    with torch.autocast("cuda", dtype=dtype):
        for rows in (64, 2304):
            got = ops.linear(x[:rows], w)
            assert got.dtype == dtype and torch.equal(got, F.linear(x[:rows], w))
        assert ops.linear_silu(x, w) is None and ops.linear_clamped_glu(x, w, 7.0, 1.702) is None
    assert ops.linear(x, w).dtype == torch.bfloat16 and ops.linear_silu(x, w) is not None


class _Tagged(torch.Tensor):
    pass


class _Products(torch.overrides.TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.seen = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        if func is F.linear:
            self.seen.append(args[0].shape[0])
        return func(*args, **(kwargs or {}))


@gpu
def test_subclasses_modes_and_the_compiler_see_the_product():
    x, w = _operands(2304, 2048, 1024, False)
    for a, b in ((x.as_subclass(_Tagged), w), (x, w.as_subclass(_Tagged))):
        for rows in (64, 2304):
            assert type(ops.linear(a[:rows], b)) is _Tagged
        assert ops.linear_silu(a, b) is None
    with _Products() as mode:
        ops.linear(x[:64], w), ops.linear(x, w)
    assert mode.seen == [64, 2304]
    whole = torch.compile(lambda a, b: ops.linear(a, b), backend="eager", fullgraph=True)
    assert torch.equal(whole(x, w), F.linear(x, w))


@gpu
@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="a device that is not the current one takes two")
def test_operands_of_another_device_than_the_current_one():
    x, w = _operands(2304, 2048, 1024, False)
    with torch.cuda.device(1):
        got = ops.linear(x, w)
    assert got.device == x.device and torch.equal(got, ops.linear(x, w))


def test_rule_of_the_tiles():
    if not ops.hip_available():
        pytest.skip("extension not built")
    rows = ops._hip_or_raise().linear_tiles_rows
    assert rows(128, 8192, 2048, 1) == 0                       # few rows
    assert rows(256, 4096, 14336, 0) == 0                      # long K on few tiles
    assert rows(1170, 4096, 14336, 0) == 5 + 16                # 128 tiles of 147 rows, in two shares each
    assert rows(7777, 4096, 4096, 0) == 0                      # 496 tiles of the 512 of two rounds
    assert rows(300, 2048, 2048, 0) == 0 and rows(1200, 4096, 4096, 0) == 0
    assert rows(300, 14336, 4096, 1) == 5                      # 224 tiles of 150 rows
    assert rows(11700, 4096, 14336, 0) == 8                    # 736 tiles in three rounds
    # plain products whose tiles fill the library's rounds, few tiles, gated products of a few workgroups; w's rows no
    # multiple of 256, where the library has no such tiles
    assert rows(6000, 8192, 2048, 0) == 0 and rows(700, 6144, 5120, 0) == 0 and rows(129, 128, 2048, 1) == 0
    assert rows(7700, 3328, 2048, 0) == 0 and rows(7700, 3216, 2048, 0) and rows(7700, 3320, 2048, 0)
    assert rows(1170, 4096, 8192, 0) == 0 and rows(4400, 2048, 8192, 0) == 5
    for M in range(1, 13000, 97):
        for N, K, act in ((4096, 4096, 0), (3216, 2048, 0), (14336, 4096, 1)):
            assert rows(M, N, K, act) in (0, 2, 3, 4, 5, 6, 7, 8)      # K below 8192: never shared
