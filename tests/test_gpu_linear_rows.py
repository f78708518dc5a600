"""trimkv_linear_rows and trimkv_linear_rows_silu (a linear layer over the rows of a decode step) against 64-bit products.

Bounds: fp32 sums of k products err by at most about k 2^-24 sum |x w| (any order), the result is rounded once (half a unit in the
last place, 2^-9 of the value in bf16 and 2^-12 in fp16; twice that here, for values that straddle)."""
import ctypes

import pytest
import torch
from torch import nn

from trimkv_amd import _lib, linear

DEV = "cuda:0"
EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _operands(rows, n, k, dtype, seed=0):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    made = lambda *shape: torch.randn(*shape, generator=gen, device=DEV).to(dtype)
    return made(rows, k), made(n, k) * 0.1, made(n)


def _check(got, x, w, bias, dtype):
    exact, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    if bias is not None:
        exact = exact + bias.double()
    bound = EPS[dtype] * exact.abs() + x.shape[1] * 2.0 ** -23 * size + 2.0 ** -24
    err = (got.double() - exact).abs()
    assert (err <= bound).all(), (float((err - bound).max()), (err > bound).nonzero()[:4].tolist())


# rows: every number of row groups and their edges; n: ends of groups of 8 columns and of tiles, every number of groups per tile and more tiles than workgroups;
# k: fewer steps than wavefronts, numbers that do not divide among them
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,n,k", [(1, 1, 64), (1, 15, 128), (7, 16, 192), (8, 17, 320), (9, 40, 64), (16, 100, 1024), (17, 33, 448), (31, 2048, 512), (32, 18, 64), (33, 1000, 704),
                                      (63, 47, 576), (64, 4096, 256), (1, 4608, 128), (16, 4612, 192), (32, 12288, 64), (5, 12291, 64), (64, 12280, 128), (64, 24576, 64),
                                      (50, 24600, 128), (8, 70001, 64), (16, 50000, 64), (64, 50002, 64),
                                      (1, 7, 64), (8, 8, 128), (33, 9, 64), (16, 2041, 192), (64, 2048, 704), (8, 2049, 64), (24, 2056, 64)])
def test_linear_rows_matches_the_product(rows, n, k, dtype):
    x, w, bias = _operands(rows, n, k, dtype, rows + n + k)
    got = linear.linear(x, w)
    _check(got, x, w, None, dtype)
    assert torch.equal(got, linear.linear(x, w))                   # the order of the sums is fixed
    _check(linear.linear(x, w, bias), x, w, bias, dtype)
    assert torch.equal(got, linear.linear(x, w, library="hybrid"))


# odd numbers of groups of 8 rows of w (3: 24 columns apiece, 5: 40), with a last tile that lacks groups or part of one; k of more steps than wavefronts, of which
# tiles begin anywhere
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [4, 16, 32, 64])
@pytest.mark.parametrize("n,k", [(4608, 1216), (4601, 704), (6144, 576), (6139, 1088), (10240, 832), (10236, 640), (10203, 1344)])
def test_odd_numbers_of_groups_and_tiles_that_begin_anywhere(n, k, rows, dtype):
    x, w, bias = _operands(rows, n, k, dtype, rows + n + k)
    got = linear.linear(x, w, bias)
    _check(got, x, w, bias, dtype)
    assert torch.equal(got, linear.linear(x, w, bias))
    if n % 2 == 0:
        a, b = (linear.linear(x, part, half) for part, half in zip(w.chunk(2), bias.chunk(2)))
        want = torch.nn.functional.silu(a.double()) * b.double()
        # silu's slope is at most 1.1; both products of either side are rounded (and their sums differ by less), then silu and the result
        bound = EPS[dtype] * (2.2 * a.double().abs() * b.double().abs() + 3.2 * want.abs()) + 1e-2 * EPS[dtype]
        assert ((linear.silu_product(x, w, bias, True).double() - want).abs() <= bound).all()


# n that is no multiple of 8: the last group of 8 columns is moved back over the one before it.  1985, 1988, 1028, 68 and 32003: the last group alone in a tile that begins
# elsewhere along k than the one before; 6139, 10236, 4601: in one tile with it
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [5, 16, 32, 64])
@pytest.mark.parametrize("n,k", [(68, 4096), (1028, 4096), (1985, 2048), (1988, 2048), (4601, 1024), (6139, 1088), (10236, 640), (32003, 1024)])
def test_every_column_has_one_writer(n, k, rows, dtype):
    """The second half of k takes back what the first half added, so that results are what rounding left of their sums and no two orders give the same.  Rows of zeros up to
    the next multiple of 8 change neither tiles nor beginnings, and no group is moved: the bits are the same."""
    x, w, bias = _operands(rows, n, k // 2, dtype, rows + n + k)
    x, w = torch.cat([x, x], 1) * 16, torch.cat([w, -w], 1) * 16
    padded = torch.nn.functional.pad(w, (0, 0, 0, -n % 8))

    def product(w):     # linear.linear sends the widest to the general product
        out = torch.empty(rows, w.shape[0], dtype=dtype, device=DEV)
        _lib.check(_lib.load().trimkv_linear_rows(x.data_ptr(), k, w.data_ptr(), k, None, out.data_ptr(), w.shape[0], rows, w.shape[0], k, _lib.dtype_code(dtype),
                                                  _lib.current_stream(x.device)), "product")
        return out
    got, want = product(w), product(padded)[:, :n]
    assert (want[:, -8:] != 0).any(1).all()
    assert torch.equal(got, want)
    if n <= 10236:
        x, gate, up = x * 64, w, w.roll(1, 0)
        got = linear.silu_product(x, torch.cat([gate, up]), None, False)
        want = linear.silu_product(x, torch.cat([torch.nn.functional.pad(t, (0, 0, 0, -n % 8)) for t in (gate, up)]), None, False)[:, :n]
        assert torch.equal(got, want)


# what linear.linear leaves to the general product is still the entry point's to take
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,n,k", [(33, 12289, 64), (64, 16384, 128), (64, 24576, 64), (50, 24600, 128), (64, 50002, 64)])
def test_many_rows_of_wide_matrices(rows, n, k, dtype):
    x, w, bias = _operands(rows, n, k, dtype, rows + n + k)
    assert torch.equal(linear.linear(x, w, bias), nn.functional.linear(x, w, bias)) and n > linear.WIDE and rows > linear.WIDE_ROWS
    out = torch.empty(rows, n, dtype=dtype, device=DEV)
    _lib.check(_lib.load().trimkv_linear_rows(x.data_ptr(), k, w.data_ptr(), k, bias.data_ptr(), out.data_ptr(), n, rows, n, k, _lib.dtype_code(dtype), _lib.current_stream(x.device)), "wide")
    _check(out, x, w, bias, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("round_all", [True, False])
@pytest.mark.parametrize("rows,inter,k", [(1, 1, 64), (3, 17, 128), (8, 100, 192), (16, 2049, 64), (16, 6144, 128), (32, 12288, 64), (40, 40, 576), (64, 1000, 64), (64, 6144, 128), (61, 12288, 64), (64, 20000, 64)])
def test_linear_rows_silu_matches_the_two_products(rows, inter, k, round_all, dtype):
    x, w, bias = _operands(rows, 2 * inter, k, dtype, rows + inter)
    for b in (None, bias):
        got = linear.silu_product(x, w, b, round_all)
        exact = x.double() @ w.double().T + (0 if b is None else b.double())
        size = (x.double().abs() @ w.double().abs().T) * (k * 2.0 ** -23)
        (g, u), (dg, du) = exact.chunk(2, -1), size.chunk(2, -1)
        act = torch.nn.functional.silu(g)
        # silu's slope is at most 1.1; g, u, silu(g) and the result are rounded (round_all) or the result alone
        dg, du = dg + EPS[dtype] * g.abs() * round_all, du + EPS[dtype] * u.abs() * round_all
        bound = 1.1 * dg * (u.abs() + du) + act.abs() * du + EPS[dtype] * (1 + round_all) * (act * u).abs() + 1e-5 * (act * u).abs() + 2.0 ** -24
        err = (got.double() - act * u).abs()
        assert (err <= bound).all(), float((err - bound).max())


@pytest.mark.gpu
def test_rows_that_are_slices_and_what_goes_to_the_general_product():
    x, w, bias = _operands(20, 300, 256, torch.bfloat16, 5)
    wide = torch.zeros(20, 1, 320, dtype=torch.bfloat16, device=DEV)
    wide[..., 64:] = x[:, None]
    big = torch.zeros(340, 264, dtype=torch.bfloat16, device=DEV)
    big[40:, 8:] = w
    want = linear.linear(x, w, bias)
    assert torch.equal(linear.linear(wide[..., 64:], big[40:, 8:], bias)[:, 0], want)
    takes = lambda *a: linear._rows(*a) is not None
    assert takes(x, w, bias) and takes(wide[..., 64:], big[40:, 8:], bias)
    assert not takes(wide[..., 60:], big[40:, 4:], None)                    # 260 features, and not 16-byte aligned
    assert not takes(wide[:, 0, 4:260], w, None)                            # 8 bytes off
    assert not takes(torch.cat([x] * 4), w, None)                           # 80 rows
    assert not takes(x[:0], w, None) and not takes(x.float(), w.float(), None) and not takes(x, w.half(), None)
    assert not takes(x, w.t().contiguous().t(), None)                       # columns are contiguous
    for args in ((wide[:, 0, 4:260], w), (torch.cat([x] * 4), w), (x[:0], w), (x, w.t().contiguous().t()), (x.float(), w.float())):
        assert linear.linear(*args).shape == (args[0].shape[0], 300)
    with torch.enable_grad():
        p = nn.Parameter(w.clone())
        assert not takes(x, p, None)
        linear.linear(x, p).float().sum().backward()
        assert p.grad is not None
    with torch.autocast("cuda", dtype=torch.float16):
        assert linear.linear(x, w).dtype == torch.float16


@pytest.mark.gpu
def test_linear_rows_on_a_stream_and_replayed_from_a_graph():
    x, w, _ = _operands(16, 4608, 256, torch.bfloat16, 9)
    want = linear.linear(x, w)
    gate = linear.silu_product(x, w)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            out, act = linear.linear(x, w), linear.silu_product(x, w)
    for i in range(3):
        out.zero_(), act.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(act, gate), i


# fewer outputs than a block has rows, in fours: the lanes of the columns that are not there store nothing
@pytest.mark.gpu
@pytest.mark.parametrize("n", [4, 8, 12])
@pytest.mark.parametrize("form,rows,dtype", [(form, rows, dtype) for form in ("plain", "silu", "norm", "norm silu") for rows in (1, 3, 16, 32, 33, 64) for dtype in (torch.bfloat16, torch.float16)
                                             if "norm" not in form or (rows <= linear.NORM_ROWS and dtype == torch.bfloat16)])
def test_outputs_narrower_than_a_block_stay_inside_of_their_rows(form, n, rows, dtype):
    k, lib, silu = 128, _lib.load(), "silu" in form
    x, w, bias = _operands(rows, n * (1 + silu), k, dtype, rows + n)
    out = torch.full((rows * n + 64,), 7.0, dtype=dtype, device=DEV)
    tail, at = (_lib.dtype_code(dtype), _lib.current_stream(x.device)), (w.data_ptr(), k, bias.data_ptr(), out.data_ptr(), n, rows, n, k)
    if "norm" in form:
        norm = torch.ones(k, dtype=dtype, device=DEV)
        squares = x.float().pow(2).view(rows, k // 8, 8).sum(-1)
        _lib.check(lib.trimkv_linear_rows_norm(x.data_ptr(), k, squares.data_ptr(), norm.data_ptr(), 1e-6, *at, int(silu), 1, *tail), form)
        x = (x.double() * torch.rsqrt(squares.double().sum(-1, keepdim=True) / k + 1e-6)).to(dtype)
    elif silu:
        _lib.check(lib.trimkv_linear_rows_silu(x.data_ptr(), k, *at, 1, *tail), form)
    else:
        _lib.check(lib.trimkv_linear_rows(x.data_ptr(), k, *at, *tail), form)
    assert (out[rows * n:] == 7.0).all()
    eps = EPS[dtype]
    exact, size = x.double() @ w.double().T + bias.double(), x.double().abs() @ w.double().abs().T
    slack = size * (k * 2.0 ** -23 + 2 * eps * ("norm" in form)) + 2.0 ** -24      # order of the sums; a normed row's last bit or two
    if silu:        # as in the test of the silu form, every step rounded
        (g, u), (dg, du) = exact.chunk(2, -1), (slack + eps * exact.abs()).chunk(2, -1)
        act = torch.nn.functional.silu(g)
        exact, slack = act * u, 1.1 * dg * (u.abs() + du) + act.abs() * du + (eps + 1e-5) * (act * u).abs()
    err = (out[:rows * n].view(rows, n).double() - exact).abs()
    assert (err <= slack + eps * exact.abs()).all(), float(err.max())


def test_bad_arguments_are_refused_without_a_launch():
    lib, one = _lib.load(), ctypes.c_void_p(16)
    call = lambda rows=4, n=16, k=64, xs=64, ws=64, os=16, x=one, w=one, dt=_lib.BF16: lib.trimkv_linear_rows(x, xs, w, ws, None, one, os, rows, n, k, dt, None)
    assert call(rows=65) == -2 and call(rows=0) == -2 and call(n=0) == -2 and call(k=96) == -2 and call(k=0) == -2
    assert call(xs=60) == -2 and call(ws=68) == -2 and call(os=8) == -2 and call(xs=1 << 25) == -2 and call(w=ctypes.c_void_p(24)) == -2
    assert call(x=None) == -1 and call(dt=_lib.F32) == -3
    assert lib.trimkv_linear_rows_silu(one, 64, one, 64, None, one, 8, 4, 16, 64, 1, _lib.BF16, None) == -2


def test_modules_that_somebody_hooked_wrapped_or_replaced_are_called():
    lin, x = nn.Linear(8, 4), torch.randn(2, 8)
    assert torch.equal(linear.run(lin, x), lin(x))
    seen = []
    hook = lin.register_forward_hook(lambda m, a, out: seen.append(out.shape) or out + 1)
    assert torch.equal(linear.run(lin, x), nn.functional.linear(x, lin.weight, lin.bias) + 1) and len(seen) == 1
    hook.remove()
    lin.forward = lambda y: y.sum()
    assert linear.run(lin, x) == x.sum()

    class Doubled(nn.Linear):
        def forward(self, y):
            return 2 * super().forward(y)
    twice = Doubled(8, 4)
    assert torch.equal(linear.run(twice, x), 2 * nn.functional.linear(x, twice.weight, twice.bias))
    from trimkv_amd import decoder_ops
    for other in (twice, nn.Sequential(nn.Linear(8, 4), nn.ReLU()), nn.Identity()):        # with a weight of its own or without
        assert torch.equal(decoder_ops.leave_or_run(other, x, True), other(x))


def test_a_packed_product_that_somebody_hooked_wrapped_or_replaced_is_called(monkeypatch):
    from trimkv_amd import hybrid
    mlp, xh, asked = hybrid.DenseMLP({"ff": 8}, 64, torch.float32), torch.randn(3, 64), []
    nn.init.normal_(mlp.gate_up.weight), nn.init.normal_(mlp.down.weight)
    monkeypatch.setattr(hybrid, "silu_product", lambda x, w, **kw: asked.append(w) or torch.zeros(len(x), 8))          # as if it took every product
    monkeypatch.setattr(hybrid.ops, "silu_gate", lambda both, ff: nn.functional.silu(both[:, :ff]) * both[:, ff:])
    want = lambda scale: mlp.down(hybrid.ops.silu_gate(scale * nn.functional.linear(xh, mlp.gate_up.weight), 8))
    assert torch.equal(mlp(None, xh)[0], torch.zeros(3, 64)) and len(asked) == 1
    hook = mlp.gate_up.register_forward_hook(lambda m, a, out: 2 * out)
    assert torch.equal(mlp(None, xh)[0], want(2))
    hook.remove()
    mlp.gate_up.forward = lambda x: 3 * nn.functional.linear(x, mlp.gate_up.weight)
    assert torch.equal(mlp(None, xh)[0], want(3))
    del mlp.gate_up.forward

    class Quadrupled(hybrid.PackedLinear):
        def forward(self, x):
            return 4 * super().forward(x)
    mlp.gate_up.__class__ = Quadrupled
    assert torch.equal(mlp(None, xh)[0], want(4)) and len(asked) == 1


def test_modules_with_a_forward_of_their_own_are_not_asked_to_leave_a_product():
    """Subclasses written before there was such an argument: the decoder calls them as it always did."""
    from trimkv_amd import qwen3
    from tests.test_gpu_qwen3_shell import _family, _tiny_config
    cfg = _tiny_config("qwen3")
    torch.manual_seed(0)
    model = _family("qwen3")[1](cfg).eval()
    layer, above = model.model.layers[:2]
    assert all(linear.may_leave(m) for m in (layer, layer.mlp, layer.self_attn))

    class OwnMLP(qwen3.MLP):
        def forward(self, x):
            return 2 * super().forward(x)

    class OwnAttention(type(layer.self_attn)):
        def forward(self, hidden_states, position_embeddings, attention_mask, past_key_values, cache_position):
            return torch.zeros_like(hidden_states)

    class OwnLayer(type(layer)):
        def forward(self, hidden_states, position_embeddings, attention_mask, past_key_values, cache_position, pending=None):
            return hidden_states + pending, torch.ones_like(hidden_states)
    above.__class__, layer.mlp.__class__, layer.self_attn.__class__ = OwnLayer, OwnMLP, OwnAttention
    assert not any(linear.may_leave(m) for m in (above, layer.mlp, layer.self_attn))
    with torch.no_grad():
        h, mlp = torch.randn(1, 6, cfg.hidden_size), layer.mlp
        total, out = layer(h, (None, None), None, None, None, leave_product=True)
        x = layer.post_attention_layernorm(h)
        assert torch.equal(total, h) and torch.allclose(out, 2 * mlp.down_proj(nn.functional.silu(mlp.gate_proj(x)) * mlp.up_proj(x)))
        assert torch.equal(above(total, None, None, None, None, out)[0], h + out)


@pytest.mark.parametrize("outputs", [128, 1024])
def test_a_product_of_another_width_than_the_residual_is_refused(outputs, monkeypatch):
    """A last product replaced by a wider or narrower one: the sum raises, as modules do; no launch adds past a row's end."""
    from trimkv_amd import qwen3
    from tests.test_gpu_qwen3_shell import _family, _tiny_config
    cfg = _tiny_config("qwen3")
    layer = _family("qwen3")[1](cfg).eval().model.layers[0]
    launched = []
    monkeypatch.setattr(linear, "can_defer_norm", lambda weight, residual: True)          # as if all of this were on a GPU
    monkeypatch.setattr(linear, "add_product", lambda p, residual: launched.append(p) or (residual, residual))
    monkeypatch.setattr(qwen3.MLP, "takes_deferred", lambda self, x: True)
    norm, hidden = layer.post_attention_layernorm, cfg.hidden_size
    x, residual = torch.randn(1, 2, 48), torch.randn(1, 2, hidden)
    with pytest.raises(RuntimeError, match="must match"):
        layer._add_norm(norm, linear.DeferredProduct(x, nn.Linear(48, outputs)), residual, layer.mlp)
    with pytest.raises(RuntimeError, match="must match"):        # ... or more rows
        layer._add_norm(norm, linear.DeferredProduct(torch.randn(1, 3, 48), nn.Linear(48, hidden)), residual, layer.mlp)
    # ... and a product of another type than the residual is added as tensors of two types are
    assert layer._add_norm(norm, linear.DeferredProduct(x, nn.Linear(48, hidden)), residual.double(), layer.mlp)[1].dtype == torch.float64
    assert not launched
    layer._add_norm(norm, linear.DeferredProduct(x, nn.Linear(48, hidden)), residual, layer.mlp)
    assert len(launched) == 1


@pytest.mark.gpu
def test_who_follows_operations_gets_the_general_product():
    from torch.autograd import forward_ad
    from torch.utils.flop_counter import FlopCounterMode
    x, w, bias = _operands(8, 64, 128, torch.bfloat16, 9)
    with torch.no_grad():
        want = nn.functional.linear(x, w, bias)
        assert torch.equal(torch.func.vmap(lambda row: linear.linear(row, w, bias))(x), torch.func.vmap(lambda row: nn.functional.linear(row, w, bias))(x))
        assert linear._rows(x, w, bias) is not None
        with forward_ad.dual_level():
            tangent = forward_ad.unpack_dual(linear.linear(forward_ad.make_dual(x, torch.ones_like(x)), w)).tangent
        assert torch.equal(tangent, nn.functional.linear(torch.ones_like(x), w))
        with FlopCounterMode(display=False) as counted:
            assert torch.equal(linear.linear(x, w, bias), want)
        assert counted.get_total_flops() == 2 * x.shape[0] * w.numel()
        traced = torch.jit.trace(lambda t: linear.linear(t, w, bias), x, check_trace=False)
        assert torch.equal(traced(x + 1), nn.functional.linear(x + 1, w, bias))


def test_function_modes_follow_operations_and_a_default_device_does_not():
    from torch.overrides import TorchFunctionMode

    class Counting(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    assert not linear.watched()
    with torch.device("cpu"):
        assert not linear.watched()
        with Counting():
            assert linear.watched()
    assert not linear.watched()


def _normed(x, norm):
    """What the modules make of x, in 64 bits between their two roundings."""
    h = x.double() * torch.rsqrt(x.double().square().mean(-1, keepdim=True) + norm.variance_epsilon)
    return (h.to(torch.bfloat16).double() * norm.weight.double()).to(torch.bfloat16)


# rows: every number of row groups and their edges; n: every number of blocks per tile, a last tile that is moved back, more tiles than
# workgroups; k: fewer steps than wavefronts, numbers that do not divide among them
@pytest.mark.gpu
@pytest.mark.parametrize("rows,n,k", [(1, 64, 64), (3, 320, 8192), (8, 4608, 192), (9, 112, 576), (16, 4624, 1024), (17, 64, 2048), (32, 2048, 704), (29, 8192, 128), (32, 8208, 64), (5, 50000, 64), (16, 2048, 128), (8, 2064, 64), (1, 16, 64)])
def test_linear_rows_with_a_residual(rows, n, k):
    x, w, bias = _operands(rows, n, k, torch.bfloat16, rows + n + k)
    wide = torch.zeros(rows, 1, n + 4, dtype=torch.bfloat16, device=DEV)
    wide[..., 4:] = torch.randn(rows, 1, n, generator=torch.Generator(device=DEV).manual_seed(k), device=DEV) * 3
    res = wide[..., 4:]
    for b in (None, bias):
        out, squares = torch.empty(rows, n, dtype=torch.bfloat16, device=DEV), torch.full((rows, n // 8), float("nan"), device=DEV)
        _lib.check(_lib.load().trimkv_linear_rows_add(x.data_ptr(), k, w.data_ptr(), k, _lib.ptr(b), res.data_ptr(), n + 4, out.data_ptr(), n, squares.data_ptr(),
                                                      rows, n, k, _lib.BF16, _lib.current_stream(x.device)), "trimkv_linear_rows_add")
        assert torch.equal(out, linear.linear(x, w, b) + res[:, 0])
        want = out.double().square().view(rows, n // 8, 8).sum(-1)
        assert ((squares.double() - want).abs() <= 8 * 2.0 ** -24 * want).all()


@pytest.mark.gpu
@pytest.mark.parametrize("silu", [False, True])
@pytest.mark.parametrize("rows,n,k", [(1, 1, 64), (3, 40, 8192), (8, 4608, 192), (9, 100, 576), (16, 4616, 1024), (16, 12288, 64), (17, 33, 2048), (32, 2048, 704), (29, 9000, 128), (32, 12300, 64),
                                      (5, 70001, 64), (16, 50000, 128)])
def test_linear_rows_behind_a_norm(rows, n, k, silu):
    """Against the norm in 64 bits with the modules' roundings: where the two disagree on a rounding, an element of the operand differs by
    2^-7 of itself; each product is allowed that."""
    from trimkv_amd.qwen3 import RMSNorm
    x, w, bias = _operands(rows, (2 if silu else 1) * n, k, torch.bfloat16, rows + n + k)
    x = (x.float() * 30).to(torch.bfloat16)
    norm = RMSNorm(k, 1e-6).to(torch.bfloat16).to(DEV)
    norm.weight.data.normal_(1.0, 0.3, generator=torch.Generator(device=DEV).manual_seed(k))
    h = _normed(x, norm)
    squares = x.float().square().view(rows, k // 8, 8).sum(-1)
    for b in (None, bias):
        with torch.no_grad():
            d = linear.DeferredNorm(x, squares, norm)
            got = linear.norm_product(d, w, b, silu)
            plain = linear.silu_product(h, w, b) if silu else linear.linear(h, w, b)
            assert (got != plain).float().mean() < 0.2                       # nearly always the very same operand
            d.tensor()
            assert linear.norm_product(d, w, b, silu) is None               # taken already
        exact = h.double() @ w.double().T + (0 if b is None else b.double())
        size = (h.double().abs() @ w.double().abs().T) * (2.0 ** -7 * min(1.0, 64 / k) + k * 2.0 ** -23)
        if not silu:
            bound = EPS[torch.bfloat16] * exact.abs() + size + 2.0 ** -24
        else:
            (g, u), (dg, du) = exact.chunk(2, -1), size.chunk(2, -1)
            exact, act = torch.nn.functional.silu(g) * u, torch.nn.functional.silu(g)
            dg, du = dg + EPS[torch.bfloat16] * g.abs(), du + EPS[torch.bfloat16] * u.abs()
            bound = 1.1 * dg * (u.abs() + du) + act.abs() * du + 2 * EPS[torch.bfloat16] * exact.abs() + 1e-5 * exact.abs() + 2.0 ** -24
        err = (got.double() - exact).abs()
        assert (err <= bound).all(), float((err - bound).max())


@pytest.mark.gpu
def test_what_is_not_left_to_a_product():
    x, w, bias = _operands(16, 320, 256, torch.bfloat16, 5)
    lin = nn.Linear(256, 320, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        takes = linear.can_defer_product
        assert takes(lin, x) and takes(lin, x[:, None]) and not takes(lin, torch.cat([x] * 3)) and not takes(nn.Linear(256, 300, device=DEV, dtype=torch.bfloat16), x)
        assert not takes(lin.half(), x.half())
        lin = lin.to(torch.bfloat16)
        hook = lin.register_forward_hook(lambda m, a, out: out)
        assert not takes(lin, x)
        hook.remove()
        weight, res = torch.ones(256, dtype=torch.bfloat16, device=DEV), torch.zeros(16, 512, dtype=torch.bfloat16, device=DEV)
        assert linear.can_defer_norm(weight, x) and not linear.can_defer_norm(weight, res[:, :256]) and not linear.can_defer_norm(weight.half(), x) and not linear.can_defer_norm(weight[:8], x)
    assert not takes(lin, x)                                                # somebody differentiates


def test_bad_arguments_around_a_norm_are_refused_without_a_launch():
    lib, one = _lib.load(), ctypes.c_void_p(16)
    norm = lambda rows=4, k=64, sq=one, nw=one, dt=_lib.BF16: lib.trimkv_linear_rows_norm(one, k, sq, nw, 1e-6, one, k, None, one, 16, rows, 16, k, 0, 1, dt, None)
    assert norm(rows=33) == -2 and norm(k=8256) == -2 and norm(nw=ctypes.c_void_p(24)) == -2 and norm(sq=ctypes.c_void_p(20)) == -2 and norm(sq=None) == -1 and norm(nw=None) == -1 and norm(dt=_lib.F16) == -3
    add = lambda rows=4, n=16, rs=16, os=16, res=one, sq=one, dt=_lib.BF16: lib.trimkv_linear_rows_add(one, 64, one, 64, None, res, rs, one, os, sq, rows, n, 64, dt, None)
    assert add(rows=33) == -2 and add(n=24, rs=24, os=24) == -2 and add(rs=12) == -2 and add(rs=18) == -2 and add(os=18) == -2 and add(res=ctypes.c_void_p(20)) == -2
    assert add(res=None) == -1 and add(sq=None) == -1 and add(dt=_lib.F32) == -3


@pytest.mark.gpu
@pytest.mark.parametrize("family,gate", [("qwen3", "rg"), ("qwen3", "rg2"), ("llama", "rg"), ("phi3", "rg")])
def test_decode_steps_leave_adds_and_norms_to_the_products(family, gate, monkeypatch):
    """Logits of decode steps with and without launches of their own for adds and norms, to rounding; hooks see what they saw."""
    from trimkv_amd import qwen3
    from tests.test_gpu_qwen3_shell import _family, _tiny_config
    cfg = _tiny_config(family, retention_gate=gate)
    torch.manual_seed(0)
    model = _family(family)[1](cfg).to(torch.bfloat16).to(DEV).eval()
    ids = torch.randint(0, cfg.vocab_size, (2, 40), generator=torch.Generator().manual_seed(4)).to(DEV)
    taken, plain = [], linear.norm_product

    def steps():
        with torch.no_grad():
            out, logits = model(ids[:, :30]), []
            for i in range(30, 34):
                out = model(ids[:, i:i + 1], past_key_values=out.past_key_values)
                logits.append(out.logits[:, -1].float())
        return torch.stack(logits)
    monkeypatch.setattr(linear, "norm_product", lambda *a: (lambda out: taken.append(out is not None) or out)(plain(*a)))
    got = steps()
    assert sum(taken) == len(taken) == 4 * (cfg.num_hidden_layers if family == "phi3" else 2 * cfg.num_hidden_layers - 1)
    monkeypatch.setattr(linear, "can_defer_product", lambda *a: False)
    want = steps()
    assert (got - want).abs().max() <= 2e-2 + 2e-2 * want.abs().max()
    monkeypatch.undo()
    seen = []
    handles = [model.model.layers[1].register_forward_hook(lambda m, a, out: seen.append(type(out[1]))), model.model.layers[0].mlp.register_forward_hook(lambda m, a, out: seen.append(type(out))),
               model.model.layers[1].self_attn.register_forward_hook(lambda m, a, out: seen.append(type(out))), model.model.layers[0].self_attn.o_proj.register_forward_hook(lambda m, a, out: seen.append(type(out)))]
    hooked = steps()
    assert seen == [torch.Tensor] * 20 and (hooked - want).abs().max() <= 2e-2 + 2e-2 * want.abs().max()
    for handle in handles:
        handle.remove()
