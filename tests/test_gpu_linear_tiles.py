"""trimkv_linear_tiles and trimkv_linear_tiles_silu (a linear layer over the rows of a prompt) against 64-bit products.

Bounds: fp32 sums of k products err by at most about k 2^-24 sum |x w| (any order), the result is rounded once (half a unit in the
last place, 2^-9 of the value in bf16; twice that here, for values that straddle)."""
import ctypes
import random

import pytest
import torch
from torch import nn

from trimkv_amd import _lib, linear

DEV = "cuda:0"
EPS = 2.0 ** -8
FORMS = [1, 2, 3, 9, 10, 11, 17, 18, 19, 25, 26, 27, 4]      # tile heights of 256, 192, 128; rows, columns, both behind whole tiles in small ones; small ones only


def _operands(rows, n, k, seed=0):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    made = lambda *shape: torch.randn(*shape, generator=gen, device=DEV).to(torch.bfloat16)
    return made(rows, k), made(n, k) * 0.1


def _tiles(x, w, form, silu=False, round_all=True, pad=0):
    rows, k = x.shape
    n = w.shape[0] // 2 if silu else w.shape[0]
    out = torch.full((rows + 1, n + pad), 7.0, dtype=x.dtype, device=DEV)
    at, tail = (x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), out.data_ptr(), n + pad, rows, n, k), (form, _lib.BF16, _lib.current_stream(x.device))
    lib = _lib.load()
    _lib.check(lib.trimkv_linear_tiles_silu(*at, int(round_all), *tail) if silu else lib.trimkv_linear_tiles(*at, *tail), "tiles")
    assert (out[rows] == 7).all() and (out[:, n:] == 7).all()      # nothing behind the rows and columns there are
    return out[:rows, :n]


def _check(got, x, w):
    exact, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    err = (got.double() - exact).abs()
    bound = EPS * exact.abs() + x.shape[1] * 2.0 ** -23 * size + 2.0 ** -24
    assert (err <= bound).all(), (float((err - bound).max()), (err > bound).nonzero()[:4].tolist())


# rows and n on either side of tile edges; one, two, three and more steps of 64 k than there are buffers; output strides that take stores of 16 bytes and that do not
@pytest.mark.gpu
@pytest.mark.parametrize("rows,n,k,pad", [(1, 1, 64, 0), (65, 127, 128, 1), (127, 128, 192, 0), (128, 129, 256, 8), (129, 255, 320, 0), (191, 256, 64, 8), (192, 257, 704, 7), (193, 384, 128, 0),
                                          (255, 385, 192, 7), (256, 512, 448, 0), (257, 640, 64, 8), (384, 264, 576, 0), (385, 1000, 128, 0), (1300, 520, 64, 0), (2049, 264, 192, 0)])
def test_every_form_matches_the_product(rows, n, k, pad):
    x, w = _operands(rows, n, k, rows + n + k)
    first = None
    for form in FORMS + [0]:
        got = _tiles(x, w, form, pad=pad)
        _check(got, x, w)
        first = got if first is None else first
        assert torch.equal(got, first), form                   # every form adds up in the same order
        assert torch.equal(_tiles(x, w, form, pad=pad), got)   # a buffer read too early or too late does not repeat itself


@pytest.mark.gpu
@pytest.mark.parametrize("round_all", [True, False])
@pytest.mark.parametrize("rows,inter,k,pad", [(1, 1, 64, 0), (65, 127, 128, 1), (128, 128, 192, 0), (129, 129, 320, 8), (192, 256, 64, 0), (257, 200, 704, 0), (385, 1000, 128, 8), (1025, 264, 192, 0)])
def test_every_silu_form_matches_the_two_products(rows, inter, k, pad, round_all):
    x, w = _operands(rows, 2 * inter, k, rows + inter)
    (g, u), (dg, du) = (t.chunk(2, -1) for t in (x.double() @ w.double().T, (x.double().abs() @ w.double().abs().T) * (k * 2.0 ** -23)))
    act = torch.nn.functional.silu(g)
    # silu's slope is at most 1.1; g, u, silu(g) and the result are rounded (round_all) or the result alone
    dg, du = dg + EPS * g.abs() * round_all, du + EPS * u.abs() * round_all
    bound = 1.1 * dg * (u.abs() + du) + act.abs() * du + EPS * (1 + round_all) * (act * u).abs() + 1e-5 * (act * u).abs() + 2.0 ** -24
    for form in (1, 2, 3, 0):
        got = _tiles(x, w, form, True, round_all, pad)
        err = (got.double() - act * u).abs()
        assert (err <= bound).all(), (form, float((err - bound).max()))


@pytest.mark.gpu
def test_operands_with_strides_and_values_that_are_not_finite():
    x, w = _operands(300, 200, 256, 3)
    wide, big = torch.full((300, 320), float("nan"), dtype=x.dtype, device=DEV), torch.full((240, 264), float("inf"), dtype=x.dtype, device=DEV)
    wide[:, 64:], big[40:, 8:] = x, w
    for form in FORMS:
        assert torch.equal(_tiles(wide[:, 64:], big[40:, 8:], form), _tiles(x, w, form))
    x[7, 5], x[200, 100], w[33, 9] = float("inf"), float("nan"), float("nan")
    for form in FORMS:
        got = _tiles(x, w, form)
        assert got[200].isnan().all() and got[:, 33].isnan().all() and not got[7].isfinite().any()
        rest = got[[i for i in range(300) if i not in (7, 200)]][:, [i for i in range(200) if i != 33]]
        assert rest.isfinite().all()


@pytest.mark.gpu
def test_which_products_of_many_rows_go_where():
    x, w = _operands(4096, 1536, 1024, 5)
    takes = lambda *a, silu=False: linear._tiles(*a, silu, None) is not None
    assert takes(x, w, None) and takes(x, w, None, silu=True)
    got = linear.linear(x, w)
    _check(got, x, w)
    assert torch.equal(got, _tiles(x, w, 0)) and torch.equal(got, linear.linear(x, w, library="hybrid"))
    assert torch.equal(linear.linear(x.view(4, 1024, 1024), w), got.view(4, 1024, 1536))
    assert torch.equal(linear.silu_product(x, w), _tiles(x, w, 0, True))
    assert torch.equal(linear.silu_product(x, w, round_all=False, library="hybrid"), _tiles(x, w, 0, True, False))
    lib = _lib.load()
    assert not lib.trimkv_linear_tiles_form(82, 2048, 2048, 0) and not lib.trimkv_linear_tiles_form(467, 2048, 6144, 0)      # too few tiles
    assert lib.trimkv_linear_tiles_form(8286, 6144, 2048, 0) and lib.trimkv_linear_tiles_form(1656, 4096, 4096, 0)
    for args in ((x[:70], w, None), (x.float(), w.float(), None), (x.half(), w.half(), None), (x, w, w[:, 0].contiguous()), (x, w.t().contiguous().t(), None),
                 (x.t().contiguous().t(), w, None), (x[:, 4:], w[:, 4:], None), (x.view(4, 1024, 1024).transpose(0, 1), w, None)):
        assert not takes(*args)
        assert torch.equal(linear.linear(*args), nn.functional.linear(*args))
    assert not takes(x, w[:1535], None, silu=True)
    with torch.enable_grad():
        p = nn.Parameter(w.clone())
        assert not takes(x, p, None)
        linear.linear(x, p).float().sum().backward()
        assert p.grad is not None
    assert torch.equal(torch.vmap(lambda t: linear.linear(t, w))(x.view(4, 1024, 1024)), torch.vmap(lambda t: nn.functional.linear(t, w))(x.view(4, 1024, 1024)))
    with torch.autocast("cuda", dtype=torch.float16):
        assert linear.linear(x, w).dtype == torch.float16


@pytest.mark.gpu
def test_on_a_stream_and_replayed_from_a_graph():
    x, w = _operands(4096, 1536, 1024, 9)
    assert linear._tiles(x, w, None, False, None) is not None
    want, gate = linear.linear(x, w), linear.silu_product(x, w)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            out, act = linear.linear(x, w), linear.silu_product(x, w)
    for _ in range(3):
        out.zero_(), act.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(act, gate)


def test_bad_arguments_are_refused_without_a_launch():
    lib, one = _lib.load(), ctypes.c_void_p(16)
    call = lambda rows=400, n=16, k=64, xs=64, ws=64, os=16, x=one, w=one, form=0, dt=_lib.BF16: lib.trimkv_linear_tiles(x, xs, w, ws, one, os, rows, n, k, form, dt, None)
    assert call(x=None) == -1 and call(dt=_lib.F16) == -3 and call(dt=_lib.F32) == -3
    for bad in (dict(rows=0), dict(n=0), dict(k=96), dict(k=0), dict(xs=60), dict(xs=68), dict(ws=56), dict(os=15), dict(x=ctypes.c_void_p(24)), dict(w=ctypes.c_void_p(20)),
                dict(xs=(1 << 20) + 8), dict(rows=(1 << 24) + 1), dict(form=5), dict(form=-1), dict(form=8), dict(form=33)):
        assert call(**bad) == -2, bad
    silu = lambda form: lib.trimkv_linear_tiles_silu(one, 64, one, 64, one, 16, 400, 16, 64, 1, form, _lib.BF16, None)
    assert silu(4) == -2 and silu(9) == -2
    assert lib.trimkv_linear_tiles_form(0, 64, 64, 0) == 0 and lib.trimkv_linear_tiles_form(64, 64, 32, 0) == 0


def test_sizes_are_asked_first(monkeypatch):
    """The host bounds prompts of a few hundred tokens: a product of too few outputs for tiles goes to the general one by its sizes alone."""
    asked = []
    monkeypatch.setattr(linear, "_plain", lambda *a: asked.append(a))
    for rows, n in ((65, 4096), (142, 6144), (300, 6300)):
        x, w = torch.randn(rows, 64).to(torch.bfloat16), torch.randn(n, 64).to(torch.bfloat16)
        assert torch.equal(linear.linear(x, w), torch.nn.functional.linear(x, w)) and linear.silu_product(x, w) is None and not asked
    assert torch.equal(linear.linear(x[:64], w), torch.nn.functional.linear(x[:64], w)) and asked      # a decode step's rows are


def test_few_outputs_are_never_done_on_tiles():
    """The line that is drawn by rows x outputs alone leaves nothing to the general product that the estimate of tiles would take."""
    rng = random.Random(5)
    for _ in range(60000):
        silu = rng.random() < 0.5
        k, n = 64 * round(2 ** rng.uniform(0, 11)), round(2 ** rng.uniform(0, 17))
        rows = (linear.LEAST_SILU_OUTPUTS if silu else linear.LEAST_OUTPUTS) * rng.uniform(0.5, 1) // n
        if rows >= 1:
            assert _lib.load().trimkv_linear_tiles_form(int(rows), n, k, int(silu)) == 0, (rows, n, k, silu)


@pytest.mark.parametrize("rows,n,k,silu,taken", [(680, 6144, 4096, 0, False), (1599, 3072, 8192, 0, False), (206, 8192, 3072, 1, False), (1409, 3072, 3072, 0, False), (4096, 1536, 1024, 0, True),
                                                 (613, 4112, 2048, 0, True), (1656, 4096, 4096, 0, True), (412, 12288, 2048, 1, True), (8192, 12288, 4096, 1, True)])
def test_products_of_long_k_need_more_of_the_chip(rows, n, k, silu, taken):
    """Sizes that were measured on either side of the rule's two lines: the general product divides k, and is faster where tiles leave compute units idle."""
    assert bool(_lib.load().trimkv_linear_tiles_form(rows, n, k, silu)) == taken
