"""trimkv_linear_f32_tiles (a linear layer over the rows of a prompt in fp32, on bf16 matrix instructions) against 64-bit products.

Bounds: fp32 sums of k products err by at most about k 2^-24 sum |x w| in any order (twice that here); the three of nine products of bf16 terms that are left
out are at most 3 * 2^-25 of |x w|.  Roundings of a sum point either way: of 6 k / 128 additions by a wavefront each is off by 2^-24 / sqrt(3) of a sum that grows as the root,
so that the 2-norm of the errors is about 2^-24 sqrt(k / 64) of that of sums of independent products, 3.4e-7 for k = 2048 (3.5e-7 measured; 1e-6 here).  Without one of the six
products of terms it is 2.5e-6 and more, whatever k is.  Results below 2^-126 are multiples of 2^-149."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

from trimkv_amd import _lib, linear

DEV = "cuda:0"
FORMS = range(1, 14)


def _operands(rows, n, k, seed=0, pad=0):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(rows, k + pad, generator=gen, device=DEV)[:, :k], torch.randn(n, k + pad, generator=gen, device=DEV)[:, :k] * 0.1


def _tiles(x, w, form, pad=0):
    (rows, k), n = x.shape, w.shape[0]
    out = torch.full((rows + 1, n + pad), 7.0, device=DEV)
    _lib.check_hybrid(_lib.load_hybrid().trimkv_linear_f32_tiles(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), out.data_ptr(), n + pad, rows, n, k, form,
                                                                 _lib.current_stream(x.device)), "trimkv_linear_f32_tiles")
    assert (out[rows] == 7).all() and (out[:, n:] == 7).all()      # nothing behind the rows and columns there are
    return out[:rows, :n]


def _check(got, x, w, tiny=0.0):
    exact, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    err = (got.double() - exact).abs()
    bound = (x.shape[1] * 2.0 ** -23 + 2.0 ** -22) * size + tiny
    assert (err <= bound).all(), (float((err - bound).max()), (err > bound).nonzero()[:4].tolist())
    usual = (x.double().square() @ w.double().square().T).sum().sqrt()        # the results' 2-norm if products had random signs
    assert err.norm() <= 1e-6 * usual + tiny * err.numel() ** 0.5, float(err.norm() / usual)


# rows and n on either side of blocks of 16 and of tiles; fewer and more steps of 32 k than wavefronts, remainders, one period and several; rows that do not lie side by side
@pytest.mark.gpu
@pytest.mark.parametrize("rows,n,k,pad", [(1, 1, 32, 0), (15, 17, 64, 4), (16, 64, 96, 0), (17, 65, 128, 1), (31, 48, 160, 0), (33, 97, 256, 3), (48, 144, 288, 0), (49, 145, 32, 4), (64, 160, 512, 0),
                                          (65, 161, 544, 8), (97, 129, 1024, 0), (300, 500, 416, 2), (811, 264, 192, 0), (200, 300, 2048, 0), (130, 170, 4096, 0)])
def test_every_form_matches_the_product(rows, n, k, pad):
    x, w = _operands(rows, n, k, rows + n + k, 4 * (pad % 3))
    for form in [*FORMS, 0]:
        got = _tiles(x, w, form, pad)
        _check(got, x, w)
        assert torch.equal(_tiles(x, w, form, pad), got), form      # a buffer read too early or too late does not repeat itself


@pytest.mark.gpu
@pytest.mark.parametrize("form", [1, 5, 13])
def test_what_bf16_terms_do_not_hold(form):
    """Infinities, NaN and numbers that round to infinity in bf16 give what fp32 products give."""
    x, w = _operands(130, 200, 256, 3)
    x, w = x.contiguous(), w.contiguous()
    x[5, 7], x[20, 100], x[21, 3], x[64, 0], x[129, 255] = torch.inf, -torch.inf, torch.nan, 3.4e38, -3.4e38
    w[11, 9], w[150, 30], w[199, :] = torch.inf, 3.399e38, 0.0
    got, want = _tiles(x, w, form), F.linear(x.cpu(), w.cpu()).to(DEV)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isposinf(), want.isposinf()) and torch.equal(got.isneginf(), want.isneginf())
    keep = want.isfinite()
    exact, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    assert ((got.double() - exact).abs() <= 256 * 2.0 ** -23 * size)[keep].all()
    x, w = _operands(40, 70, 128, 4)
    _check(_tiles((x * 2.0 ** 100).contiguous(), w, form), x * 2.0 ** 100, w)


@pytest.mark.gpu
@pytest.mark.parametrize("form", FORMS)
def test_terms_hold_all_bits(form):
    """One product to a sum, of a number of 24 bits with a power of two: exactly that number times it, on either side, wherever in k it stands."""
    rows, n, k = 100, 170, 416
    gen = torch.Generator(device=DEV).manual_seed(form)
    bits = lambda *s: (1 << 23 | torch.randint(0, 1 << 23, s, generator=gen, device=DEV)).float() * (torch.randint(0, 2, s, generator=gen, device=DEV) * 2 - 1) * 2.0 ** -20
    power = lambda *s: torch.exp2(torch.randint(-30, 30, s, generator=gen, device=DEV).float())
    at = torch.arange(rows, device=DEV) * 37 % k
    for one, other in ((bits, power), (power, bits)):
        x, w = torch.zeros(rows, k, device=DEV), other(n, k)
        x[torch.arange(rows, device=DEV), at] = one(rows)
        assert torch.equal(_tiles(x, w, form), x[torch.arange(rows, device=DEV), at, None] * w[:, at].T)
        at = torch.arange(n, device=DEV) * 37 % k
        x, w = other(rows, k), torch.zeros(n, k, device=DEV)
        w[torch.arange(n, device=DEV), at] = one(n)
        assert torch.equal(_tiles(x, w, form), x[:, at] * w[torch.arange(n, device=DEV), at])
        at = torch.arange(rows, device=DEV) * 37 % k


# 2^-103: the last number of which bf16 terms hold all; 2^-110 and less: of which they lose some; 2^-133 and less: all; 2^-149: the smallest there is
@pytest.mark.gpu
@pytest.mark.parametrize("form", [1, 2, 5, 8, 9, 12, 13])
def test_the_smallest_numbers(form):
    """Blocks with numbers that bf16 terms do not hold are done again, and nothing but these."""
    x, w = _operands(130, 200, 416, 4)
    x, w = x.contiguous(), w.contiguous()
    normal = _tiles(x, w, form)
    for e in (-60, -100, -103, -108, -112, -118, -126, -134, -145):
        small, great = x * 2.0 ** e, w * 2.0 ** 100
        _check(_tiles(small, great, form), small, great)
        _check(_tiles(great[:130].contiguous(), small, form), great[:130], small)
        _check(_tiles(small, w, form), small, w, tiny=416 * 2.0 ** -148)
    for r, c in ((0, 0), (77, 300), (129, 415)):        # the only number of its row, against large ones
        a, b = x.clone(), w.clone()
        a[r], b[:, c] = 0, b[:, c] * 2.0 ** 120
        a[r, c] = 1.2345678 * 2.0 ** -121
        got = _tiles(a, b, form)
        _check(got, a, b)
        assert torch.equal(got[r], a[r, c] * b[:, c])
        a, b = x.clone(), w.clone()
        b[r], a[:, c] = 0, a[:, c] * 2.0 ** 120
        b[r, c] = -1.7654321 * 2.0 ** -130
        got = _tiles(a, b, form)
        _check(got, a, b)
        assert torch.equal(got[:, r], a[:, c] * b[r, c])
    zeros = x.clone()
    zeros[::3, ::2] = 0
    _check(_tiles(zeros, w, form), zeros, w)
    assert torch.equal(_tiles(x, w, form), normal)


@pytest.mark.gpu
def test_linear_takes_it_where_it_is_faster():
    """Linear layers of the hybrid decoders in fp32: the tiles from a few hundred rows on, else, and for operands of another form, the general product."""
    calls, lib = [], _lib.load_hybrid()
    real = lib.trimkv_linear_f32_tiles

    class Spy:
        def __getattr__(self, name):
            return (lambda *a: calls.append(a[6:9]) or real(*a)) if name == "trimkv_linear_f32_tiles" else getattr(lib, name)
    _lib._hybrid["hybrid"] = Spy()
    try:
        x, w = _operands(811, 2048, 2048, 5)
        x, w = x.contiguous(), w.contiguous()
        taken = lambda x, w, **kw: (calls.clear(), linear.linear(x, w, library="hybrid", **kw), len(calls))[1:]
        for a, took in ((x, 1), (x.view(1, 811, 2048), 1), (x[:20], 0), (x[:, :2000], 0), (x.t().contiguous().t(), 0), (x[:, 1:], 0)):
            b = w if a.shape[-1] == 2048 else w[:, :a.shape[-1]]
            got, n = taken(a, b)
            assert n == took, (a.shape, a.stride())
            _check(got.reshape(-1, 2048), a.reshape(-1, a.shape[-1]), b)
        assert taken(x, w, bias=torch.zeros(2048, device=DEV))[1] == 0
        with torch.autocast("cuda", dtype=torch.bfloat16):
            got, n = taken(x, w)
        assert n == 0 and got.dtype == torch.bfloat16
        y = x.clone().requires_grad_()
        got, n = taken(y, w)
        assert n == 0 and got.requires_grad
        got, n = taken(torch.empty(0, 2048, device=DEV), w)
        assert n == 0 and got.shape == (0, 2048)
    finally:
        _lib._hybrid["hybrid"] = lib


def test_other_devices_need_no_library(monkeypatch):
    def missing(*_):
        raise _lib.TrimKVLibraryError("missing")
    monkeypatch.setattr(_lib, "load_hybrid", missing)
    linear._f32_form.cache_clear()
    x, w = torch.randn(300, 64), torch.randn(96, 64)
    assert torch.equal(linear.linear(x, w, library="hybrid"), F.linear(x, w))
    assert linear.linear(x.to("meta"), w.to("meta"), library="hybrid").shape == (300, 96)


def test_bad_calls_are_refused():
    lib = ctypes.CDLL(_lib.HYBRID_LIB_PATHS["hybrid"])
    fn = lib.trimkv_linear_f32_tiles
    fn.argtypes = _lib.HYBRID_SIGNATURES["hybrid"]["trimkv_linear_f32_tiles"][1]
    one = ctypes.c_void_p(64)
    call = lambda rows=400, n=16, k=64, xs=64, ws=64, os=16, x=one, w=one, o=one, form=0: fn(x, xs, w, ws, o, os, rows, n, k, form, None)
    assert call(x=None) == -1 and call(w=None) == -1 and call(o=None) == -1
    for kw in (dict(rows=0), dict(n=0), dict(k=0), dict(k=48), dict(xs=63), dict(ws=60), dict(xs=66), dict(xs=1 << 21), dict(os=15), dict(rows=1 << 23), dict(x=ctypes.c_void_p(68)),
               dict(o=ctypes.c_void_p(66)), dict(form=14), dict(form=-1)):
        assert call(**kw) == -2, kw
    form = lib.trimkv_linear_f32_tiles_form
    assert form(0, 64, 64) == 0 and form(64, 64, 48) == 0 and form(20, 2048, 2048) == 0 and form(811, 2048, 2048) > 0
