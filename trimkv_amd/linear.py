"""Linear layers over the rows of a decode step on trimkv_linear_rows and over those of a prompt on trimkv_linear_tiles, those of the hybrid decoders in fp32 on
trimkv_linear_f32_tiles; everything else goes to ``F.linear``.

All give fp32 sums rounded once; the order of the sums differs.
"""
from __future__ import annotations

import functools
from typing import Optional

import torch
from torch import nn
import torch.nn.functional as F
from torch.autograd import forward_ad
from torch.nn.modules import module as _module
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

from . import _lib

MAX_ROWS = 64      # rows that trimkv_linear_rows takes
# More rows than WIDE_ROWS times more outputs than WIDE, heads of language models above all, are left to the general product.  us here | general, 33 rows, 48 and 64.  For it:
# 151936 x 5120 303 | 291, 324 | 295, 337 | 298; 128256 x 4096 205 | 206, 218 | 207, 221 | 209; 13824 x 5120 31.8 | 29.4, 33.4 | 30.6, 35.4 | 31.7; 100352 x 5120 209 | 280,
# 219 | 184, 233 | 215.  Alike or mixed: 34816 x 5120 78 | 80, 82 | 81, 86 | 86; 32064 x 3072 41.6 | 39.5, 42.4 | 52.3, 42.2 | 38.7; 151936 x 4096 241 | 254, 254 | 268, 260 | 259;
# 16384 x 3072 22.7 | 23.3, 22.8 | 23.6, 23.2 | 23.8.  Given up, since tiles take any number of 8 rows of w: 16384 x 4096 27 | 31 all three, 24576 x 4096 39 | 46, 28672 x 4096 47 | 51,
# 47 | 60, 49 | 52, 49152 x 2048 40 | 49, 41 | 48, 43 | 49, 151936 x 2048 130 | 153, 135 | 143, 141 | 152; a line in k as well as n would keep these.  Below it: 12288 x 4096 20 | 25,
# 21 | 25, 22 | 26, 8192 x 8192 27 | 31, 29 | 32, 31.5 | 31.7 (one row 22.6 | 28.6).  Up to 32 rows all are taken, in blocks of 16 rows of w then: 32064 x 3072 with 1, 16, 32 rows
# 31.5 | 41.0, 33.2 | 42.0, 39.4 | 37.1; 151936 x 2048 101 | 207, 109 | 208, 128 | 153; 151936 x 5120 238 | 307, 263 | 330, 319 | 364.
WIDE_ROWS, WIDE = 32, 12288


# Fewer rows x outputs than this are never done on tiles, whatever k is: they would fill less than half of the chip.  (trimkv_linear_tiles_form wants the
# operations at its rate for no less than a round of tiles takes by its estimate, 0.77 (1 + 0.49 k / 64) us, with silu 0.77 (1 + 0.83 k / 64).)  Sizes are asked before
# all else, because the host bounds prompts of a few hundred tokens: with the other checks in front 142 tokens through three layers of 2048 took 750 us
# for 615, through two layers with recurrence 337 for 298.
LEAST_OUTPUTS, LEAST_SILU_OUTPUTS = 1_900_000, 1_370_000


def watched() -> bool:
    """Somebody follows the operations themselves (vmap and torch.func, forward-mode derivatives, tracing, compiling, dispatch modes, function
    modes other than that of a default device): a launch of ours would be lost on them, and inside of vmap a tensor has no address."""
    return (torch.compiler.is_compiling() or torch._C._functorch.peek_interpreter_stack() is not None or forward_ad._current_level >= 0
            or torch._C._get_tracing_state() is not None or torch._C._len_torch_dispatch_stack() > 0
            or (torch._C._len_torch_function_stack() > 0 and any(type(mode) is not DeviceContext for mode in _get_current_function_mode_stack())))


def _plain(*tensors: Optional[torch.Tensor], dtypes=(torch.bfloat16, torch.float16)) -> bool:
    """Ordinary tensors of one dtype (of 16 bits, if not told otherwise) on the current GPU that nobody differentiates, casts or follows."""
    first = tensors[0]
    if not first.is_cuda or first.dtype not in dtypes or torch.is_autocast_enabled("cuda") or watched():
        return False
    grad = torch.is_grad_enabled()
    for t in tensors:
        if t is None:
            continue
        if type(t) not in (torch.Tensor, nn.Parameter) or t.dtype != first.dtype or t.device != first.device or (grad and t.requires_grad):
            return False
    return first.device.index == torch.cuda.current_device()


def _rows(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor]) -> Optional[torch.Tensor]:
    """x as [rows, k] the way trimkv_linear_rows reads it, or None where it does not take this product."""
    k = x.shape[-1] if x.dim() else 0
    return _step_rows(x, weight, bias, k) if 0 < x.numel() <= MAX_ROWS * k else None


def _step_rows(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor], k: int) -> Optional[torch.Tensor]:
    """``_rows`` of no more of them than trimkv_linear_rows takes, and of one at least."""
    if k % 64 or not _plain(x, weight, bias):
        return None
    if weight.dim() != 2 or weight.shape[1] != k or weight.shape[0] == 0 or weight.stride(1) != 1 or weight.stride(0) < k or weight.stride(0) % 8 or weight.data_ptr() % 16:
        return None
    if bias is not None and (bias.shape != weight.shape[:1] or not bias.is_contiguous()):
        return None
    x2 = x if x.dim() == 2 else x.reshape(-1, k)
    if x2.stride(1) != 1 or x2.data_ptr() % 16 or (x2.shape[0] > 1 and (x2.stride(0) < k or x2.stride(0) % 8)):
        return None
    return None if max(x2.stride(0), weight.stride(0)) > 1 << 24 else x2


@functools.lru_cache(maxsize=4096)
def _form(rows: int, n: int, k: int, silu: bool, library: Optional[str]) -> int:
    return (_lib.load() if library is None else _lib.load_hybrid(library)).trimkv_linear_tiles_form(rows, n, k, int(silu))


def _tiles(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor], silu: bool, library: Optional[str]):
    """``(x as [rows, k], form)`` the way trimkv_linear_tiles takes this product, or None where it does not or is not faster."""
    k = x.shape[-1] if x.dim() else 0
    return _prompt_rows(x, weight, bias, k, x.numel(), silu, library) if x.numel() > MAX_ROWS * k else None


def _prompt_rows(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor], k: int, size: int, silu: bool, library: Optional[str]):
    """``_tiles`` of more rows than trimkv_linear_rows takes; ``size``: the numbers of x."""
    if bias is not None or k == 0 or k % 64 or x.dtype != torch.bfloat16 or not x.is_cuda or weight.dim() != 2 or weight.shape[1] != k or weight.shape[0] == 0:
        return None
    rows, n = size // k, weight.shape[0] // 2 if silu else weight.shape[0]
    # sizes in front of what takes longer to find out; sizes that are no numbers belong to somebody who follows the operations
    if torch.compiler.is_compiling() or type(rows) is not int or type(n) is not int or max(rows, n) > 1 << 24 or (silu and weight.shape[0] % 2):
        return None
    form = _form(rows, n, k, silu, library)
    if not form or not _plain(x, weight) or weight.stride(1) != 1 or weight.stride(0) < k or weight.stride(0) % 8 or weight.data_ptr() % 16:
        return None
    if x.dim() != 2 and not x.is_contiguous():
        return None
    x2 = x if x.dim() == 2 else x.view(-1, k)
    if x2.stride(1) != 1 or x2.data_ptr() % 16 or x2.stride(0) < k or x2.stride(0) % 8 or max(x2.stride(0), weight.stride(0)) > 1 << 20:
        return None
    return x2, form


@functools.lru_cache(maxsize=4096)
def _f32_form(rows: int, n: int, k: int, library: str) -> int:
    return _lib.load_hybrid(library).trimkv_linear_f32_tiles_form(rows, n, k)


def _f32_rows(x: torch.Tensor, weight: torch.Tensor, library: str):
    """``(x as [rows, k], form)`` the way trimkv_linear_f32_tiles takes this product, or None where it does not or is not faster."""
    k = x.shape[-1] if x.dim() else 0
    if not x.is_cuda or torch.compiler.is_compiling() or k == 0 or weight.dim() != 2 or weight.shape[1] != k or weight.shape[0] == 0:
        return None
    rows, n = x.numel() // k, weight.shape[0]
    if type(rows) is not int or type(n) is not int or not 0 < rows <= 1 << 22 or n > 1 << 22:
        return None
    form = _f32_form(rows, n, k, library)
    if not form or not _plain(x, weight, dtypes=(torch.float32,)) or weight.stride(1) != 1 or weight.stride(0) < k or weight.stride(0) % 4 or weight.data_ptr() % 16:
        return None
    if x.dim() != 2 and not x.is_contiguous():
        return None
    x2 = x if x.dim() == 2 else x.view(-1, k)
    if x2.stride(1) != 1 or x2.data_ptr() % 16 or x2.stride(0) < k or x2.stride(0) % 4 or max(x2.stride(0), weight.stride(0)) > 1 << 20:
        return None
    return x2, form


def _f32_product(x: torch.Tensor, weight: torch.Tensor, library: str) -> torch.Tensor:
    many = _f32_rows(x, weight, library)
    if many is None:
        return F.linear(x, weight)
    x2, form = many
    (rows, k), n = x2.shape, weight.shape[0]
    out = torch.empty(*x.shape[:-1], n, dtype=x.dtype, device=x.device)
    rc = _lib.load_hybrid(library).trimkv_linear_f32_tiles(x2.data_ptr(), x2.stride(0), weight.data_ptr(), weight.stride(0), out.data_ptr(), n, rows, n, k, form,
                                                           _lib.current_stream(x.device))
    if rc:
        _lib.check_hybrid(rc, "trimkv_linear_f32_tiles", library)
    return out


def linear(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None, library: Optional[str] = None) -> torch.Tensor:
    """``F.linear(x, weight, bias)``.  ``library``: which one holds the kernel (a name of ``_lib.SHARED``; None: libtrimkv_hip.so)."""
    if library is not None and bias is None and x.dtype == torch.float32:
        return _f32_product(x, weight, library)
    k, size = x.shape[-1] if x.dim() else 0, x.numel()
    if size > MAX_ROWS * k:
        if size * weight.numel() < LEAST_OUTPUTS * k * k:
            return F.linear(x, weight, bias)
        many = _prompt_rows(x, weight, bias, k, size, False, library)
        return F.linear(x, weight, bias) if many is None else _tile_product(x, *many, weight, library)
    x2 = _step_rows(x, weight, bias, k) if size else None
    if x2 is None:
        return F.linear(x, weight, bias)
    if x2.shape[0] > WIDE_ROWS and weight.shape[0] > WIDE:
        return F.linear(x, weight, bias)
    rows, k = x2.shape
    n = weight.shape[0]
    out = torch.empty(*x.shape[:-1], n, dtype=x.dtype, device=x.device)
    lib = _lib.load() if library is None else _lib.load_hybrid(library)
    rc = lib.trimkv_linear_rows(x2.data_ptr(), x2.stride(0) if rows > 1 else k, weight.data_ptr(), weight.stride(0), _lib.ptr(bias), out.data_ptr(), n, rows, n, k,
                                _lib.dtype_code(x.dtype), _lib.current_stream(x.device))
    if rc:
        _lib.check(rc, "trimkv_linear_rows") if library is None else _lib.check_hybrid(rc, "trimkv_linear_rows", library)
    return out


def _tile_product(x: torch.Tensor, x2: torch.Tensor, form: int, weight: torch.Tensor, library: Optional[str], silu: bool = False, round_all: bool = True) -> torch.Tensor:
    rows, k = x2.shape
    n = weight.shape[0] // 2 if silu else weight.shape[0]
    out = torch.empty(*x.shape[:-1], n, dtype=x.dtype, device=x.device)
    lib = _lib.load() if library is None else _lib.load_hybrid(library)
    at, tail = (x2.data_ptr(), x2.stride(0), weight.data_ptr(), weight.stride(0), out.data_ptr(), n, rows, n, k), (form, _lib.BF16, _lib.current_stream(x.device))
    rc = lib.trimkv_linear_tiles_silu(*at, int(round_all), *tail) if silu else lib.trimkv_linear_tiles(*at, *tail)
    if rc:
        _lib.check(rc, "trimkv_linear_tiles") if library is None else _lib.check_hybrid(rc, "trimkv_linear_tiles", library)
    return out


def silu_product(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None, round_all: bool = True, library: Optional[str] = None) -> Optional[torch.Tensor]:
    """``silu(x @ gate.T) * (x @ up.T)`` with ``weight`` = gate over up, in one launch; None where neither trimkv_linear_rows_silu nor
    trimkv_linear_tiles_silu takes it."""
    k, size = x.shape[-1] if x.dim() else 0, x.numel()
    if size > MAX_ROWS * k:
        if size * weight.numel() < 2 * LEAST_SILU_OUTPUTS * k * k:
            return None
        many = _prompt_rows(x, weight, bias, k, size, True, library)
        return None if many is None else _tile_product(x, *many, weight, library, True, round_all)
    x2 = _step_rows(x, weight, bias, k) if size else None
    if x2 is None:
        return None
    if weight.shape[0] % 2:
        return None
    rows, k = x2.shape
    inter = weight.shape[0] // 2
    out = torch.empty(*x.shape[:-1], inter, dtype=x.dtype, device=x.device)
    lib = _lib.load() if library is None else _lib.load_hybrid(library)
    rc = lib.trimkv_linear_rows_silu(x2.data_ptr(), x2.stride(0) if rows > 1 else k, weight.data_ptr(), weight.stride(0), _lib.ptr(bias), out.data_ptr(), inter, rows, inter, k,
                                     int(round_all), _lib.dtype_code(x.dtype), _lib.current_stream(x.device))
    if rc:
        _lib.check(rc, "trimkv_linear_rows_silu") if library is None else _lib.check_hybrid(rc, "trimkv_linear_rows_silu", library)
    return out


def unhooked(module: nn.Module) -> bool:
    """Nobody has hooked the module or replaced its ``forward``: calling it does what its class says."""
    return not (module._forward_hooks or module._forward_pre_hooks or module._backward_hooks or module._backward_pre_hooks
                or _module._global_forward_hooks or _module._global_forward_pre_hooks or _module._global_backward_hooks or _module._global_backward_pre_hooks
                or "forward" in module.__dict__)


def untouched(module: nn.Module) -> bool:
    """An ``nn.Linear`` that nobody has hooked, wrapped or replaced: its parameters say all that calling it does."""
    return type(module) is nn.Linear and unhooked(module)


def leaving(forward):
    """Marks a module's ``forward`` that takes ``leave_product``; what a subclass puts in its place need not."""
    forward.leaves_product = True
    return forward


def may_leave(module: nn.Module) -> dict:
    """The keyword argument with which ``module`` may leave its last product to the caller, if it knows it and nobody looks at its output."""
    return {"leave_product": True} if getattr(type(module).forward, "leaves_product", False) and unhooked(module) else {}


NORM_ROWS, NORM_K = 32, 8192      # what trimkv_linear_rows_add and trimkv_linear_rows_norm take


class DeferredProduct:
    """``module(x)`` of an untouched ``nn.Linear``, not taken yet: whoever adds a residual to it does so in its launch (``add_product``);
    anybody else calls ``tensor``."""

    __slots__ = ("x", "module")

    def __init__(self, x: torch.Tensor, module: nn.Linear):
        self.x, self.module = x, module

    shape = property(lambda self: (*self.x.shape[:-1], self.module.weight.shape[0]))

    def tensor(self) -> torch.Tensor:
        return run(self.module, self.x)


class DeferredNorm:
    """``norm(x)`` not taken yet, with the sums of squares of ``add_product``: a product takes it in its own launch (``norm_product``);
    anybody else calls ``tensor``."""

    __slots__ = ("x", "squares", "norm", "normed")

    def __init__(self, x: torch.Tensor, squares: torch.Tensor, norm):
        self.x, self.squares, self.norm, self.normed = x, squares, norm, None

    shape = property(lambda self: self.x.shape)

    def tensor(self) -> torch.Tensor:
        if self.normed is None:
            self.normed = self.norm(self.x)
        return self.normed


def tensor_of(x) -> torch.Tensor:
    return x.tensor() if type(x) in (DeferredNorm, DeferredProduct) else x


def can_defer_product(module: nn.Module, x: torch.Tensor) -> bool:
    """Whether ``module(x)`` may wait for the residual that is added to it."""
    if not untouched(module):
        return False
    w = module.weight
    return (x.dtype == torch.bfloat16 and 0 < x.numel() <= NORM_ROWS * x.shape[-1] and w.shape[0] % 64 == 0 and w.shape[0] <= NORM_K
            and _rows(x, w, module.bias) is not None)


def can_defer_norm(weight: torch.Tensor, residual: torch.Tensor) -> bool:
    """Whether the product behind the norm of a sum with ``residual`` may take it along."""
    k = residual.shape[-1]
    return weight.shape == (k,) and weight.is_contiguous() and residual.is_contiguous() and not (weight.data_ptr() | residual.data_ptr()) % 16 and _plain(residual, weight)


def add_product(p: DeferredProduct, residual: torch.Tensor):
    """``(residual + module(x), squares)`` in one launch; both have passed ``can_defer_product`` and ``can_defer_norm`` and are of one shape."""
    w, bias = p.module.weight, p.module.bias
    x2, n = _rows(p.x, w, bias), w.shape[0]
    rows, k = x2.shape
    out = torch.empty(residual.shape, dtype=residual.dtype, device=residual.device)
    squares = torch.empty(rows, n // 8, dtype=torch.float32, device=residual.device)
    _lib.check(_lib.load().trimkv_linear_rows_add(x2.data_ptr(), x2.stride(0) if rows > 1 else k, w.data_ptr(), w.stride(0), _lib.ptr(bias), residual.data_ptr(), n,
                                                  out.data_ptr(), n, squares.data_ptr(), rows, n, k, _lib.BF16, _lib.current_stream(residual.device)), "trimkv_linear_rows_add")
    return out, squares


def norm_product(d: DeferredNorm, weight: torch.Tensor, bias: Optional[torch.Tensor], silu: bool = False) -> Optional[torch.Tensor]:
    """``linear(d, weight, bias)`` or, ``silu``, ``silu_product`` of it with the norm in the same launch; None where that is not to be done
    (the norm has been taken already, or the kernel does not take this product)."""
    x2 = _rows(d.x, weight, bias) if d.normed is None else None
    if x2 is None or (silu and weight.shape[0] % 2):
        return None
    rows, k = x2.shape
    n = weight.shape[0] // 2 if silu else weight.shape[0]
    out = torch.empty(*d.x.shape[:-1], n, dtype=d.x.dtype, device=d.x.device)
    _lib.check(_lib.load().trimkv_linear_rows_norm(x2.data_ptr(), x2.stride(0) if rows > 1 else k, d.squares.data_ptr(), d.norm.weight.data_ptr(), float(d.norm.variance_epsilon),
                                                   weight.data_ptr(), weight.stride(0), _lib.ptr(bias), out.data_ptr(), n, rows, n, k, int(silu), 1, _lib.BF16,
                                                   _lib.current_stream(d.x.device)), "trimkv_linear_rows_norm")
    return out


def run(module: nn.Module, x: torch.Tensor) -> torch.Tensor:
    """``module(x)``; an untouched ``nn.Linear`` goes to ``linear`` with its parameters."""
    return linear(x, module.weight, module.bias) if untouched(module) else module(x)
