"""FP8 linear layers and the FP8 weight cache, on the HIP library (gfx950).

Mirrors flower/precision.py (the torchao-based FP8 conversion) with this build's own FP8 linear:

``_FP8_DIM_ALIGNMENT``, ``_block_index``, ``fp8_module_filter``  -- precision.py:56-98, the same
    guardrails (aligned dims, only Linears under ``blocks.<i>``, first/last ``keep`` blocks bf16).
``Fp8Linear``          -- replaces torchao ``Float8Linear``: forward is the HIP FP8 GEMM
    (e4m3 weight x e4m3 per-row activation, fp32 accumulate, bf16 out, the ``_fp8_head``
    recipe of base.py:911-923). recipe "rowwise": per-output-channel weight scales, per-row
    activation scales; "tensorwise": one weight scale and one activation scale; "weight_only":
    per-output-channel e4m3 weights times the bf16 activations as they are (W8A16: the weight is
    widened to bf16 in the kernel, bf16 MFMA; needs K % 64 == 0).
    Backward ("rowwise" / "tensorwise", as torchao's Float8Linear does under
    ``training.fp8_linear``): both gradient GEMMs in FP8 on the same kernel —
    dgrad  grad_x = g W:    per-row e4m3 g (per tensor for "tensorwise") x the weight's per-column
                            e4m3 codes stored transposed (cached with the forward codes);
    wgrad  grad_W = g^T x:  per-column e4m3 of g and of x (the token axis becomes the contiguous
                            reduction), written transposed by flw_quant_cols_e4m3.
    "weight_only" (and ``backward_fp8 = False``) keeps the bf16 matmul pair.
``convert_model_to_fp8`` / ``maybe_convert_fp8`` -- precision.py:134-195, 356-381; the default
    recipe is the reference's, "tensorwise".
``fp8_weight_cache``   -- precision.py:198-353: quantise every FP8 weight ONCE on entry, patch
    the layers' forwards to reuse it across grad-accumulation microsteps, restore the forwards
    on exit (also on an exception), and raise RuntimeError("...stale...") when a sampled
    fingerprint of any cached weight changed while the cache was live.
``fp8_head`` / ``compute_logits`` -- the FP8 LM head of base.py:865-924 on the same quantiser and
    GEMM (eval only, as the reference routes it).
"""

from __future__ import annotations

import torch
import torch.nn as nn

from . import _lib

_FP8_DIM_ALIGNMENT = 16
RECIPES = ("rowwise", "tensorwise", "weight_only")
# The reference's default recipe: convert_model_to_fp8(..., recipe="tensorwise") (precision.py:137)
# and training.fp8_recipe "tensorwise" (config.py:593).
DEFAULT_RECIPE = "tensorwise"


def _block_index(fqn: str) -> int | None:
    """The integer i of the first ``blocks.<i>`` pair in a module's dotted name, else None (the LM
    head, MTP heads and anything hung off the model root)."""
    parts = fqn.split(".")
    return next((int(nxt) for cur, nxt in zip(parts, parts[1:]) if cur == "blocks" and nxt.isdigit()), None)


def fp8_module_filter(num_layers: int, keep_bf16_blocks: int):
    """``(module, fqn) -> bool`` deciding which Linears become FP8 (the precision.py:73-98 rules):
    an ``nn.Linear`` whose in and out sizes are both multiples of 16 (the FP8 GEMM's alignment),
    inside some ``blocks.<i>``, and, when ``keep_bf16_blocks`` k > 0, with k <= i < num_layers - k
    (the first and last k blocks stay bf16)."""
    k = max(int(keep_bf16_blocks), 0)
    kept = range(k, num_layers - k) if k else None

    def eligible(module: nn.Module, fqn: str) -> bool:
        if not isinstance(module, nn.Linear):
            return False
        if (module.in_features | module.out_features) % _FP8_DIM_ALIGNMENT:
            return False
        i = _block_index(fqn)
        return i is not None and (kept is None or i in kept)

    return eligible


# ---------------------------------------------------------------- weight / activation quantisers

_CUS: dict = {}


def _compute_units(device) -> int:
    idx = torch.device(device).index or 0
    if idx not in _CUS:
        _CUS[idx] = torch.cuda.get_device_properties(idx).multi_processor_count
    return _CUS[idx]


def _quantize_tensorwise(x2: torch.Tensor):
    """(x8 [R, C], scale [1]): one e4m3 scale for the whole matrix x2 [R, C] (bf16 / fp32, rows of
    stride C' >= C). The amax, the scale and every code are those of the matrix itself whatever grid
    the native body lays over it."""
    return _lib.native().quant_tensorwise(x2, _compute_units(x2.device), _lib.stream_of(x2))


def quantize_weight(weight: torch.Tensor, recipe: str = "rowwise"):
    """(w8 [N, K] uint8 e4m3 codes, w_scale float32 [N] or [1]) on the weight's device."""
    _lib.load()
    _lib.require_gpu(weight)
    w = weight.detach()
    if w.dtype not in (torch.float32, torch.bfloat16):
        w = w.to(torch.bfloat16)
    w = w.contiguous()
    if recipe in ("rowwise", "weight_only"):
        return _lib.native().quant_rows(w, "quantize_weight", _lib.stream_of(w))
    if recipe == "tensorwise":
        return _quantize_tensorwise(w)
    raise RuntimeError(f"training.fp8_recipe must be one of {sorted(RECIPES)}, got {recipe!r}")


def quantize_cols(x2: torch.Tensor, granularity: str, ld: int | None = None):
    """(codes_t [C, ld] uint8, scale float32 [C] or [1]): e4m3 of each column of x2 [R, C] (bf16 or
    fp32, rows contiguous), transposed; rows past R up to ld (a multiple of 16) are coded 0."""
    _lib.load()
    _lib.require_gpu(x2)
    if x2.dtype not in (torch.float32, torch.bfloat16):
        x2 = x2.to(torch.bfloat16)
    x2 = _lib.native().rows16(x2)
    R = x2.shape[0]
    ld = ((R + 15) // 16) * 16 if ld is None else ld
    return _lib.native().quant_cols(x2, granularity == "column", ld, _lib.stream_of(x2))


def quantize_weight_cols(weight: torch.Tensor, recipe: str = "rowwise"):
    """The weight's codes for dgrad: (w8c [K, N] = per-column e4m3 of W [N, K], transposed;
    scales [K] ("rowwise") or [1] ("tensorwise"))."""
    w = weight.detach()
    return quantize_cols(w, "column" if recipe == "rowwise" else "tensor", ld=w.shape[0])


def _quantize_rows(x2: torch.Tensor, recipe: str):
    """(x8 [M, K], scale [M] or [1]) of a contiguous bf16 / fp32 matrix, per row ("rowwise") or
    per tensor ("tensorwise")."""
    if recipe == "rowwise":
        return _lib.native().quant_rows(x2, "quantize rows", _lib.stream_of(x2))
    return _quantize_tensorwise(x2)


def scaled_mm(a8: torch.Tensor, sa: torch.Tensor, b8: torch.Tensor, sb: torch.Tensor) -> torch.Tensor:
    """bf16 [M, N] = (a8 [M, K] . b8 [N, K]^T) * sa[m] * sb[n] through flw_fp8_scaled_mm_ws (split
    over K into a workspace for a long K and an output of a third of the GPU's 256 x 256 tiles)."""
    return _lib.native().scaled_mm(a8, sa, b8, sb, None, True, _lib.stream_of(a8))


def _quantize_tensorwise_t(x2: torch.Tensor, ld: int, amax: torch.Tensor | None = None):
    """(x8 [R, C], x8t [C, ld], scale [1]): the tensorwise codes of a bf16 matrix x2 [R, C] (unit
    column stride, C % 16 == 0) in rows and transposed (columns past R zero) from one pass
    (flw_quant_tensor_t_e4m3): the codes of _quantize_tensorwise, and transpose_codes of them.
    amax: x2's |x| maximum as a device fp32 bit pattern from its producer (int32 [1]): then the
    quantise pass alone (flw_quant_tensor_t_e4m3_amax)."""
    return _lib.native().quant_tensor_t(x2, ld, amax, _lib.stream_of(x2))


def scaled_mm_plain(a8: torch.Tensor, sa: torch.Tensor, b8: torch.Tensor, sb: torch.Tensor) -> torch.Tensor:
    """bf16 [M, N] = (a8 [M, K] . b8 [N, K]^T) * sa * sb through flw_fp8_scaled_mm (never split over
    K): the forward GEMM of fp8_linear_forward's tensorwise route."""
    return _lib.native().scaled_mm(a8, sa, b8, sb, None, False, _lib.stream_of(a8))


def scaled_mm_residual(a8: torch.Tensor, sa: torch.Tensor, b8: torch.Tensor, sb: torch.Tensor,
                       res: torch.Tensor) -> torch.Tensor:
    """bf16 [M, N] = res + bf16((a8 . b8^T) * sa * sb), both terms rounded to bf16 as torch adds a
    Linear's output to a tensor (flw_fp8_scaled_mm_residual; never split over K). res: [M, N] bf16
    rows with a unit column stride."""
    return _lib.native().scaled_mm(a8, sa, b8, sb, res, False, _lib.stream_of(a8))


def transpose_codes(c8: torch.Tensor, ld: int | None = None) -> torch.Tensor:
    """[C, ld] uint8: the e4m3 codes c8 [R, C] transposed (ld >= R, a multiple of 16; columns past R
    zero). Under one scale per tensor a matrix's column codes are its row codes, so this gives
    quantize_cols(x, "tensor")'s codes from the row codes without reading x again."""
    ld = ((c8.shape[0] + 15) // 16) * 16 if ld is None else ld
    return _lib.native().transpose_codes(c8, ld, _lib.stream_of(c8))


def fp8_linear_backward(g2: torch.Tensor, x2: torch.Tensor, w_cols, recipe: str,
                        need_x: bool = True, need_w: bool = True, x_codes=None, g_amax=None):
    """FP8 gradient GEMMs of y = x W^T: (grad_x [M, K], grad_W [N, K]), bf16.

    g2: [M, N] output gradient, x2: [M, K] the forward input, w_cols: (w8c [K, N], scale) from
    ``quantize_weight_cols`` (or a callable returning it). Row / column granularity per recipe:
    "rowwise" -> g per row for dgrad, g and x per column for wgrad; "tensorwise" -> one scale per
    tensor everywhere. The token axis is zero-padded to a multiple of 128 for wgrad.
    x_codes: (x8t [K, ld], scale [1]), the forward's tensorwise codes of x2 transposed (ld = M
    rounded up to 128, zero past M); with it x2 is not read (it may be None), and g is quantised
    once into both layouts (rows for dgrad, columns for wgrad): the same codes and scales as
    quantize_cols(.., "tensor"), since one scale per tensor makes a matrix's column codes its row
    codes. g_amax: g2's |g| maximum from its producer (see _quantize_tensorwise_t), tensorwise
    with x_codes only."""
    gx = gw = None
    g2 = g2.to(torch.bfloat16).contiguous()
    if recipe == "tensorwise" and x_codes is not None and need_w and g2.shape[1] % 16 == 0:
        M = g2.shape[0]
        g8, g8t, sg = _quantize_tensorwise_t(g2, ((M + 127) // 128) * 128, g_amax)
        if need_x:
            w8c, swc = w_cols() if callable(w_cols) else w_cols
            gx = scaled_mm(g8, sg, w8c, swc)
        x8t, sx = x_codes
        return gx, scaled_mm(g8t, sg, x8t, sx)
    g8 = sg = None
    if need_x:
        g8, sg = _quantize_rows(g2, recipe)
        w8c, swc = w_cols() if callable(w_cols) else w_cols
        gx = scaled_mm(g8, sg, w8c, swc)
    if need_w:
        M = g2.shape[0]
        ld = ((M + 127) // 128) * 128
        if recipe == "tensorwise" and x_codes is not None:
            if g8 is None:
                g8, sg = _quantize_rows(g2, recipe)
            x8t, sx = x_codes
            gw = scaled_mm(transpose_codes(g8, ld), sg, x8t, sx)
        else:
            gran = "column" if recipe == "rowwise" else "tensor"
            g8c, sgc = quantize_cols(g2, gran, ld)
            x8c, sxc = quantize_cols(x2, gran, ld)
            gw = scaled_mm(g8c, sgc, x8c, sxc)
    return gx, gw


def fp8_linear_forward(x: torch.Tensor, w8: torch.Tensor, w_scale: torch.Tensor,
                       recipe: str = "rowwise", return_codes: bool = False, x_amax=None, residual=None):
    """bf16 y[..., N] = x[..., K] @ dequant(w8)^T through the HIP FP8 GEMM. With return_codes
    (tensorwise only): (y, x8t [K, ld], x_scale [1]), x's codes transposed (ld = M rounded up to
    128, zero past M) for the backward's wgrad, written by the same pass as the forward's; x_amax
    (with return_codes): x's |x| maximum from its producer, which spares that pass its amax pass.
    residual (bf16, x's leading shape by N): returns residual + y as torch's add of the two bf16
    tensors gives it, in the tensorwise GEMM's epilogue (after the GEMM otherwise)."""
    native = _lib.native()
    _lib.require_gpu(x, w8)
    N, K = w8.shape
    lead = x.shape[:-1]
    x2 = x.reshape(-1, K)
    if x2.dtype != torch.bfloat16:
        x2 = x2.to(torch.bfloat16)
    x2 = native.rows16(x2)
    M = x2.shape[0]
    if M == 0:
        y = torch.empty((*lead, N), dtype=torch.bfloat16, device=x.device)
        return (y, None, None) if return_codes else y
    stream = _lib.stream_of(x2)
    if recipe != "tensorwise":
        y = native.linear(x2, w8, w_scale, recipe == "weight_only", stream).view(*lead, N)
        return y if residual is None else residual + y
    ld = ((M + 127) // 128) * 128
    x8t = None
    if return_codes and K % 16 == 0:
        x8, x8t, sx = _quantize_tensorwise_t(x2, ld, x_amax)
    else:
        x8, sx = _quantize_tensorwise(x2)
    r2 = native.rows16(residual.reshape(M, N).to(torch.bfloat16)) if residual is not None else None
    y = native.scaled_mm(x8, sx, w8, w_scale, r2, False, stream).view(*lead, N)
    if return_codes:
        return y, (transpose_codes(x8, ld) if x8t is None else x8t), sx
    return y


class _Fp8LinearFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, bias, w8, w_scale, recipe, mod, x_amax=None, residual=None, w8t=None):
        ctx.has_bias = bias is not None
        ctx.recipe, ctx.mod = recipe, mod
        ctx.x_shape, ctx.x_dtype = x.shape, x.dtype
        N, K = weight.shape
        # Tensorwise with the FP8 backward: keep the forward's e4m3 codes of x (transposed, for
        # wgrad, written by the forward's quantise pass) and of W (1 byte a value) instead of x;
        # the backward transposes W's for dgrad rather than quantising W again along columns.
        ctx.keep_codes = (recipe == "tensorwise" and getattr(mod, "backward_fp8", True)
                          and N % 16 == 0 and K % 16 == 0 and x.numel() > 0)
        ctx.has_residual = residual is not None
        fused_res = residual if bias is None else None      # residual + (y + bias) otherwise
        if ctx.keep_codes:
            y, x8t, sx = fp8_linear_forward(x, w8, w_scale, recipe, return_codes=True, x_amax=x_amax,
                                            residual=fused_res)
            ctx.save_for_backward(x8t, sx, w8, w_scale, weight, w8t)
        else:
            ctx.save_for_backward(x, weight)
            y = fp8_linear_forward(x, w8, w_scale, recipe, residual=fused_res)
        if bias is not None:
            y = y + bias.to(y.dtype)
            if residual is not None:
                y = residual + y
        return y

    @staticmethod
    def backward(ctx, g):
        g2 = g.reshape(-1, g.shape[-1])
        need_x, need_w = ctx.needs_input_grad[0], ctx.needs_input_grad[1]
        if ctx.keep_codes:
            x8t, sx, w8, sw, weight, w8t = ctx.saved_tensors
            N = weight.shape[0]
            mod = ctx.mod

            def w_cols():            # the weight cache's column codes while one is active
                if getattr(mod, "_fp8_cached", None) is not None:
                    return mod.weight_col_codes()
                return (w8t if w8t is not None else transpose_codes(w8, N)), sw
            gx, gw = fp8_linear_backward(g2, None, w_cols, "tensorwise", need_x, need_w, x_codes=(x8t, sx))
            gx = gx.reshape(ctx.x_shape).to(ctx.x_dtype) if gx is not None else None
            gw = gw.to(weight.dtype) if gw is not None else None
            gb = g2.sum(0) if ctx.has_bias and ctx.needs_input_grad[2] else None
            return gx, gw, gb, None, None, None, None, None, (g if ctx.has_residual else None), None
        x, weight = ctx.saved_tensors
        N, K = weight.shape
        # FP8 gradient GEMMs need 16-aligned dims (the conversion filter guarantees them; a
        # hand-built Fp8Linear may not): otherwise the bf16 pair below.
        fp8 = (ctx.recipe in ("rowwise", "tensorwise") and getattr(ctx.mod, "backward_fp8", True)
               and N % 16 == 0 and K % 16 == 0)
        gx = gw = None
        if fp8 and (need_x or need_w):
            x2 = x.reshape(-1, x.shape[-1])
            gx, gw = fp8_linear_backward(g2, x2, ctx.mod.weight_col_codes, ctx.recipe, need_x, need_w)
            gx = gx.reshape(x.shape).to(x.dtype) if gx is not None else None
            gw = gw.to(weight.dtype) if gw is not None else None
        else:
            w = weight.to(g2.dtype)
            gx = (g2 @ w).reshape(x.shape).to(x.dtype) if need_x else None
            if need_w:
                gw = (g2.t() @ x.reshape(-1, x.shape[-1]).to(g2.dtype)).to(weight.dtype)
        gb = g2.sum(0) if ctx.has_bias and ctx.needs_input_grad[2] else None
        return gx, gw, gb, None, None, None, None, None, (g if ctx.has_residual else None), None


class Fp8Linear(nn.Linear):
    """``nn.Linear`` whose forward runs the HIP FP8 GEMM (weights quantised on every call unless
    an ``fp8_weight_cache`` is active). Shares the Parameters of the Linear it was built from."""

    def __init__(self, in_features: int, out_features: int, bias: bool = True, device=None,
                 dtype=None, *, recipe: str = DEFAULT_RECIPE) -> None:
        _check_recipe(recipe)
        super().__init__(in_features, out_features, bias=bias, device=device, dtype=dtype)
        self.recipe = recipe
        self.backward_fp8 = True

    @classmethod
    def from_linear(cls, lin: nn.Linear, recipe: str = DEFAULT_RECIPE) -> "Fp8Linear":
        _check_recipe(recipe)
        new = cls.__new__(cls)
        nn.Module.__init__(new)
        new.in_features, new.out_features = lin.in_features, lin.out_features
        # same Parameter objects: an optimizer built before or after conversion sees them
        new.register_parameter("weight", lin.weight)
        new.register_parameter("bias", lin.bias)
        new.recipe = recipe
        new.backward_fp8 = True
        new.train(lin.training)
        return new

    def quantize_weight(self):
        return quantize_weight(self.weight, self.recipe)

    def weight_codes(self):
        """(w8, w_scale): the fp8_weight_cache's copy while one is active, else quantised now."""
        cached = getattr(self, "_fp8_cached", None)
        return cached if cached is not None else self.quantize_weight()

    def tensorwise_codes(self):
        """(w8 [N, K], scale [1], w8t [K, N] or None) for the tensorwise recipe's training step: the
        fp8_weight_cache's codes while one is active (w8t None: its column codes serve dgrad),
        else the weight's codes in rows and transposed from one pass (flw_quant_tensor_t_e4m3),
        the transpose being the dgrad operand the backward would otherwise make from w8."""
        cached = getattr(self, "_fp8_cached", None)
        if cached is not None:
            return cached[0], cached[1], None
        w = self.weight.detach()
        N, K = w.shape
        if w.dtype != torch.bfloat16 or N % 16 or K % 16 or not w.is_cuda:
            w8, sw = self.quantize_weight()
            return w8, sw, None
        w8, w8t, sw = _quantize_tensorwise_t(w.contiguous(), N)
        return w8, sw, w8t

    def weight_col_codes(self):
        """(w8c [K, N], scale) for the dgrad GEMM: quantised once per fp8_weight_cache context
        (on the first backward inside it), else on every call."""
        cached = getattr(self, "_fp8_cached_cols", None)
        if cached is not None:
            return cached
        codes = quantize_weight_cols(self.weight, self.recipe)
        if getattr(self, "_fp8_cached", None) is not None:       # a cache context is active
            self._fp8_cached_cols = codes
        return codes

    def forward_with(self, x: torch.Tensor, w8: torch.Tensor, w_scale: torch.Tensor, x_amax=None,
                     residual=None, w8t=None) -> torch.Tensor:
        """x_amax: x's |x| maximum (int32 [1] fp32 bit pattern) from the kernel that produced x, used
        by the tensorwise recipe's cast of x in place of its own amax pass. residual: returns
        ``residual + self(x)`` (the block's ``x + ff(...)``), the add in the GEMM's epilogue where
        the recipe allows, rounded as torch's add of the two bf16 tensors. w8t: w8 transposed [K, N]
        (the tensorwise dgrad operand), when the caller made it with w8."""
        if torch.is_autocast_enabled():
            x = x.to(torch.get_autocast_gpu_dtype())
            x_amax = None
        return _Fp8LinearFn.apply(x, self.weight, self.bias, w8, w_scale, self.recipe, self, x_amax, residual, w8t)

    def forward(self, x: torch.Tensor, x_amax=None, residual=None) -> torch.Tensor:
        if self.recipe == "tensorwise" and self.backward_fp8 and torch.is_grad_enabled() and x.is_cuda:
            w8, w_scale, w8t = self.tensorwise_codes()
            return self.forward_with(x, w8, w_scale, x_amax, residual, w8t)
        w8, w_scale = self.quantize_weight()
        return self.forward_with(x, w8, w_scale, x_amax, residual)

    def extra_repr(self) -> str:
        return super().extra_repr() + f", recipe={self.recipe}"


def _check_recipe(recipe: str) -> None:
    if recipe not in RECIPES:
        raise RuntimeError(f"training.fp8_recipe must be one of {sorted(RECIPES)}, got {recipe!r}")


def convert_model_to_fp8(model: nn.Module, *, recipe: str = DEFAULT_RECIPE, keep_bf16_blocks: int = 1,
                         use_fast_accum: bool = False, verbose: bool = True):
    """Replace every Linear that ``fp8_module_filter`` admits by an ``Fp8Linear`` sharing its
    Parameters, in place (precision.py:134-195); returns (model, info) with the info keys the
    reference logs. The block-range guardrail needs ``model.blocks``: a model without it is refused
    rather than converted wholesale. ``use_fast_accum`` is recorded only (the MFMA accumulates in
    fp32 in every GEMM here)."""
    _check_recipe(recipe)
    num_layers = len(getattr(model, "blocks", []))
    if num_layers == 0:
        raise RuntimeError(
            "convert_model_to_fp8 found no `blocks` on the model; the block-range "
            "guardrail cannot be applied. Refusing to convert blindly.")
    admit = fp8_module_filter(num_layers, keep_bf16_blocks)
    named = list(model.named_modules())
    targets = [(fqn, m) for fqn, m in named if admit(m, fqn)]
    for fqn, mod in targets:
        owner, _, attr = fqn.rpartition(".")
        setattr(model.get_submodule(owner) if owner else model, attr, Fp8Linear.from_linear(mod, recipe))
    info = {"fp8_recipe": recipe, "fp8_keep_bf16_blocks": keep_bf16_blocks, "fp8_use_fast_accum": use_fast_accum,
            "fp8_converted_linears": len(targets),
            "fp8_total_linears": sum(isinstance(m, nn.Linear) for _, m in named)}
    if verbose:
        print(f"[fp8] recipe={recipe} converted {len(targets)}/{info['fp8_total_linears']} Linear layers "
              f"(blocks {keep_bf16_blocks}..{num_layers - keep_bf16_blocks - 1} of {num_layers}; "
              f"first/last {keep_bf16_blocks} and the tied LM head stay bf16)", flush=True)
    return model, info


def maybe_convert_fp8(model: nn.Module, training_cfg, device):
    """The training entry point (precision.py:356-381): a no-op returning (model, {}) unless
    ``training.fp8_linear`` is set; then a GPU and ``training.precision == "bf16"`` are required and
    the conversion runs with the config's recipe (``training.fp8_recipe``, "tensorwise" when the
    config object does not carry one, as config.py:593 defaults it)."""
    if not getattr(training_cfg, "fp8_linear", False):
        return model, {}
    if device.type != "cuda":
        raise RuntimeError("training.fp8_linear requires a GPU (ROCm)")
    if training_cfg.precision != "bf16":
        raise RuntimeError(
            "training.fp8_linear requires training.precision: bf16 "
            f"(FP8 layers consume bf16 activations), got {training_cfg.precision!r}")
    return convert_model_to_fp8(model, recipe=getattr(training_cfg, "fp8_recipe", DEFAULT_RECIPE),
                                keep_bf16_blocks=int(training_cfg.fp8_keep_bf16_blocks),
                                use_fast_accum=bool(getattr(training_cfg, "fp8_use_fast_accum", False)))


class _CachedLayer:
    """One layer held by an fp8_weight_cache: the module, the forward it had before, and the
    weight's sampled checksum at entry (None when not verifying)."""

    __slots__ = ("module", "forward", "checksum")

    def __init__(self, module, forward, checksum):
        self.module, self.forward, self.checksum = module, forward, checksum


class fp8_weight_cache:
    """Quantise every Fp8Linear weight of ``model`` once for the duration of a ``with`` block
    (precision.py:198-353), instead of on every forward of every accumulation microstep.

        with fp8_weight_cache(model):
            for _ in range(accum):
                model(batch).backward()
        optimizer.step()                 # outside: the weights may change only after the block

    Inside the block each layer's forward uses the codes and scales made at entry (and its dgrad
    reuses the transposed codes made at its first backward). A weight changed in place inside the
    block would leave those codes describing an old weight; an in-place ``p.data -= ...`` does not
    bump the tensor's version counter, so nothing can detect it on the fly. Instead, on leaving,
    every layer's forward is put back (always, also when an exception is propagating) and, with
    ``verify`` on and no exception in flight, a checksum of every 4096th weight element taken at
    entry is compared with a fresh one; any mismatch raises RuntimeError naming the cached codes
    stale. Exceptions from the block propagate (``__exit__`` returns False)."""

    _FINGERPRINT_STRIDE = 4096

    def __init__(self, model: nn.Module, *, verify: bool = True) -> None:
        self.model = model
        self.verify = verify
        self.entries: list[_CachedLayer] = []

    @classmethod
    def _fingerprint(cls, w) -> float:
        return float(w.detach().reshape(-1)[:: cls._FINGERPRINT_STRIDE].float().sum())

    def __enter__(self):
        for mod in self.model.modules():
            if isinstance(mod, Fp8Linear):
                codes = mod.quantize_weight()
                mod._fp8_cached = codes
                entry = _CachedLayer(mod, mod.forward, self._fingerprint(mod.weight) if self.verify else None)
                mod.forward = (lambda x, x_amax=None, residual=None, _m=mod, _c=codes:
                               _m.forward_with(x, *_c, x_amax=x_amax, residual=residual))
                self.entries.append(entry)
        return self

    def __exit__(self, exc_type, exc, tb):
        moved = 0
        for e in self.entries:
            e.module.forward = e.forward
            e.module._fp8_cached = e.module._fp8_cached_cols = None
            if e.checksum is not None and exc_type is None and self._fingerprint(e.module.weight) != e.checksum:
                moved += 1
        self.entries = []
        if moved:
            raise RuntimeError(
                f"fp8_weight_cache: {moved} weight(s) changed inside the cache's block, so the FP8 codes "
                "quantised at entry are stale for them. Leave the block before the optimizer step; "
                "the cache refuses to let a forward run on out-of-date weights unnoticed.")
        return False


# ---------------------------------------------------------------- FP8 LM head

def fp8_head(x_normed: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """bf16 logits [B, T, vocab] = x_normed [B, T, D] @ weight [vocab, D]^T in FP8: the recipe of
    ``CausalLM._fp8_head`` (base.py:887-924) -- per-row activation scales and per-vocab-row weight
    scales, each max(amax / 448, 1e-12) in fp32, both operands divided by their scale and cast
    without a clamp, fp32 accumulation, bf16 out. The weight is quantised on every call, as the
    reference does (it is the tied embedding, which training keeps changing)."""
    B, T, D = x_normed.shape
    w8, w_scale = quantize_weight(weight, "rowwise")
    return fp8_linear_forward(x_normed.reshape(-1, D), w8, w_scale, "rowwise").view(B, T, -1)


def compute_logits(head: nn.Linear, x_normed: torch.Tensor, fp8_lm_head: bool, training: bool) -> torch.Tensor:
    """The reference's head routing (``_compute_logits``, base.py:865-886): the FP8 head only in
    eval, for bf16 activations on the GPU; otherwise the plain ``head`` Linear."""
    if fp8_lm_head and not training and x_normed.dtype == torch.bfloat16 and x_normed.is_cuda:
        return fp8_head(x_normed, head.weight)
    return head(x_normed)
