"""y = x . W^T for a weight stored [out, in], the one projection every part uses.

Which kernel runs depends only on the types of the operands:

* float32 x, float32 W  -> the fixed-order float32 kernel (the true 32-bit path);
* bfloat16 x, bfloat16 W -> the kernel that ops.choose_product names for the sizes: hand-written
  MFMA kernels for few rows (decode) and, where they were measured ahead, for many, else the
  vendor library (hipBLASLt through torch), as the reference uses cuBLAS for its projections
  (infer/src/ops/linear.rs:921-959);
* bfloat16 x, float32 W (a tensor that the checkpoint stores in 32 bits stays so):
  x is widened and the float32 kernel runs.

The few-rows kernel may split K over workgroups and leave a stack of float32 partial products
[S, T, out] behind.  A caller whose consumer can add such a stack in order (the residual add fused
into RMSNorm, the q/k/v preparation) says `partials_ok=True` and passes it on; otherwise the stack
is added here.

With `tiles=True` a bfloat16 weight is held a second time as operand tiles (ops.pack_weight_tiles): the
few-rows kernels then read one contiguous kilobyte a wave and k step instead of sixteen pieces a row apart,
which is worth a fifth of their time on MI355X.  The library needs the rows, so both copies stay.

A projection whose result goes into the residual can be left to the norm behind it (`late`): for up to eight rows product, add
and norm are then one kernel (ops.gemm_strips), for which `lay_strips` holds the weight in that kernel's layout too where the
tiles are not that layout already.
"""
from __future__ import annotations

import torch

from ..kernels import ops


class LateProduct:
    """A projection that has not run: `norm` runs it with the residual's add and most of the norm behind it, `now` by itself."""

    def __init__(self, linear: "Linear", x: torch.Tensor):
        self.linear, self.x = linear, x

    def now(self) -> torch.Tensor:
        return self.linear(self.x, partials_ok=True)

    def norm(self, residual: torch.Tensor, weight: torch.Tensor, eps: float) -> ops.ScaledRows:
        return ops.gemm_strips(self.x, self.linear.strips, residual, weight, eps)


class Linear:
    def __init__(self, weight: torch.Tensor, tiles: bool = False, packed: torch.Tensor | None = None, strips: bool = False):
        """packed: operand tiles that exist already (of a matrix that this weight is rows of, from the first row of a tile on)."""
        if weight.dim() != 2 or not weight.is_contiguous():
            raise ValueError("a projection weight must be a contiguous [out, in] matrix")
        self.weight = weight
        self.out_features, self.in_features = weight.shape
        self.tiles = packed
        if packed is None and tiles and weight.dtype == torch.bfloat16 and weight.is_cuda and self.in_features % 8 == 0:
            self.tiles = ops.pack_weight_tiles(weight)
        self.strips = None
        if strips:
            self.lay_strips()

    def lay_strips(self) -> None:
        """From here on `late` may leave the projection to the norm behind it."""
        if (self.strips is None and self.weight.dtype == torch.bfloat16 and self.weight.is_cuda
                and ops.strips_preferred(self.out_features, self.in_features)):
            same = self.tiles is not None and ops.strip_columns(self.out_features, self.in_features) == 16
            self.strips = self.tiles if same else ops.pack_weight_strips(self.weight)

    def takes_scaled(self, rows: int) -> bool:
        """Whether this projection of `rows` rows can read ops.ScaledRows."""
        return self.weight.dtype == torch.bfloat16 and ops.takes_scaled(rows, self.out_features, self.in_features, tiled=self.tiles is not None,
                                                                       fused=False)

    def late(self, x: torch.Tensor):
        """The projection for the norm behind it to run where it can, else as with `partials_ok`."""
        if (self.strips is not None and 1 <= x.shape[0] <= ops.STRIP_ROWS and x.dtype == torch.bfloat16 and x.stride(1) == 1
                and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0):
            return LateProduct(self, x)
        return self(x, partials_ok=True)

    def __call__(self, x: torch.Tensor, out_dtype: torch.dtype | None = None, partials_ok: bool = False) -> torch.Tensor:
        """x [T, in] -> [T, out] in `out_dtype` (default: the type of x); with `partials_ok` possibly a
        float32 stack [S, T, out] whose sum over S, in order, is the product."""
        out_dtype = out_dtype or x.dtype
        w = self.weight
        if type(x) is ops.ScaledRows:
            return ops.gemm_bf16(x.rows, w, out_dtype, partials_ok=partials_ok, tiles=self.tiles, scaled=x)
        if x.shape[0] == 0:
            return torch.empty((0, self.out_features), dtype=out_dtype, device=x.device)
        if w.dtype == torch.float32:
            y = ops.gemm_f32(x if x.dtype == torch.float32 else x.float(), w)
            return y if out_dtype == torch.float32 else y.to(out_dtype)
        if x.dtype != torch.bfloat16:
            raise ops.ShapeError(f"a bfloat16 weight needs bfloat16 activations, got {x.dtype}")
        return ops.gemm_bf16(x, w, out_dtype, partials_ok=partials_ok, tiles=self.tiles)
