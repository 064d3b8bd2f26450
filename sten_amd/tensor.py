"""``GroupedNMTensor`` -- the grouped n:m container, API-compatible with the reference class
(src/sten/grouped_nm/grouped_nm_tensor.py:877-958: ``val``, ``idx``, ``nm_strides``,
``from_dense``, ``to_dense``, ``set_spmm_opt``) and extended with what a wrapped format needs on
a GPU: ``dtype`` / ``device`` / ``shape`` / ``to``, same-pattern re-compression
(the disabled ``clone_layout``, :904-951) and in-place ``add_`` / ``mul_`` for optimizers.

All compute goes through libnmg_hip.so; tensors must live on the GPU.
"""
import functools
import weakref

import torch

from . import native
from ._host_loader import host as _host
from .layout import NMGLayout

_layout = functools.lru_cache(maxsize=512)(NMGLayout)      # geometry only: frozen, shared by every tensor of a shape


class GroupedNMTensor(_host.Core):
    """``val`` and ``idx``, the layout, the options of the products and the operands derived for them
    (``rowpack()``, ``fragpack()``, ``densefrag()``, ...) live in the native base class."""

    def __init__(self, val, idx, layout):
        if isinstance(layout, dict):  # accept the reference's nm_strides dict
            layout = NMGLayout(tuple(layout["dense_shape"]), layout["n"], layout["m"],
                               layout["group_size"], layout["sparse_dim"], layout["group_dim"])
        self.layout = layout
        self.val = val
        self.idx = idx
        self.spmm_opt = {"kernel": "auto"}

    # ---- construction ----------------------------------------------------------------------
    @staticmethod
    def from_dense(tensor, n, m, sparse_dim, group_size, group_dim):
        """Per-tile magnitude selection, bit-exact with the reference CPU sparsifier
        (grouped_nm_tensor.py:883-890 -> :701-710 -> :255-297)."""
        native.require_gpu(tensor)
        out = GroupedNMTensor.__new__(GroupedNMTensor)
        out.layout = _layout(tuple(tensor.shape), n, m, group_size, sparse_dim % tensor.dim(), group_dim % tensor.dim())
        out.spmm_opt["kernel"] = "auto"
        _host.sparsify(out, tensor)
        return out

    def clone_layout(self, dense_tensor):
        """New tensor with this tensor's pattern and the values of ``dense_tensor`` at the kept
        positions (what grouped_nm_tensor.py:908-951 describes)."""
        if tuple(dense_tensor.shape) != tuple(self.layout.dense_shape):
            raise ValueError(
                f"Shape mismatch: expected {self.layout.dense_shape}, received {tuple(dense_tensor.shape)}")
        return self._gather(dense_tensor)

    # ---- reference-compatible surface ------------------------------------------------------------
    @property
    def nm_strides(self):
        d = self.layout.as_nm_strides()
        d.update(self.spmm_opt)
        return d

    def set_spmm_opt(self, tile_a=None, acc_width=None, tile_b=None, kernel=None):
        """Reference signature (grouped_nm_tensor.py:892-902).  The CPU tile parameters have no
        meaning here; ``kernel`` selects the GPU matmul kernel: auto | mfma | smfmac | skinny."""
        if kernel is not None:
            if kernel not in native.KERNELS:
                raise ValueError(f"kernel must be one of {sorted(native.KERNELS)}")
            self.spmm_opt["kernel"] = kernel
        for k, v in (("tile_a", tile_a), ("acc_width", acc_width), ("tile_b", tile_b)):
            if v is not None:
                self.spmm_opt[k] = v

    # ---- tensor-like attributes the wrapper machinery looks for -------------------------------
    @property
    def dtype(self):
        return self.val.dtype

    @property
    def device(self):
        return self.val.device

    @property
    def shape(self):
        return torch.Size(self.layout.dense_shape)

    def size(self, dim=None):
        return self.shape if dim is None else self.shape[dim]

    def dim(self):
        return len(self.layout.dense_shape)

    def numel(self):
        return self.shape.numel()

    def to(self, device=None, dtype=None, non_blocking=False, copy=False, **_):
        val = self.val.to(device=device, dtype=dtype, non_blocking=non_blocking, copy=copy)
        idx = self.idx.to(device=device, non_blocking=non_blocking, copy=copy)
        out = GroupedNMTensor(val, idx, self.layout)
        out.spmm_opt = dict(self.spmm_opt)
        return out

    def clone(self):
        return self.to(copy=True)

    # ---- serialization: the canonical val/idx and the layout; derived operands are rebuilt ----
    def __getstate__(self):
        return {"val": self.val, "idx": self.idx, "layout": self.layout, "spmm_opt": dict(self.spmm_opt)}

    def __setstate__(self, state):
        self.__init__(state["val"], state["idx"], state["layout"])
        self.spmm_opt = state.get("spmm_opt", {"kernel": "auto"})

    # ---- in-place updates that keep the pattern (used by optimizers) ------------------------
    def _same_pattern(self, other):
        """True when ``other`` keeps the same positions in the same slots: it shares this
        tensor's ``idx`` (every ``clone_layout`` result does) or holds an equal copy.  The
        comparison of two distinct ``idx`` tensors is made once per pair and remembered."""
        if other.idx is self.idx or (other.idx.data_ptr() == self.idx.data_ptr()
                                     and other.idx.shape == self.idx.shape):
            return True
        cached = getattr(self, "_pattern_eq", None)
        if (cached is not None and cached[0]() is other.idx and cached[1] == other.idx._version
                and cached[2] == self.idx._version):
            return cached[3]
        same = other.idx.device == self.idx.device and bool(torch.equal(other.idx, self.idx))
        # remembered per tensor object (weak reference), not per address: a freed idx block comes
        # back at the same address with another pattern in it
        self._pattern_eq = (weakref.ref(other.idx), other.idx._version, self.idx._version, same)
        return same

    def _other_val(self, other):
        if isinstance(other, GroupedNMTensor):
            if other.layout != self.layout:
                raise ValueError("layout mismatch")
            if self._same_pattern(other):
                return other.val
            # same layout, another choice of columns: slot s of the two tensors names different
            # positions, so the values go through the dense view and are gathered at this
            # tensor's kept positions
            return self.clone_layout(other.to_dense()).val
        if hasattr(other, "wrapped_tensor"):
            return self._other_val(other.wrapped_tensor)
        if hasattr(other, "to_dense") and not isinstance(other, torch.Tensor):
            other = other.to_dense()
        if isinstance(other, torch.Tensor) and other.dim() > 0:
            return self.clone_layout(other).val
        return other

    def add_(self, other, *, alpha=1):
        self.val.add_(self._other_val(other), alpha=alpha)
        self._drop_operands()
        return self

    def mul_(self, other):
        self.val.mul_(self._other_val(other))
        self._drop_operands()
        return self

    def zero_(self):
        self.val.zero_()
        self._drop_operands()
        return self

    def copy_(self, other):
        self.val.copy_(self._other_val(other))
        self._drop_operands()
        return self

    # ---- weight gradient -------------------------------------------------------------------------
    def masked_product(self, rows_op, cols_op, reduction_last=False):
        """New tensor with this tensor's pattern whose kept entries are those of
        ``rows_op^T @ cols_op`` (``rows_op`` [T, R], ``cols_op`` [T, C] for a weight [R, C]): the
        weight gradient of a linear layer, accumulated in fp32 and written straight into the
        ``val`` layout.  16-bit types; extents that are multiples of 8.
        ``reduction_last=True`` takes the operands transposed, ``rows_op`` [R, T] and ``cols_op``
        [C, T] (the product ``rows_op @ cols_op^T``, as the weight gradient of ``torch.mm(W, B)``
        finds them: grad_out and B); T must then be a multiple of 8, R and C may be anything."""
        return self._masked_product(rows_op, cols_op, reduction_last)

    def masked_product_supported(self, rows_op, cols_op, reduction_last=False):
        return self._masked_product_supported(rows_op, cols_op, reduction_last)

    def __repr__(self):
        lay = self.layout
        return (f"GroupedNMTensor(shape={tuple(lay.dense_shape)}, n:m:g={lay.n}:{lay.m}:{lay.group_size}, "
                f"sparse_dim={lay.sparse_dim}, group_dim={lay.group_dim}, dtype={self.val.dtype}, "
                f"device={self.val.device})")


def spmm_tt(weight, b):
    """C = W @ B for a 2-D ``GroupedNMTensor`` W [R, C] and a dense B [C, N] (``torch.mm``), contiguous where N > 16 and
    the data is 16-bit.  On the sparse matrix cores where the pattern fits 2 of 4 along dim 1, else on the dense ones:
    from a transposed copy of B, from B as it lies where that is faster (short reductions), or cut along the reduction
    (few columns).  What these do not take goes through ``spmm`` on the transposed operands."""
    return _host.spmm_tt(weight, b)


def spmm_tt_dense(weight, b, *, reduce_dim):
    """C = op(W) @ B on the dense matrix cores:
    ``reduce_dim=0``: B is [R, N], C = W^T @ B is [C, N] (the gradient with respect to B of
    ``torch.mm(W, B)``); ``reduce_dim=1``: B is [C, N], C = W @ B is [R, N].  Takes 16-bit data, an
    m that is a power of two or three times one and more than 16 columns; the rest goes through ``spmm`` on the
    transposed operands."""
    return _host.spmm_tt_dense(weight, b, reduce_dim)


def spmm(weight, x, bias=None, *, reduce_dim, kernel=None):
    """Y = X @ op(W) for a 2-D ``GroupedNMTensor`` W of shape [R, C].

    ``reduce_dim=1``: X is [T, C], Y = X @ W^T is [T, R]  (F.linear forward).
    ``reduce_dim=0``: X is [T, R], Y = X @ W   is [T, C]  (gradient w.r.t. the input).
    The route is chosen in ``csrc/nmg_host.cpp``.
    """
    return _host.spmm(weight, x, bias, reduce_dim, kernel)
