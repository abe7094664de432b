"""onebitsparsemul_amd - one-bit 2:4 sparse GEMM for MI355X (gfx950).

Python surface of the reference package ``onebit_sparse_mul`` (onebit_sparse_mul/__init__.py:12-145) on top
of libonebitmul.so: same callables, same argument meaning, intended semantics where the reference's own code
is inconsistent (result allocated on the operands' device, metadata passed in the binding's argument order,
``y = x @ W.T`` in the linear layer). GPU work always goes through the HIP library; nothing falls back to a
host computation.
"""
import torch
import torch.nn as nn

from . import _native
from ._semi_structured_conversions import (
    mask_creator,
    sparse_semi_structured_from_dense_cutlass,
    sparse_semi_structured_to_dense_cutlass,
)

__all__ = [
    "cuda_binary_mul", "cuda_binary_mul_", "binary_quant", "pack_binary", "unpack_binary", "dequant_desparse_tile",
    "py_binary_gemm", "BinaryLinear_2_4", "PreparedWeight", "mask_creator", "sparse_semi_structured_from_dense_cutlass",
    "sparse_semi_structured_to_dense_cutlass", "set_weight_cache", "clear_weight_cache",
]


_compiled = None


def _binding():
    """The compiled torch binding `onebit_sparse_cuda` (reference: onebit_sparse_mul/torch_kernel_cuda.cpp), which also has the
    host side of this package's own calls."""
    global _compiled
    if _compiled is None:
        from . import onebit_sparse_cuda  # noqa: PLC0415  (compiled module, built in-tree)
        _compiled = onebit_sparse_cuda
    return _compiled


def set_weight_cache(entries):
    """Let `cuda_binary_mul` / `onebit_mul` / the C entry points keep the reordered copy of up to `entries` weights
    per GPU, keyed by the weight tensors' addresses (0, the default, keeps nothing: the reference's behaviour).
    Only for weights that are neither modified nor freed while cached; see include/onebit_sparse_tensor.h."""
    _native.set_weight_cache(entries)


def clear_weight_cache():
    _native.clear_weight_cache()


def cuda_binary_mul(A, B, meta):
    """C = W @ B with W the one-bit 2:4 weight stored as (A bits, meta); returns fp32 (m, n) on B's device.
    Reference: onebit_sparse_mul/__init__.py:12-15."""
    return _binding().binary_mul(A, B, meta)


def cuda_binary_mul_(A, B, C, meta):
    """In-place form: writes into C (fp32 or fp16, (m, n)). Reference: onebit_sparse_mul/__init__.py:17-19."""
    _binding().onebit_mul(A, B, meta, C)
    return C


def binary_quant(tensor):
    """value > 0 -> 1, else 0. Reference: onebit_sparse_mul/__init__.py:22-23."""
    return (tensor > 0).to(torch.int64)


def pack_binary(tensor):
    """(rows, cols) of 0/1 -> (rows, cols/8) uint8; element 8c+i of a row is bit i of byte c.
    Reference: onebit_sparse_mul/__init__.py:25-34."""
    rows, cols = tensor.shape
    if cols % 8:
        raise ValueError("last dimension must be a multiple of 8")
    weights = (1 << torch.arange(8, device=tensor.device, dtype=torch.int64))
    return (tensor.reshape(rows, cols // 8, 8).to(torch.int64) * weights).sum(-1).to(torch.uint8)


def unpack_binary(packed_tensor):
    """Inverse of pack_binary; returns uint8 0/1. Reference: onebit_sparse_mul/__init__.py:36-45."""
    rows, pcols = packed_tensor.shape
    shifts = torch.arange(8, device=packed_tensor.device, dtype=torch.int64)
    bits = (packed_tensor.to(torch.int64)[..., None] >> shifts) & 1
    return bits.reshape(rows, pcols * 8).to(torch.uint8)


def dequant_desparse_tile(packed_sparse_tile, meta_tile):
    """(k/2, m/8) packed bits + (m, k/16) reordered metadata -> dense (m, k) weight with values in {-1, 0, +1}.
    Reference: onebit_sparse_mul/__init__.py:47-65 (whose shapes do not compose; this is the intended result)."""
    bits = unpack_binary(packed_sparse_tile).T.contiguous()  # (m, k/2)
    values = torch.where(bits == 1, 1, -1).to(torch.int32)
    return sparse_semi_structured_to_dense_cutlass(values, meta_tile)


def py_binary_gemm(x, packed_sparse_tensor, sparse_meta):
    """Host check: x (batch, k) @ W.T with W = dequant_desparse_tile(...), as torch.matmul on the dense weight.
    Reference: onebit_sparse_mul/__init__.py:67-97."""
    if packed_sparse_tensor.dtype != torch.uint8:
        raise ValueError("packed_sparse_tensor must be `torch.uint8`")
    if sparse_meta.dtype != torch.int16:
        raise ValueError("Sparse Meta must be `torch.int16`")
    if packed_sparse_tensor.shape[0] * 2 != x.shape[1]:
        raise ValueError("x.shape[1] must equal 2 * packed_sparse_tensor.shape[0] (the weight's in-features)")
    dense = dequant_desparse_tile(packed_sparse_tensor, sparse_meta)
    return torch.matmul(x, dense.to(x.dtype).T)


class PreparedWeight:
    """A packed weight reordered once for the gfx950 kernels (see include/onebit_sparse_tensor.h)."""

    def __init__(self, packed_binary_sparse, meta, layout=_native.META_REFERENCE):
        self.m = meta.shape[0]
        self.k = meta.shape[1] * 16
        self.buffer = _binding().prepare(packed_binary_sparse, meta, self.m, self.k, layout)

    def matmul(self, b, out=None, c=None, alpha=1.0, beta=0.0, out_dtype=torch.float16):
        return _binding().matmul_prepared(self.buffer, b, c, out, self.m, self.k, alpha, beta, out_dtype)

    def linear(self, x, bias=None, out=None, out_dtype=torch.float16):
        """y (tokens, m) = x (tokens, k) @ W.T (+ bias): the layer's form, x and y token-major, no transposes."""
        if x.data_ptr() % 16:
            x = x.clone()  # a view that starts inside a 16-byte unit
        if out is None:
            out = torch.empty((x.shape[0], self.m), dtype=out_dtype, device=x.device)
        return _native.linear_prepared(self.buffer, x, out, self.m, self.k, bias=bias)


class BinaryLinear_2_4(nn.Module):
    """1-bit 2:4 sparse linear layer: y = x @ W.T (+ bias when one has been assigned), W (outfeatures, infeatures)
    stored at 1.5 bits per weight. Reference: onebit_sparse_mul/__init__.py:101-145."""

    def __init__(self, infeatures: int, outfeatures: int, out_dtype=None):
        """out_dtype: dtype of the kernel's result. None (default): float16 for float16 activations (the sums are
        accumulated in fp32 and rounded once; a sum of infeatures/2 terms of +-x can exceed float16's range for large
        activations), bfloat16 for bfloat16 activations (which are multiplied as they are) and float32 for every other
        activation dtype, so that the only precision loss is the cast of x to float16. torch.float32 returns the
        reference layer's fp32 product for 16-bit activations as well (onebit_sparse_mul/__init__.py:12-14:
        cuda_binary_mul returns an fp32 C)."""
        super().__init__()
        if infeatures % 32 != 0 or outfeatures % 64 != 0:
            raise ValueError("`infeatures` must be divisible by 32 and `outfeatures` by 64.")
        if out_dtype not in (None, torch.float16, torch.float32):
            raise ValueError("out_dtype must be None, torch.float16 or torch.float32")
        self.infeatures = infeatures
        self.outfeatures = outfeatures
        self.out_dtype = out_dtype
        self.register_buffer("packed_binary_sparse", torch.zeros((infeatures // 2, outfeatures // 8), dtype=torch.uint8))
        self.register_buffer("meta", torch.zeros((outfeatures, infeatures // 16), dtype=torch.int16))
        self.vaild = False
        self._prepared = None
        self.bias = None  # optional (outfeatures,) tensor added to the output; the model script assigns it

    def pack(self, weight):
        """weight (outfeatures, infeatures): prune to 2:4 by magnitude, keep the signs.
        Reference: onebit_sparse_mul/__init__.py:130-145."""
        if tuple(weight.shape) != (self.outfeatures, self.infeatures):
            raise ValueError(f"weight must have shape ({self.outfeatures}, {self.infeatures})")
        if weight.is_cuda and weight.dtype in (torch.float16, torch.bfloat16, torch.float32):
            # one fused HIP kernel (mask, compress, quantise, transpose-pack, reorder); same result as below
            weight = weight.contiguous()
            if weight.data_ptr() % 16:
                weight = weight.clone()  # a view that starts inside a 16-byte unit
            a, meta = _binding().pack_weight(weight, True, _native.META_REFERENCE)
            buffers = self._buffers
            # where nn.Module.__setattr__ puts a registered buffer, without its 1.5 us per attribute: not for a class that sets
            # attributes its own way, nor where a registration hook is to see the buffer (or torch keeps those elsewhere)
            if (type(self).__setattr__ is nn.Module.__setattr__ and "packed_binary_sparse" in buffers and "meta" in buffers
                    and getattr(nn.modules.module, "_global_buffer_registration_hooks", None) == {}):
                buffers["packed_binary_sparse"], buffers["meta"] = a, meta
                object.__setattr__(self, "vaild", True)
                object.__setattr__(self, "_prepared", None)
            else:
                self.packed_binary_sparse, self.meta = a, meta
                self.vaild = True
                self._prepared = None
            return
        w = weight * mask_creator(weight).to(weight.dtype)
        if w.dtype not in (torch.half, torch.bfloat16, torch.int32):
            w = w.to(torch.half)
        sparse, meta = sparse_semi_structured_from_dense_cutlass(w)
        bits = binary_quant(sparse).T.contiguous()
        self.packed_binary_sparse = pack_binary(bits)
        self.meta = meta
        self.vaild = True
        self._prepared = None

    def _load_from_state_dict(self, state_dict, prefix, local_metadata, strict, missing_keys, unexpected_keys,
                              error_msgs):
        super()._load_from_state_dict(state_dict, prefix, local_metadata, strict, missing_keys, unexpected_keys,
                                      error_msgs)
        # a packed weight is there only if both buffers came from the state dict
        if prefix + "packed_binary_sparse" in state_dict and prefix + "meta" in state_dict:
            self.vaild = True
        self._prepared = None

    def _prepared_on(self, device):
        if not self.vaild:
            raise NotImplementedError("the BinaryLinear_2_4 layer holds no packed weight: call pack() first")
        prepared = self._prepared
        if prepared is None or prepared.buffer.device != device:
            prepared = self._prepared = PreparedWeight(self.packed_binary_sparse.to(device), self.meta.to(device))
        return prepared.buffer

    def forward(self, x):
        # one kernel: reads the tokens where they lie, adds the bias, writes (tokens, outfeatures)
        prepared = self._prepared
        if prepared is not None and self.vaild:
            y = _binding().layer_forward(prepared.buffer, x, self.bias, self.outfeatures, self.infeatures, self.out_dtype)
            if y is not None:
                return y  # else x is on another device than the prepared weight
        return _binding().layer_forward(self._prepared_on(x.device), x, self.bias, self.outfeatures, self.infeatures,
                                        self.out_dtype)


def forward_grouped(layers, xs):
    """The forward passes of several BinaryLinear_2_4 layers on inputs with the same number of tokens, in one library
    call (one kernel launch per 16 layers for up to 64 tokens): the q / k / v or gate / up projections of a decoder
    layer. xs: one tensor for all layers, or one per layer. Returns the list of outputs, each what layer(x) returns."""
    layers = list(layers)
    shared = isinstance(xs, torch.Tensor)
    xs = [xs] if shared else list(xs)
    if not shared and len(xs) != len(layers):
        raise ValueError("one input per layer (or one for all)")
    if not layers:
        return []
    ys = _binding().grouped_forward(layers, xs)
    if ys is None:  # a layer's weight is not prepared yet, or on another device than its input
        for i, layer in enumerate(layers):
            layer._prepared_on(xs[0 if shared else i].device)
        ys = _binding().grouped_forward(layers, xs)
    # nothing to share (token counts or types differ, or one layer with inputs on two devices): the layers one by one
    return ys or [layer(xs[0 if shared else i]) for i, layer in enumerate(layers)]
