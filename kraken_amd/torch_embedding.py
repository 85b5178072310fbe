"""The reference's worker-side embedding modules on GPU tensors.

`kraken/pytorch/embedding.py` and `jagged_embedding.py` wrap an autograd Function around
`kraken_native.pull_sparse_table / push_sparse_table`, which reject device tensors
(pytorch/py/pytorch.cc:42,102,116,188) and send the request to a server. Here the table lives on
the same GPU as the tensors: forward is one pull (or one pooled pull) straight into a torch
tensor, backward is one fused dedup + sum + optimizer step on the gradient torch hands over.
Nothing is copied to the host and nothing is synchronised: the table enqueues its kernels on
torch's current stream.

PyTorch is plumbing here (it owns the tensors and the stream); the arithmetic is the table
engine's. The autograd functions are native (csrc/torch_binding.cpp, built with the library).
Importing this module needs torch; nothing else in the package does.
"""
import torch

from . import api
from .configs import as_initializer, as_optim

_native = None


def _load_native():
    """The native autograd functions; loaded with the first table, so that the module (JaggedTensor, the
    classes) can be imported where nothing is built."""
    global _native
    if _native is None:
        api.lib()                               # the native module links against it
        try:
            from . import _torch_native
        except ImportError as e:
            raise ImportError("kraken_amd/_torch_native.so is missing or was built against another torch: build it "
                              "with `python -m kraken_amd.build`") from e
        _native = _torch_native
    return _native


class GpuSparseTable(torch.nn.Parameter):
    """pytorch/sparse_table.py: a Parameter that stands for the table so that autograd calls the
    Function's backward. The rows are not in this tensor but in the engine's table.
    `initializer` and `optim` are the engine's (api.Initializer / api.Optim) or the reference's
    descriptions of them (configs.NormalInitializer(...), configs.Adagrad(...))."""

    def __new__(cls, dimension, initializer=None, optim=None, lr=0.01, capacity_hint=0):
        self = super().__new__(cls, torch.empty(0), requires_grad=True)
        self._dimension = int(dimension)
        self._bound_table = api.SparseTable(dimension, as_initializer(initializer) or api.Initializer.create(
            api.InitializerType.kNormal, {}), capacity_hint=capacity_hint)
        self._bound_optim = as_optim(optim) or api.Optim.create(api.OptimType.kSGD)
        self._native = _load_native().Table(self._bound_table.h, self._bound_optim.raw, self._dimension, float(lr))
        return self

    # the native side reads the handle and the optimizer of these objects: another one is bound there too
    @property
    def _table(self):
        return self._bound_table

    @_table.setter
    def _table(self, table):
        self._native.bind_table(table.h)
        self._bound_table = table

    @property
    def _optim(self):
        return self._bound_optim

    @_optim.setter
    def _optim(self, optim):
        self._native.bind_optim(optim.raw)
        self._bound_optim = optim

    @property
    def lr(self):
        return self._native.lr

    @lr.setter
    def lr(self, lr):
        self._native.lr = float(lr)

    def dimension(self):
        return self._dimension

    def table(self):
        return self._table


class EmbeddingFunction:
    """pytorch/embedding.py:9-23: pulls the rows of `indices`; its backward pushes their gradients."""

    @staticmethod
    def apply(sparse_table, indices):
        return _native.embedding(sparse_table._native, sparse_table, indices)


class Embedding(torch.nn.Module):
    """pytorch/embedding.py:26-43 with the table on the GPU. The optimizer step of the rows is
    part of backward (the reference applies it on the server when the push arrives)."""

    def __init__(self, dimension, initializer=None, optim=None, lr=0.01, capacity_hint=0):
        super().__init__()
        self.sparse_table = GpuSparseTable(dimension, initializer, optim, lr, capacity_hint)

    def forward(self, indices):
        return EmbeddingFunction.apply(self.sparse_table, indices)


class JaggedTensor:
    """pytorch/jagged_tensor.py: tensors that agree in all but their first dimension, kept as one
    `values` tensor and the `offsets` of the pieces (offsets[0] = 0, offsets[-1] = len(values)),
    with optional per-row `weights`. Offsets that live on the GPU are not read back to be checked
    (that would wait for the device); the pooling kernels clamp them to the values' range."""

    def __init__(self, values, offsets, weights=None):
        if not offsets.is_cuda:
            o = offsets.tolist()
            if not o or o[0] != 0 or o[-1] != values.shape[0] or any(b < a for a, b in zip(o, o[1:])):
                raise ValueError("JaggedTensor's offsets is invalid:%s, values shape:%s" % (o, tuple(values.shape)))
        if weights is not None and weights.shape != values.shape:
            raise ValueError("JaggedTensor need values and weights has same shape but got weights shape:%s, "
                             "values shape:%s." % (tuple(weights.shape), tuple(values.shape)))
        self._values, self._offsets, self._weights = values, offsets, weights

    def values(self):
        return self._values

    def offsets(self):
        return self._offsets

    def weights(self):
        return self._weights

    def to(self, device):
        return JaggedTensor(self._values.to(device), self._offsets.to(device),
                            None if self._weights is None else self._weights.to(device))

    @staticmethod
    def from_list_tensors(list_values, list_weights=None):
        """pytorch/jagged_tensor.py:56-84"""
        assert len(list_values) > 0
        tail = list_values[0].shape[1:]
        offsets = [0]
        for v in list_values:
            if v.shape[1:] != tail:
                raise ValueError("JaggedTensor need values has tha same dimension except the first rank.")
            offsets.append(offsets[-1] + v.shape[0])
        weights = None
        if list_weights:
            assert len(list_values) == len(list_weights)
            weights = torch.cat(list_weights, dim=0)
        return JaggedTensor(torch.cat(list_values, dim=0), torch.as_tensor(offsets), weights)


class JaggedEmbeddingFunction:
    """pytorch/jagged_embedding_funcs.py over pytorch/py/jagged_ops.cc, fused with the table."""

    @staticmethod
    def apply(sparse_table, indices, offsets, weights, mode, patch_value):
        return _native.jagged(sparse_table._native, sparse_table, indices, offsets, weights, mode, patch_value)


class JaggedEmbedding(torch.nn.Module):
    """pytorch/jagged_embedding.py:10-52: values / offsets / optional weights of a jagged batch,
    pooled per bag with sum or mean; an empty bag yields patch_value."""

    def __init__(self, dimension, initializer=None, optim=None, lr=0.01, mode="sum", patch_value=0.0,
                 capacity_hint=0):
        super().__init__()
        if mode not in ("sum", "mean"):
            raise ValueError("JaggedEmbedding's mode only support sum/mean.")
        self.sparse_table = GpuSparseTable(dimension, initializer, optim, lr, capacity_hint)
        self._mode = 0 if mode == "sum" else 1
        self._patch_value = float(patch_value)

    def forward(self, values, offsets=None, weights=None):
        """forward(JaggedTensor), as the reference's module is called, or forward(values, offsets,
        weights) with the three tensors themselves."""
        if isinstance(values, JaggedTensor):
            values, offsets, weights = values.values(), values.offsets(), values.weights()
        return JaggedEmbeddingFunction.apply(self.sparse_table, values, offsets, weights, self._mode,
                                             self._patch_value)


class GpuCombineSparseTable(torch.nn.Parameter):
    """pytorch/combine_sparse_table.py: the tables of one combined request. Tables of equal
    dimension form one group of the engine (one launch serves a group); the reference allows
    mixed dimensions, which gives one group per distinct dimension here."""

    def __new__(cls, dimensions, initializers=None, optim=None, lr=0.01, capacity_hint=0):
        self = super().__new__(cls, torch.empty(0), requires_grad=True)
        if initializers is not None and len(initializers) != len(dimensions):
            raise ValueError("dimensions and initializers must have the same length")
        self._dimensions = [int(d) for d in dimensions]
        self._tables = [
            api.SparseTable(d, as_initializer(initializers[i] if initializers else None) or api.Initializer.create(
                api.InitializerType.kNormal, {}), capacity_hint=capacity_hint)
            for i, d in enumerate(self._dimensions)]
        self._members = {}                        # dimension -> positions of its tables in the request
        for i, d in enumerate(self._dimensions):
            self._members.setdefault(d, []).append(i)
        self._groups = {d: api.TableGroup([self._tables[i] for i in idx]) for d, idx in self._members.items()}
        self._bound_optim = as_optim(optim) or api.Optim.create(api.OptimType.kSGD)
        self._native = _load_native().Combine(
            [(self._groups[d].h, d, idx) for d, idx in self._members.items()], [t.h for t in self._tables],
            self._dimensions, self._bound_optim.raw, float(lr))
        return self

    @property
    def _optim(self):
        return self._bound_optim

    @_optim.setter
    def _optim(self, optim):
        self._native.bind_optim(optim.raw)
        self._bound_optim = optim

    @property
    def lr(self):
        return self._native.lr

    @lr.setter
    def lr(self, lr):
        self._native.lr = float(lr)

    def dimensions(self):
        return self._dimensions

    def tables(self):
        return self._tables


class CombineEmbeddingFunction:
    """pytorch/combine_embedding.py:10-31 over Emitter::CombinePullSparseTable /
    CombinePushSparseTable (worker/emitter.cc:185-283, 552-632): ids may repeat, within a table
    and across tables."""

    @staticmethod
    def apply(table, *indices):
        return _native.combine(table._native, table, indices)


class CombineEmbedding(torch.nn.Module):
    """pytorch/combine_embedding.py:34-55: one call pulls every table's rows, one backward pushes
    every table's gradients."""

    def __init__(self, dimensions, initializers=None, optim=None, lr=0.01, capacity_hint=0):
        super().__init__()
        self.combine_sparse_table = GpuCombineSparseTable(dimensions, initializers, optim, lr, capacity_hint)

    def forward(self, indices):
        if len(indices) != len(self.combine_sparse_table.dimensions()):
            raise ValueError("one index tensor per table")
        return CombineEmbeddingFunction.apply(self.combine_sparse_table, *indices)


class CombineJaggedEmbeddingFunction:
    """The pooling of pytorch/combine_jagged_embedding.py:47-80 fused with the tables: a
    pooled pull forward and a pooled push backward, so the [n, dim] rows that the
    reference pulls, scales and then pools (JaggedEmbeddingSum/MeanFunction over
    pytorch/py/jagged_ops.cc) never exist in memory."""

    @staticmethod
    def apply(table, modes, patch_values, values, offsets, weights):
        return _native.combine_jagged(table._native, table, modes, patch_values, values, offsets, weights)


class CombineJaggedEmbedding(torch.nn.Module):
    """pytorch/combine_jagged_embedding.py:11-80: one JaggedTensor per table, pooled per table
    with its own mode and patch value. Per-row weights scale the rows before the pooling, as
    the reference's `embeddings *= weights.unsqueeze(-1)` means to (its `if weights:` raises for
    a tensor of more than one element, so there only a batch without weights gets through)."""

    def __init__(self, dimensions, initializers=None, modes=None, patch_values=None, optim=None, lr=0.01,
                 capacity_hint=0):
        super().__init__()
        if modes:
            assert len(dimensions) == len(modes)
            for mode in modes:
                if mode not in ("sum", "mean"):
                    raise ValueError("CombineJaggedEmbedding's mode only support sum/mean.")
        if patch_values:
            assert len(dimensions) == len(patch_values)
        self.combine_sparse_table = GpuCombineSparseTable(dimensions, initializers, optim, lr, capacity_hint)
        self._modes = [0 if m == "sum" else 1 for m in (modes or ["sum"] * len(dimensions))]
        self._patch_values = [float(p) for p in (patch_values or [0.0] * len(dimensions))]

    def forward(self, inputs):
        assert len(self._modes) == len(inputs)
        return CombineJaggedEmbeddingFunction.apply(
            self.combine_sparse_table, self._modes, self._patch_values, [x.values() for x in inputs],
            [x.offsets() for x in inputs], [x.weights() for x in inputs])
