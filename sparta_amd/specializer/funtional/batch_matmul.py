"""Batched block-sparse matmul: forward kernel plus the two kernels its gradients
need, derived from the forward mode and transposes.

Interface of sparta/specializer/funtional/batch_matmul.py:12-179.
"""
from typing import Any, Dict, List, Optional, Tuple

import torch

from sparta_amd import _lib
from sparta_amd.specializer.kernels import SparTASparseMatMulKernel, OpenAISparseMatMulKernel
from sparta_amd.specializer.funtional.sparse_ctx_base import SparseCtxBase, KernelPlaceholder


def _derive_kernels(mode: str, transpose_A: bool, transpose_B: bool, biased: bool):
    """For C = op(A) op(B): the gradient w.r.t. A and B are matmuls of the other
    two tensors.  Returns, per kernel name, (biased, operand order, transA, transB)
    where the operand order says which of A, B, C plays the role of the new
    kernel's first, second and output tensor."""
    return {
        'forward:C': (biased, 'ABC', transpose_A, transpose_B),
        'backward:A': (False, 'BCA' if transpose_A else 'CBA',
                       transpose_A and transpose_B, transpose_A or not transpose_B),
        'backward:B': (False, 'CAB' if transpose_B else 'ACB',
                       not transpose_A or transpose_B, transpose_A and transpose_B),
    }


def _tile_dims(mode: str, trans_A: bool, trans_B: bool) -> Tuple[str, str]:
    if mode == 'sdd':
        return ('K', 'M') if trans_A else ('M', 'K')
    if mode == 'dsd':
        return ('N', 'K') if trans_B else ('K', 'N')
    return ('M', 'N')


class SparseBatchMatMulCtx(SparseCtxBase):

    def __init__(self, mode: str, transpose_A: bool, transpose_B: bool, biased: bool, compressed: bool,
                 drop_batch: bool = False):
        """`drop_batch`: the result comes without its batch axis (of one entry)."""
        super().__init__()
        self._drop_batch = drop_batch
        self._mode = mode
        self._transpose_A = transpose_A
        self._transpose_B = transpose_B
        self._biased = biased
        self._compressed = compressed
        self._activation: Optional[str] = None
        sparse_tensor = 'ABC'[mode.index('s')]
        self._tesa_shapes: Dict[str, Tuple[str, str]] = {}
        for name, (bias, order, tA, tB) in _derive_kernels(mode, transpose_A, transpose_B, biased).items():
            # letter i of the derived mode = sparsity letter of the tensor in role i
            derived_mode = ''.join(mode['ABC'.index(t)] for t in order)
            self._kernels[name] = KernelPlaceholder(
                name=name,
                impls={'sparta': SparTASparseMatMulKernel, 'openai': OpenAISparseMatMulKernel},
                args=dict(mode=derived_mode, biased=bias, transpose_A=tA, transpose_B=tB,
                          compressed=compressed),
                port_map={sparse_tensor: 'ABC'[order.index(sparse_tensor)]},
                connectable=compressed,
            )
            self._tesa_shapes[name] = _tile_dims(derived_mode, tA, tB)
        self._init_sparse_ports([sparse_tensor])

    def set_shape(self, batch_size: int, M: int, K: int, N: int):
        self._kernels['forward:C'].set_shape(batch_size, M, K, N)
        self._kernels['backward:A'].set_shape(*((batch_size, K, N, M) if self._transpose_A
                                                else (batch_size, M, N, K)))
        self._kernels['backward:B'].set_shape(*((batch_size, N, M, K) if self._transpose_B
                                                else (batch_size, K, M, N)))

    def set_activation(self, activation: Optional[str]):
        """Fuse an activation (None or 'relu') into the forward kernel's epilogue; the
        autograd function then masks the incoming gradient with the sign of the output."""
        if activation not in (None, 'relu'):
            raise ValueError(f'unsupported fused activation: {activation!r}')
        if activation is not None and self._mode == 'dds':
            raise ValueError('the fused activation covers the sdd and dsd kernels only')
        self._activation = activation
        fwd = self._kernels['forward:C'].active_kernel()
        if fwd is not None:
            fwd.set_epilogue(activation)
            if fwd.ready:
                self._bind_operator()

    def _bind_operator(self):
        """The native operator object: the active kernels' launch objects and the autograd node
        that connects them."""
        launch = [None if k.active_kernel() is None else k.active_kernel()._func
                  for k in (self._kernels[name] for name in ('forward:C', 'backward:A', 'backward:B'))]
        self.apply = _lib.native().MatmulOp(*launch, self._transpose_A, self._transpose_B,
                                      self._activation == 'relu', self._drop_batch)

    def build(self, config: Dict[str, Dict[str, Any]]):
        super().build(config)
        fwd = self._kernels['forward:C'].active_kernel()
        if fwd is not None:
            fwd.set_epilogue(self._activation)
        bwd_A = self._kernels['backward:A'].active_kernel()
        if bwd_A is not None:
            if self._transpose_A:
                self.backward_A = lambda grad_C, B: bwd_A(B, grad_C)
            else:
                self.backward_A = lambda grad_C, B: bwd_A(grad_C, B)
        bwd_B = self._kernels['backward:B'].active_kernel()
        if bwd_B is not None:
            if self._transpose_B:
                self.backward_B = lambda grad_C, A: bwd_B(grad_C, A)
            else:
                self.backward_B = lambda grad_C, A: bwd_B(A, grad_C)
        if fwd is not None:
            self._bind_operator()

    def set_sample_inputs(self, sample_inputs: List[torch.Tensor],
                          sample_grads: Optional[List[torch.Tensor]] = None):
        A, B = sample_inputs[0], sample_inputs[1]
        fwd_inputs = [A, B] + ([sample_inputs[2].detach()] if self._biased else [])
        self._kernels['forward:C'].set_sample_inputs(fwd_inputs)
        if sample_grads is None:
            return
        grad_C = sample_grads[0]
        self._kernels['backward:A'].set_sample_inputs([B, grad_C] if self._transpose_A else [grad_C, B])
        self._kernels['backward:B'].set_sample_inputs([grad_C, A] if self._transpose_B else [A, grad_C])

    def get_connections(self, backward: bool = False):
        """Block dimensions that must agree between kernels sharing a compressed
        tensor: one dict per tile axis, kernel name -> parameter name."""
        if not (self._compressed and backward):
            return []
        return [
            {name: f'BLOCK_SIZE_{dims[axis]}_VALUE' for name, dims in self._tesa_shapes.items()}
            for axis in (0, 1)
        ]

    def dense_forward(self, *args):
        return self._kernels['forward:C'].dense_func(*args)


class SparseBatchMatMulFunc:
    """C = op(A) op(B) (+ bias) with its gradients: the autograd node is part of the native
    operator object that the context holds once it is built."""

    @staticmethod
    def apply(sparta_ctx: SparseBatchMatMulCtx, input: torch.Tensor, weight: torch.Tensor,
              bias: Optional[torch.Tensor] = None) -> torch.Tensor:
        return sparta_ctx.apply(input, weight, bias)
