"""Registration of the torch operators, and the one formula the batch product and both convolution variants share for
their second derivatives."""
from __future__ import annotations

import threading

import torch

from .build_ext import TORCH_LIB_PATH

NAMESPACE = "openequivariance_amd"
_library = None
_library_lock = threading.Lock()


def _operators() -> "torch.library.Library":
    """The operators' library, with the C++ autograd kernels (csrc/oeq_torch.cpp) loaded."""
    global _library
    with _library_lock:
        if _library is None:
            if not TORCH_LIB_PATH.exists():
                raise RuntimeError(f"{TORCH_LIB_PATH} is missing: build it with `python -m openequivariance_amd.build_ext`")
            torch.ops.load_library(str(TORCH_LIB_PATH))
            _library = torch.library.Library(NAMESPACE, "FRAGMENT")
        return _library


def define_operator(name: str, arguments, returns: str, implementation, fake, device: str = "CUDA"):
    """Operator ``name`` with tensor ``arguments``, its GPU implementation and its fake kernel.  Registered without the
    wrappers of torch.library.custom_op, which take as long per call as launching a small product does: a forward without
    a graph 14 -> 4.5 us of dispatch, a training step 104 -> 51 us (one CPU, kernels left out; 45 us of that is what
    torch's own product of three tensors takes)."""
    lib = _operators()
    lib.define(f"{name}({', '.join('Tensor ' + a for a in arguments)}) -> {returns}", tags=(torch.Tag.pt2_compliant_tag,))
    lib.impl(name, torch._disable_dynamo(implementation), device)
    torch.library.register_fake(f"{NAMESPACE}::{name}", fake, lib=lib)
    return getattr(getattr(torch.ops, NAMESPACE), name).default


def define_derivatives(forward: str, backward: str, arguments, second_derivatives) -> None:
    """Makes operator ``backward`` (arguments: the first three, the output's gradient, the rest) the derivative of
    ``forward``, and ``second_derivatives(x, y, w, dz, ddx, ddy, ddw, *index)`` that of ``backward``."""
    lib = _operators()
    name, index = backward + "_derivative", list(arguments[3:])
    names = [*arguments[:3], "L3_grad", "L1_cot", "L2_cot", "weights_cot", *index]
    lib.define(f"{name}({', '.join('Tensor ' + a for a in names)}) -> Tensor[]")
    lib.impl(name, second_derivatives, "CompositeImplicitAutograd")
    ops = getattr(torch.ops, NAMESPACE)
    ops.register_derivative(NAMESPACE, forward, backward, 3)
    ops.register_derivative(NAMESPACE, backward, name, 4)


def double_backward_terms(forward, backward_helper, x, y, w, dz, ddx, ddy, ddw, index=(), fused=None):
    """Gradients of ``backward_helper(x, y, w, dz) -> (dx, dy, dw)`` with respect to ``(x, y, w, dz)``
    for incoming cotangents ``(ddx, ddy, ddw)`` of its three outputs, composed from the operator's own
    forward and backward launches (reference: TensorProductBase.py:281-298,
    convolution/ConvolutionBase.py:618-636 and :691-709).  The product is trilinear in (x, y, w), so
    every second derivative is the first-order operator with one argument replaced by its cotangent.
    ``index`` are the trailing graph arguments of the convolution (rows, cols[, transpose_perm]).
    ``fused``, when given, computes all four from one read of the operands; it is not differentiable itself, so a
    graph of the second derivatives (create_graph=True, for third derivatives) is built from the composition."""
    # (a loss that uses only some of the three gradients brings None for the others)
    ddx, ddy, ddw = (torch.zeros_like(like) if cot is None else cot for cot, like in ((ddx, x), (ddy, y), (ddw, w)))
    if fused is not None and not torch.is_grad_enabled():
        return tuple(fused(x, y, w, dz, ddx, ddy, ddw, *index))
    a = backward_helper(ddx, ddy, w, dz, *index)       # x and y replaced
    b = backward_helper(x, y, ddw, dz, *index)         # w replaced
    c = backward_helper(ddx, y, w, dz, *index)
    d = backward_helper(x, ddy, w, dz, *index)
    grad_dz = forward(ddx, y, w, *index) + forward(x, ddy, w, *index) + forward(x, y, ddw, *index)
    return a[0] + b[0], a[1] + b[1], c[2] + d[2], grad_dz
