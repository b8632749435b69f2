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


class Native:
    """An operator's part in the C++ kernels (csrc/oeq_torch.cpp): what they run, and the scratch that they are lent.  None of it
    is taken back: operators live as long as the process."""
    KINDS = {"tp_forward": 0, "tp_backward": 1, "tp_double": 2, "conv_forward": 3, "conv_backward": 4, "conv_double": 5}

    def __init__(self, id: int):
        self.id, self.ops = id, getattr(torch.ops, NAMESPACE)

    @classmethod
    def create(cls, handles, dtype64, index64, dims, scratch=0, conv=False, shared=False, deterministic=False, overwrites=True,
               few_limits=(0, 0), first=(), second=()):
        """``handles``: kernel sets (main, for few rows, of the double backward; None where there is none).  None where the
        main one is not a handle of the C library."""
        from . import runtime as rt
        raw = [getattr(getattr(h, "_h", None), "value", None) or 0 for h in handles]
        if not raw[0]:
            return None
        _operators()
        ops = getattr(torch.ops, NAMESPACE)
        ops.native_library(rt.entry_points())
        return cls(ops.native_operator([int(dtype64), int(index64), *dims, int(scratch), int(conv), int(shared), int(deterministic),
                                        int(overwrites), *raw, *few_limits], [int(v) for t in first for v in t],
                                       [int(v) for t in second for v in t]))


def define_operator(name: str, arguments, returns: str, implementation, fake, device: str = "CUDA", native=None, kind: str = ""):
    """Operator ``name`` with tensor ``arguments``, its GPU implementation and its fake kernel.  With ``native`` the C++ kernel
    of ``kind`` is its implementation, and ``implementation`` that of the operator ``name``_general, which takes what the kernel
    leaves.  Registered without the
    wrappers of torch.library.custom_op, which take as long per call as launching a small product does: a forward without
    a graph 14 -> 4.5 us of dispatch, a training step 104 -> 51 us (one CPU, kernels left out; 45 us of that is what
    torch's own product of three tensors takes)."""
    lib = _operators()
    general = name if native is None else name + "_general"
    for n in {name, general}:
        lib.define(f"{n}({', '.join('Tensor ' + a for a in arguments)}) -> {returns}", tags=(torch.Tag.pt2_compliant_tag,))
    lib.impl(general, torch._disable_dynamo(implementation), device)
    if native is not None:
        native.ops.native_kernel(NAMESPACE, name, general, native.id, native.KINDS[kind])
    torch.library.register_fake(f"{NAMESPACE}::{name}", fake, lib=lib)
    return getattr(getattr(torch.ops, NAMESPACE), name).default


def define_derivatives(forward: str, backward: str, arguments, second_derivatives, native=None, fused=None) -> None:
    """Makes operator ``backward`` (arguments: the first three, the output's gradient, the rest) the derivative of
    ``forward``, and ``second_derivatives(x, y, w, dz, ddx, ddy, ddw, *index)`` that of ``backward``: with ``native`` and the name
    of the ``fused`` operator, where that one cannot serve directly."""
    lib = _operators()
    name, index = backward + "_derivative", list(arguments[3:])
    names = [*arguments[:3], "L3_grad", "L1_cot", "L2_cot", "weights_cot", *index]
    general = name if native is None or fused is None else name + "_general"
    for n in {name, general}:
        lib.define(f"{n}({', '.join('Tensor ' + a for a in names)}) -> Tensor[]")
    lib.impl(general, second_derivatives, "CompositeImplicitAutograd")
    if general != name:
        native.ops.native_derivative(NAMESPACE, name, fused, general, native.id)
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
