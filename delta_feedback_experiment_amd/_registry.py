"""Registration of this package's operators with PyTorch's dispatcher.

Each operator is a schema with a device kernel, a fake implementation and,
where it has one, an autograd formula -- what ``torch.library.custom_op``
registers, written straight onto the dispatcher keys.  A single call of a
decode step or a small block is mostly host time: ``custom_op``'s generic
layers (argument trees flattened and rebuilt around the autograd function,
schema defaults filled in, alias and disabled-kernel checks around the
kernel) took about half of the 33 us of each operator of a decode token, and
more for the training operator, whose outputs hold a list.

The dispatcher's own order is kept: autograd, version counters, then tracing
modes and functionalization, then the device kernel, so fake tensors, ``torch.compile``,
saved-tensor hooks and the refusal of CPU tensors work as for any operator.
"""

from __future__ import annotations

from functools import partial

import torch
from torch import _C

# kept over a reload of this module, which leaves the operators standing
_LIBRARIES: dict[str, torch.library.Library] = globals().get("_LIBRARIES", {})  # one an operator
_WRITTEN: dict = globals().get("_WRITTEN", {})  # operator -> positions of the arguments it writes
_FORMULAS: dict = globals().get("_FORMULAS", {})  # operator -> its setup_context and backward


def device_op(schema: str):
    """Decorator: register ``fn`` as the device kernel of ``schema`` (``name(args)
    -> returns``) and return the operator, with ``fn``'s docstring and
    ``custom_op``'s ways to add to it (``register_kernel`` for another device,
    ``register_vmap``, ...).  Arguments the schema marks as written have their
    version counters raised, whichever kernel runs.  A name defined again (its
    module reloaded) replaces the operator."""

    def register(fn):
        name = schema.split("(", 1)[0]
        if name in _LIBRARIES:
            _LIBRARIES.pop(name)._destroy()
        lib = _LIBRARIES[name] = torch.library.Library("pkda_mi355x", "FRAGMENT")
        lib.define(schema, tags=(torch.Tag.pt2_compliant_tag,))
        op = getattr(torch.ops.pkda_mi355x, name).default
        _WRITTEN[op] = [i for i, a in enumerate(op._schema.arguments)
                        if a.alias_info is not None and a.alias_info.is_write]
        lib.impl(name, fn, "CUDA")
        if _WRITTEN[op]:
            _versions(op, name, lib)
        _autograd(op, name, lib)
        op.__doc__ = fn.__doc__
        for way in ("register_kernel", "register_vmap", "register_torch_dispatch"):
            setattr(op, way, partial(getattr(torch.library, way), op, lib=lib))
        op.register_fake = partial(torch.library.register_fake, op, lib=lib, allow_override=True)
        op.register_autograd = lambda backward, *, setup_context=None: register_autograd(op, backward, setup_context)
        return op

    return register


def _raise_versions(op, args) -> None:
    for i in _WRITTEN[op]:
        t = args[i]
        if t is not None and not t.is_inference():
            torch.autograd.graph.increment_version(t)


def _versions(op, name: str, lib) -> None:
    def kernel(keyset, *args):
        _raise_versions(op, args)
        with _C._AutoDispatchBelowADInplaceOrView():
            return op.redispatch(keyset & _C._after_ADInplaceOrView_keyset, *args)

    lib.impl(name, kernel, "ADInplaceOrView", with_keyset=True)


def register_fake(op, fn) -> None:
    torch.library.register_fake(op.name(), fn, lib=_LIBRARIES[op._schema.name.split("::")[1]])


def register_autograd(op, backward, setup_context) -> None:
    """Give ``op`` a backward formula, ``backward(ctx, *output_grads)`` and
    ``setup_context(ctx, inputs, output)`` as ``torch.library.register_autograd``
    takes them (a list output's gradients come one by one, after the others)."""
    _FORMULAS[op] = (setup_context or (lambda ctx, inputs, output: None), backward)


def _autograd(op, name: str, lib) -> None:
    returns = op._schema.returns
    listed = bool(returns) and isinstance(returns[-1].type, _C.ListType)  # its tensors become outputs one by one

    def flat(out):
        if not listed:
            return out
        return (*out[:-1], *out[-1]) if len(returns) > 1 else tuple(out)

    def forward(ctx, keyset, *args):
        with _C._AutoDispatchBelowAutograd():
            out = op.redispatch(keyset & _C._after_autograd_keyset, *args)
        if op in _FORMULAS:
            _FORMULAS[op][0](ctx, args, out)
        return flat(out)

    def backward(ctx, *grads):
        # under create_graph the formula's own operator, which has none, takes
        # part in the graph and raises when a second derivative reaches it
        if op not in _FORMULAS:
            raise RuntimeError(f"Trying to backward through {op} but no autograd formula was registered.")
        return (None, *_FORMULAS[op][1](ctx, *grads))

    function = type(f"pkda_mi355x_{name}", (torch.autograd.Function,),
                    {"forward": staticmethod(forward), "backward": staticmethod(backward)})

    def kernel(keyset, *args):
        if _C.is_grad_enabled() and _C._any_requires_grad(*args):
            out = function.apply(keyset, *args)
            if not listed:
                return out
            last = list(out[len(returns) - 1:])
            return (*out[:len(returns) - 1], last) if len(returns) > 1 else last
        with _C._AutoDispatchBelowAutograd():
            return op.redispatch(keyset & _C._after_autograd_keyset, *args)

    lib.impl(name, kernel, "Autograd", with_keyset=True)


def call(op, *args):
    """``op(*args)``, past the autograd and version keys when nothing asks for
    gradients: the same dispatch below them, without the round trips through
    the kernels above.  (Dynamo traces the plain call.)"""
    if torch.compiler.is_compiling() or (_C.is_grad_enabled() and _C._any_requires_grad(*args)):
        return op(*args)
    _raise_versions(op, args)
    with _C._AutoDispatchBelowADInplaceOrView():
        return op(*args)
