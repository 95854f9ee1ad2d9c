"""The operators' registration: what a backward through an operator without a
formula, a second derivative and a CPU tensor raise, the version counters of
what an operator writes, symbolic sizes, and what can be added to one."""

from __future__ import annotations

import subprocess
import sys

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from delta_feedback_experiment_amd import (_registry, pkda_controls, pkda_norm_gate, pkda_qkv_conv,
                                           pkda_qkv_conv_cached_, pkda_recurrence)
from delta_feedback_experiment_amd.serve import qkv_conv_cached_op

from conftest import ROOT


def _meta(*shape, grad=False):
    return torch.empty(*shape, device="meta", requires_grad=grad)


def test_backward_without_a_formula_raises():
    args = (_meta(2, 3, 96, grad=True), _meta(96, 4), 32, 64, 1e-6, _meta(4, 3, 96), None, True)
    for call in (qkv_conv_cached_op, lambda *a: _registry.call(qkv_conv_cached_op, *a)):
        q, _, _ = call(*args)
        assert q.requires_grad
        with pytest.raises(RuntimeError, match="no autograd formula"):
            q.sum().backward()


def _norm_gate():
    leaves = [_meta(5, 64, grad=True), _meta(5, 64, grad=True), _meta(64, grad=True)]
    return leaves, pkda_norm_gate(*leaves, 1e-6)[0]


def _conv():
    leaves = [_meta(2, 5, 96, grad=True), _meta(96, 4, grad=True)]
    return leaves, pkda_qkv_conv(*leaves, 32, 64, 1e-6)[0]


def _recurrence():
    token, head = (1, 5, 2, 64), (1, 5, 2)
    leaves = [_meta(*s, grad=True) for s in (*[token] * 4, *[head] * 3, (2,), (128,), (2,))]
    return leaves, pkda_recurrence(*leaves, 0.125, 1.5, 1e-6, False)[0]


def _controls():
    leaves = [_meta(2, 5, 2 * 64 + 3 * 2, grad=True), _meta(2, grad=True), _meta(2, grad=True)]
    return leaves, pkda_controls(*leaves, 64, 2)[1]


@pytest.mark.parametrize("make", [_norm_gate, _conv, _recurrence, _controls])
def test_second_derivative_raises(make):
    """Alone, and beside the first derivative, where a second one left out
    would leave gradients that look whole."""
    for penalty in (lambda y, dx: dx.square().sum(), lambda y, dx: y.sum() + dx.square().sum()):
        leaves, y = make()
        dx, = torch.autograd.grad(y.sum(), leaves[:1], create_graph=True)
        assert dx.shape == leaves[0].shape
        with pytest.raises(RuntimeError, match="no autograd formula"):
            penalty(y, dx).backward()
    leaves, y = make()
    grads = torch.autograd.grad(y.sum(), leaves)
    assert [g.shape for g in grads] == [t.shape for t in leaves] and not any(g.requires_grad for g in grads)


def test_statistics_have_no_gradient():
    x, gate, w = _meta(5, 64, grad=True), _meta(5, 64, grad=True), _meta(64, grad=True)
    y, rstd = pkda_norm_gate(x, gate, w, 1e-6)
    assert y.requires_grad and not rstd.requires_grad


def test_saved_tensor_hooks_see_the_inputs():
    packed = []
    x, w = _meta(2, 5, 96, grad=True), _meta(96, 4, grad=True)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(tuple(t.shape)) or t, lambda t: t):
        q, k, v = pkda_qkv_conv(x, w, 32, 64, 1e-6)
    assert packed == [(2, 5, 96), (96, 4)]
    torch.autograd.grad((q, k, v), (x, w), [torch.empty_like(t) for t in (q, k, v)])


def _cached_calls(x, pool):
    """The ways into one writing operator: its public function and itself."""
    w = _meta(96, 4)
    return (lambda: pkda_qkv_conv_cached_(x, w, 32, 64, 1e-6, pool),
            lambda: qkv_conv_cached_op(x, w, 32, 64, 1e-6, pool, None, True))


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("inference", [False, True])
def test_written_tensors_change_version_without_a_device(grad, inference):
    """Once per call, whatever kernel stands in for the device's."""
    pool = _meta(4, 3, 96)
    for call in _cached_calls(_meta(2, 1, 96, grad=grad), pool):
        before = pool._version
        with torch.inference_mode(inference):
            call()
        assert pool._version == before + 1
    with torch.inference_mode():  # tensors that count no versions
        for call in _cached_calls(_meta(2, 1, 96), _meta(4, 3, 96)):
            call()
    with FakeTensorMode():
        pool = torch.empty(4, 3, 96, device="meta")
        before = pool._version
        qkv_conv_cached_op(torch.empty(2, 1, 96, device="meta"), torch.empty(96, 4, device="meta"), 32, 64, 1e-6,
                           pool, None, True)
        assert pool._version == before + 1


def test_saved_tensor_written_before_backward_raises():
    for i in range(2):
        pool = _meta(4, 3, 96)
        y = (pool * _meta(4, 3, 96, grad=True)).sum()
        _cached_calls(_meta(2, 1, 96), pool)[i]()
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            y.backward()


class _ConvOfAnyWidth(torch.nn.Module):
    def forward(self, x, w):
        return pkda_qkv_conv(x, w, 32, 2 * x.shape[2] // 3, 1e-6)


def test_integers_may_be_symbolic():
    """One graph for all widths under a dynamic compile, an export with a
    dynamic width that runs at another one, and the same for every integer
    argument of the other operators."""
    graphs = []
    run = torch.compile(_ConvOfAnyWidth(), backend=lambda g, _: graphs.append(g) or g.forward, dynamic=True,
                        fullgraph=True)
    for heads in (2, 3, 5):
        assert run(_meta(2, 5, 96 * heads), _meta(96 * heads, 4))[0].shape == (2, 5, 32 * heads)
    assert len(graphs) == 1
    heads = torch.export.Dim("heads", min=2, max=64)
    program = torch.export.export(_ConvOfAnyWidth(), (_meta(2, 5, 384), _meta(384, 4)),
                                  dynamic_shapes=({2: 96 * heads}, {0: 96 * heads}))
    assert program.module()(_meta(2, 5, 576), _meta(576, 4))[0].shape == (2, 5, 192)
    ops = torch.ops.pkda_mi355x
    for op in (ops.pkda_qkv_conv, ops.pkda_qkv_conv_backward, ops.pkda_controls_act, ops.pkda_controls_backward,
               ops.qkv_conv_cached_):
        assert " int " not in str(op.default._schema) and "SymInt" in str(op.default._schema)


def test_cpu_tensors_are_refused():
    x = torch.zeros(5, 64)
    with pytest.raises(NotImplementedError, match="CPU"):
        pkda_norm_gate(x, x, torch.ones(64), 1e-6)


def test_operators_can_be_added_to_and_defined_again():
    """custom_op's ways to add to an operator, its docstring, and a module that
    defines it a second time."""

    def define(factor):
        @_registry.device_op("registry_test(Tensor x, float by) -> Tensor")
        def registry_test(x, by):
            """Scaled."""
            raise AssertionError("no device here")

        _registry.register_fake(registry_test, lambda x, by: torch.empty_like(x))
        registry_test.register_kernel("cpu", lambda x, by: factor * by * x)
        return registry_test

    x = torch.randn(3, 4, requires_grad=True)
    for factor in (2.0, 3.0):
        op = define(factor)
        assert op.__doc__ == "Scaled."
        assert torch.equal(op(x, by=5.0), factor * 5.0 * x)
        with pytest.raises(RuntimeError, match="no autograd formula"):
            op(x, 5.0).sum().backward()
        op.register_autograd(lambda ctx, dy: (factor * 5.0 * dy, None))
        assert torch.equal(torch.autograd.grad(op(x, 5.0).sum(), x)[0], torch.full_like(x, factor * 5.0))
        op.register_vmap(lambda info, in_dims, x, by: (op(x, by) + 1, in_dims[0]))
        assert torch.equal(torch.vmap(lambda r: op(r, 5.0))(x.detach()), factor * 5.0 * x.detach() + 1)
        assert op(_meta(3, 4), 5.0).shape == (3, 4)
    assert pkda_norm_gate.__doc__.startswith("Fused RMSNorm")


def test_operator_modules_reload():
    program = """
import importlib, torch
from delta_feedback_experiment_amd import _registry, controls, conv, norm_gate, ops, pkda, serve
meta = lambda *s: torch.empty(*s, device="meta", requires_grad=True)
for modules in ((_registry,), (pkda, controls, conv, norm_gate, ops, serve), (_registry, norm_gate, serve)):
    for module in modules:
        importlib.reload(module)
    y, _ = norm_gate.pkda_norm_gate(meta(5, 64), meta(5, 64), meta(64), 1e-6)
    y.sum().backward()
    pool = torch.empty(4, 3, 96, device="meta")
    q, _, _ = serve.pkda_qkv_conv_cached_(meta(2, 1, 96), meta(96, 4), 32, 64, 1e-6, pool)
    assert y.shape == (5, 64) and q.shape == (2, 1, 32) and pool._version == 1
"""
    subprocess.run([sys.executable, "-c", program], check=True, cwd=ROOT)


@pytest.mark.gpu
def test_written_tensors_change_version():
    from delta_feedback_experiment_amd import pkda_decode_step_, pkda_qkv_conv_cached_

    print("[gpu] version counters of the pools", flush=True)
    dev = torch.device("cuda:0")
    pool, a_pool, conv = (torch.zeros(*s, device=dev) for s in ((3, 1, 64, 64), (3, 1, 64), (3, 3, 192)))
    q, g, idx = torch.ones(2, 1, 64, device=dev), torch.zeros(2, 1, device=dev), torch.tensor([2, 0], device=dev).int()
    before = [t._version for t in (pool, a_pool, conv)]
    for grad in (False, True):  # with gradients asked for, through the operator's autograd kernel
        pkda_decode_step_(q.clone().requires_grad_(grad), q, q, g, g, pool, idx, a_pool=a_pool, g_atk=g, beta_atk=g,
                          log_atk_scale=torch.zeros(1, device=dev))
        pkda_qkv_conv_cached_(torch.ones(2, 1, 192, device=dev, requires_grad=grad), torch.ones(192, 4, device=dev),
                              64, 128, 1e-6, conv, idx)
        after = [t._version for t in (pool, a_pool, conv)]
        assert all(b > a for a, b in zip(before, after)), (before, after)
        before = after
    with torch.inference_mode():
        pkda_decode_step_(q, q, q, g, g, pool.clone(), idx)
    torch.cuda.synchronize()
