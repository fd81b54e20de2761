"""The native functions behind the package (mops_amd/csrc/array_ops.cpp) against the same calls through
the interpreter: same bits, same choice of outputs, and every argument they do not take left to it."""
import numpy as np
import pytest

from tests import support

pytestmark = pytest.mark.gpu

CASES = {
    "hpe": lambda dtype: support.hpe_case(1, dtype, I=70, nA=12, J=90, K=3),
    "sap": lambda dtype: support.sap_case(2, dtype, I=70, nA=5, nB=6, K=40, nO=7),
    "opsa": lambda dtype: support.opsa_case(3, dtype, J=210, K=5, L=9, n_out=8),
    "opsaw": lambda dtype: support.opsaw_case(4, dtype, E=210, K=5, L=9, n_nodes=8),
    "sasaw": lambda dtype: support.sasaw_case(5, dtype, E=210, nA=4, L=9, n_nodes=8, n2=3, n3=5, N=30),
}


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("op", list(CASES))
def test_native_functions(device, op, dtype, monkeypatch):
    import torch

    import mops_amd
    from mops_amd import _c_lib, ops

    native = ops._native
    assert not isinstance(native, _c_lib._NoFunctions), "mops_amd/lib/_array_ops.so has not been built"
    spec = support.OPS[op]
    t = support.to_device(support.add_cotangents(CASES[op](dtype), op), device)
    inputs = [t[name] for name in spec.inputs]
    forward_inputs = inputs + ([t["output_size"]] if "output_size" in t else [])
    gradients = [t["grad_grad_" + name] for name in spec.differentiable]

    def through_the_interpreter(function, *arguments, **flags):
        with monkeypatch.context() as patch:
            patch.setattr(ops, "_native", _c_lib._NoFunctions())
            return getattr(mops_amd, function)(*arguments, **flags)

    def same(a, b):
        a, b = (x if isinstance(x, tuple) else (x,) for x in (a, b))
        assert len(a) == len(b)
        for x, y in zip(a, b):
            assert (x is None) == (y is None)
            assert x is None or (x.dtype == y.dtype and torch.equal(x, y))

    calls = [(spec.function, forward_inputs), (spec.function + "_vjp", [t["grad_output"], *inputs])]
    if op in support.SECOND_ORDER:
        calls.append((spec.function + "_vjp_vjp", [*gradients, t["grad_output"], *inputs]))
    for function, arguments in calls:
        expected = through_the_interpreter(function, *arguments)
        same(getattr(mops_amd, function)(*arguments), expected)
        # (and from copies that are not laid out as the kernels want them, which ops.py converts)
        odd = [
            x if not isinstance(x, torch.Tensor) else x.long() if x.dtype == torch.int32
            else torch.stack([x, x], -1)[..., 0]
            for x in arguments
        ]  # fmt: skip
        same(getattr(mops_amd, function)(*odd), expected)
    function, arguments = calls[1]
    flags = {"compute_grad_A": False}
    same(getattr(mops_amd, function)(*arguments, **flags), through_the_interpreter(function, *arguments, **flags))
    with pytest.raises(mops_amd.MopsError):
        getattr(mops_amd, function)(t["grad_output"], inputs[0][:-1], *inputs[1:])
