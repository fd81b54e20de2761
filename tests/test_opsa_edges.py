"""OPSA / OPSAW gradients of many edges (mops_amd/csrc/opsa_edges.hip) against the oracle.

Rows at the edges of its tiles of 16 columns and of its steps of four; nodes of one edge, of about 16
and of thousands, and nodes without edges; the edges of every sender listed beside it in slots, by
arrival, and by a counting sort; indices outside the tensor.
"""
import numpy as np
import pytest

from tests import support
from tests.support import cpu_vjp, hip_vjp, to_device

pytestmark = pytest.mark.gpu

SHAPES = [  # edges, nodes, columns of A, columns of B
    (30000, 900, 17, 33),
    (60001, 29000, 32, 63),
    (100003, 6000, 16, 35),
    (100000, 3, 4, 47),
    (200000, 9000, 13, 49),
    (400001, 25000, 1, 17),
    (550000, 20000, 21, 40),
]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("op", ["opsa", "opsaw"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_against_the_oracle(oracle, device, shape, op, dtype):
    edges, nodes, n_a, n_b = shape
    make = support.opsaw_case if op == "opsaw" else support.opsa_case
    size = {"E": edges, "n_nodes": nodes} if op == "opsaw" else {"J": edges, "n_out": nodes}
    case = make(sum(shape), dtype, K=n_a, L=n_b, allow_empty=True, **size)
    exact, absolute, on_device = support.in_float64(case), support.magnitudes(case), to_device(case, device)
    single = dtype == np.float32
    expected = cpu_vjp(oracle, op, exact)
    bound = cpu_vjp(oracle, op, case if single else absolute)
    gradients = hip_vjp(op, on_device)
    again = hip_vjp(op, on_device)
    for key, gradient in gradients.items():
        support.assert_calibrated(
            gradient.cpu().numpy(), expected[key], dtype, f"{shape} grad_{key}", bound[key] if single else None,
            None if single else bound[key],
        )  # fmt: skip
        # the same bits twice, and alone
        assert (gradient == again[key]).all(), key
        assert (gradient == hip_vjp(op, on_device, wanted=[key])[key]).all(), key


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nodes", [1500, 7000])
def test_senders_outside_the_tensor_count_as_zero(oracle, device, nodes, dtype):
    case = support.opsaw_case(3, dtype, E=100000, K=18, L=37, n_nodes=nodes)
    lost = np.random.default_rng(1).integers(0, 100000, 5000)
    with_zero = dict(case, B=case["B"].copy())
    with_zero["B"][lost] = 0
    case["indices_W"] = case["indices_W"].copy()
    case["indices_W"][lost] = np.where(lost % 2 == 0, -1, nodes)
    gradients = hip_vjp("opsaw", to_device(case, device))
    expected = cpu_vjp(oracle, "opsaw", with_zero)
    support.assert_close(gradients["W"].cpu().numpy(), expected["W"], dtype, "grad_W")
    support.assert_close(gradients["A"].cpu().numpy(), expected["A"], dtype, "grad_A")
    assert (gradients["B"][lost] == 0).all()
