"""HPE with many monomials or features (mops_amd/csrc/hpe_tiles.hip) against the oracle.

The shapes sit at the edges of its layout: rows of a tile (4, 8, 16) and one more or less, shares of
the monomials and of the features that do not come out even, features without a monomial, every
order, the largest feature counts that fit in LDS, a counting sort of one and of several workgroups
and with four wavefronts instead of sixteen.
"""
import numpy as np
import pytest

from tests import support
from tests.support import cpu_forward, cpu_vjp, hip_forward, hip_vjp, to_device

pytestmark = pytest.mark.gpu

SHAPES = [  # rows, features, monomials, order
    (1, 300, 5, 1),
    (3, 250, 1025, 2),
    (17, 257, 1000, 3),
    (33, 999, 2049, 4),
    (65, 400, 3001, 5),
    (16, 1201, 700, 6),
    (700, 5, 2400, 6),
    (1100, 21, 4801, 2),
    (4097, 40, 900, 3),
    (9, 3001, 2200, 2),
    (5, 4900, 6000, 2),
    (6, 9900, 300, 3),
]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_against_the_oracle(oracle, device, shape, dtype):
    rows, features, monomials, order = shape
    case = support.hpe_case(sum(shape), dtype, I=rows, nA=features, J=monomials, K=order)
    case = support.add_cotangents(case, "hpe")
    exact, absolute, on_device = support.in_float64(case), support.magnitudes(case), to_device(case, device)
    single = dtype == np.float32

    def check(name, run, actual):
        support.assert_calibrated(
            actual.cpu().numpy(), run(exact), dtype, f"{shape} {name}", run(case) if single else None,
            None if single else run(absolute),
        )  # fmt: skip

    check("output", lambda c: cpu_forward(oracle, "hpe", c), hip_forward("hpe", on_device))
    gradient = hip_vjp("hpe", on_device)["A"]
    check("grad_A", lambda c: cpu_vjp(oracle, "hpe", c)["A"], gradient)
    assert (gradient == hip_vjp("hpe", on_device)["A"]).all(), "the same call twice gave different bits"
    second = support.hip_vjp_vjp("hpe", on_device)
    for key in ("grad_output", "A"):
        check(f"second {key}", lambda c: support.cpu_vjp_vjp(oracle, "hpe", c)[key], second[key])
    for key in ("grad_output", "A"):  # one of the two alone
        alone = support.hip_vjp_vjp("hpe", on_device, wanted=[key])[key]
        assert (alone == second[key]).all(), key
