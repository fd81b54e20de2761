"""SAP with a lane per row (mops_amd/csrc/sap_rows_kernels.hpp) against the oracle.

Batches just large enough for it, whose last wavefront is full, nearly empty and in between; either
index as the inner one, padded and not; columns in one tile and in several, the last one narrower, of
even and odd width; more columns than the matrix cores take; repeated entries of the table.
"""
import numpy as np
import pytest

from tests import support
from tests.support import cpu_forward, cpu_vjp, hip_forward, hip_vjp, to_device

pytestmark = pytest.mark.gpu

SHAPES = [  # rows, values of A, of B, of the output, entries
    (300001, 5, 2, 3, 20),
    (300096, 16, 16, 8, 60),
    (100001, 13, 7, 20, 300),
    (100032, 16, 3, 33, 200),
    (100063, 9, 6, 17, 1500),
    (50001, 4, 9, 90, 700),
    (50048, 20, 3, 66, 900),
    (50000, 3, 24, 65, 1200),
]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_against_the_oracle(oracle, device, shape, dtype):
    rows, n_a, n_b, n_out, entries = shape
    case = support.sap_case(sum(shape), dtype, I=rows, nA=n_a, nB=n_b, K=entries, nO=n_out, sort_output=entries % 3 != 0)
    case = support.add_cotangents(case, "sap")
    exact, absolute, on_device = support.in_float64(case), support.magnitudes(case), to_device(case, device)
    single = dtype == np.float32

    def check(name, run, actual):
        support.assert_calibrated(
            actual.cpu().numpy(), run(exact), dtype, f"{shape} {name}", run(case) if single else None,
            None if single else run(absolute),
        )  # fmt: skip

    check("output", lambda c: cpu_forward(oracle, "sap", c), hip_forward("sap", on_device))
    gradients = hip_vjp("sap", on_device)
    again = hip_vjp("sap", on_device)
    for key in ("A", "B"):
        check(f"grad_{key}", lambda c: cpu_vjp(oracle, "sap", c)[key], gradients[key])
        assert (gradients[key] == again[key]).all(), key
        assert (gradients[key] == hip_vjp("sap", on_device, wanted=[key])[key]).all(), key
    second = support.hip_vjp_vjp("sap", on_device)
    for key in ("grad_output", "A", "B"):
        check(f"second {key}", lambda c: support.cpu_vjp_vjp(oracle, "sap", c)[key], second[key])
