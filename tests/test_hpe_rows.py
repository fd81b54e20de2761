"""HPE with a lane per row (mops_amd/csrc/hpe_rows.hip) against the oracle, and which kernels a shape takes.

The shapes sit at the edges of the layout: one row more or less than tiles of 64 and 128 rows hold,
one or two rows per lane, groups of features that do not come out even, features without a
monomial, lists of more than 64 terms, every order, factors outside the tensor.
"""
import os
import subprocess

import numpy as np
import pytest

from tests import support
from tests.support import cpu_forward, cpu_vjp, hip_forward, hip_vjp, to_device

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHAPES = [  # rows, features, monomials, order
    (10000, 1, 1, 1),
    (10049, 10, 50, 3),
    (10111, 16, 65, 2),
    (11240, 4, 300, 3),
    (12801, 33, 100, 2),
    (13000, 30, 150, 4),
    (14001, 20, 31, 6),
    (16001, 33, 330, 2),
    (16447, 7, 129, 5),
    (18001, 100, 200, 3),
    (20000, 119, 70, 2),
    (10300, 174, 64, 3),
]

PROGRAM = """
#include <cstdio>
#include <cstdlib>
#include "dispatch_thresholds.hpp"
int main(int n, char** a) {
    using namespace mops::amd::thresholds;
    const char* names[] = {"tiles", "rows", "few"};
    for (int i = 1; i + 3 < n; i += 4) {
        const long long r = atoll(a[i]), f = atoll(a[i + 1]), t = atoll(a[i + 2]), e = atoll(a[i + 3]);
        printf("%s %s %s\\n", names[int(hpe_forward(r, f, t, e))], names[int(hpe_vjp(r, f, t, e))],
               names[int(hpe_vjp_vjp(r, f, t, e))]);
    }
}
"""


def chosen(tmp_path, points):
    source = tmp_path / "chosen.cpp"
    source.write_text(PROGRAM)
    program = tmp_path / "chosen"
    include = os.path.join(ROOT, "mops_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-I", include, "-o", str(program), str(source)], check=True)
    arguments = [str(value) for point in points for value in point]
    done = subprocess.run([str(program), *arguments], check=True, capture_output=True, text=True)
    return [line.split() for line in done.stdout.splitlines()]


def test_short_tables_of_many_rows_do_not_take_the_tiles(tmp_path):
    """Points at which the tiles were measured at 2 to 7 times the time of the kernels chosen here (and
    the other way round for the long tables)."""
    expected = {  # rows, features, factors, bytes per value
        (100000, 10, 150, 4): ["rows", "rows", "few"],
        (100000, 10, 150, 8): ["rows", "rows", "few"],
        (100000, 100, 600, 4): ["rows", "rows", "tiles"],
        (100000, 250, 600, 8): ["rows", "tiles", "tiles"],
        (4000, 250, 600, 8): ["few", "few", "few"],
        (100000, 10, 8000, 4): ["tiles", "tiles", "tiles"],
        (1000, 2000, 400000, 4): ["tiles", "tiles", "tiles"],
        (100, 10, 150, 8): ["tiles", "few", "few"],
    }
    assert dict(zip(expected, chosen(tmp_path, expected))) == expected


def case_of(shape, dtype):
    rows, features, monomials, order = shape
    case = support.hpe_case(sum(shape), dtype, I=rows, nA=features, J=monomials, K=order)
    return support.add_cotangents(case, "hpe")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_against_the_oracle(oracle, device, shape, dtype):
    case = case_of(shape, dtype)
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


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_factors_outside_the_tensor_count_as_zero(device, dtype):
    """(and an infinity in a row reaches no other row)"""
    import torch

    case = case_of((10100, 12, 80, 3), dtype)
    indices = case["indices_A"].copy()
    indices[5, 1], indices[11, 0], indices[70, 2] = -1, 12, 2**31 - 1
    kept = np.delete(indices, [5, 11, 70], axis=0)
    spoiled = to_device(dict(case, indices_A=indices), device)
    clean = to_device(dict(case, indices_A=kept, C=np.delete(case["C"], [5, 11, 70])), device)
    # (a monomial with a factor outside is zero, and so are its terms in the gradients of its other
    # factors; the sums are made in another order where monomials are missing: 80 terms, rounded 80 times
    # at most, of which the largest sum is a fifth of all magnitudes: 80 * 5 * the unit of rounding)
    bound = 400 * np.finfo(dtype).eps / 2
    for got, want in ((hip_forward("hpe", spoiled), hip_forward("hpe", clean)), (hip_vjp("hpe", spoiled)["A"], hip_vjp("hpe", clean)["A"])):
        assert (got - want).abs().max() <= bound * want.abs().max()
    with_infinity = dict(clean, A=clean["A"].clone())
    with_infinity["A"][77, 3] = float("inf")
    others = torch.arange(10100, device=device) != 77
    assert torch.equal(hip_forward("hpe", with_infinity)[others], hip_forward("hpe", clean)[others])
    assert torch.equal(hip_vjp("hpe", with_infinity)["A"][others], hip_vjp("hpe", clean)["A"][others])
