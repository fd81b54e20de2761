"""Senders with more edges than they have places in the lists (mops_amd/csrc/sender_buckets.hpp:
edges_of_sender), in graphs whose other senders do not: the weight gradients of OPSAW and SASAW against
the oracle.

The hubs are the first and the last sender, two next to each other and one alone; the index is longer
than the 1024 positions that are looked at together and does not come out even in quarters; the
per-edge rows have one, two and four columns per lane; edges in slots and by arrival, below and above
48 edges per sender on average, and in shares. (SASAW lists its senders' edges otherwise, but where it looks through the index
for every sender, in `slots` here but for 16 components in double; see test_sasaw_columns.py.)
"""
import numpy as np
import pytest

from tests import support
from tests.support import cpu_vjp, hip_vjp, to_device

pytestmark = pytest.mark.gpu

SIZES = {  # edges, senders, edges of a hub
    "slots": (9011, 331, 90),
    "slots_of_a_long_index": (60007, 2003, 700),
    "by_arrival_dense": (50003, 901, 129),
    "by_arrival_many_senders": (90001, 4503, 400),
}


def with_hubs(case, key, senders, edges_of_hub, seed):
    rng = np.random.default_rng(seed)
    index = case[key].copy()
    edges = rng.permutation(len(index))
    for number, hub in enumerate((0, 5, 6, senders // 2, senders - 1)):
        index[edges[number * edges_of_hub : (number + 1) * edges_of_hub]] = hub
    return dict(case, **{key: index})


def compare(oracle, device, op, case, key, dtype, what):
    import torch

    single = dtype == np.float32
    exact = cpu_vjp(oracle, op, support.in_float64(case))["W"]
    other = cpu_vjp(oracle, op, case if single else support.magnitudes(case))["W"]
    on_device = to_device(case, device)
    # the index as it is, and one element off the 16-byte boundaries
    beside = torch.empty(on_device[key].numel() + 1, dtype=torch.int32, device=device)[1:]
    beside.copy_(on_device[key])
    for inputs in (on_device, dict(on_device, **{key: beside})):
        gradient = hip_vjp(op, inputs)["W"]
        support.assert_calibrated(
            gradient.cpu().numpy(), exact, dtype, what, other if single else None, None if single else other
        )
        assert (gradient == hip_vjp(op, inputs)["W"]).all(), "the same call twice gave different bits"


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("columns", [3, 32, 100, 200])
@pytest.mark.parametrize("size", list(SIZES))
def test_opsaw(oracle, device, size, columns, dtype):
    edges, senders, of_hub = SIZES[size]
    case = support.opsaw_case(edges + columns, dtype, E=edges, K=2, L=columns, n_nodes=senders, allow_empty=True)
    compare(oracle, device, "opsaw", with_hubs(case, "indices_W", senders, of_hub, columns), "indices_W", dtype, f"{size} grad_W")


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize(
    "shape",
    [  # edges, senders, K, L, edges of a hub: one to four columns per lane, senders split by a launch of its own
        (60007, 26701, 65, 3, 2200),
        (60007, 26701, 65, 20, 2200),
        (60007, 26701, 65, 50, 2200),
        (60007, 26701, 65, 100, 2200),
        (60007, 26701, 65, 140, 2200),
        (330007, 5001, 17, 33, 3000),  # split by the edges' kernel
    ],
    ids=lambda s: "x".join(map(str, s)),
)
def test_opsaw_in_shares(oracle, device, shape, dtype):
    """Senders in shares and buckets (mops_amd/csrc/sender_shares.hpp), some with more edges than a bucket's place in LDS."""
    edges, senders, rows, columns, of_hub = shape
    case = support.opsaw_case(edges + columns, dtype, E=edges, K=rows, L=columns, n_nodes=senders, allow_empty=True)
    compare(oracle, device, "opsaw", with_hubs(case, "indices_W", senders, of_hub, columns), "indices_W", dtype, f"{shape} grad_W")


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("components,columns", [(4, 5), (9, 32), (16, 20)])
@pytest.mark.parametrize("size", ["slots", "slots_of_a_long_index"])
def test_sasaw(oracle, device, size, components, columns, dtype):
    edges, senders, of_hub = SIZES[size]
    case = support.sasaw_case(
        edges + columns, dtype, E=edges, nA=components, L=columns, n_nodes=senders, n2=components, n3=components, N=40,
        allow_empty=True,
    )  # fmt: skip
    compare(oracle, device, "sasaw", with_hubs(case, "indices_W_1", senders, of_hub, columns), "indices_W_1", dtype, f"{size} grad_W")
