"""SASAW with a lane per feature column (mops_amd/csrc/sasaw_columns.hip) against the oracle.

4, 9 and 16 values of every component index; columns at the edges of its tiles of 16, 32 and 64 and
just beside them; lists of edges around the number it asks for ahead and around 64; nodes without
edges, a single node, and more nodes than wavefronts; senders outside the tensor; every way the edges
of a sender are listed.
"""
import numpy as np
import pytest

from tests import support
from tests.support import cpu_forward, cpu_vjp, hip_forward, hip_vjp, to_device

pytestmark = pytest.mark.gpu

SHAPES = [  # edges, nodes, components, entries, columns
    (1, 1, 4, 10, 1),
    (3, 2, 9, 40, 31),
    (65, 1, 9, 250, 33),
    (130, 2, 16, 300, 17),
    (400, 300, 4, 24, 64),
    (900, 30, 9, 250, 65),
    (1000, 20, 16, 800, 48),
    (1500, 50, 9, 1100, 100),
    (2000, 40, 4, 30, 130),
    (6000, 5000, 9, 100, 20),
    (30000, 1000, 16, 100, 12),
    # the senders' edges by a counting sort, in one level and in two
    (9000, 3, 4, 12, 5),
    (40000, 600, 4, 12, 3),
]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_against_the_oracle(oracle, device, shape, dtype):
    edges, nodes, n, entries, columns = shape
    case = support.sasaw_case(
        sum(shape), dtype, E=edges, nA=n, L=columns, n_nodes=nodes, n2=n, n3=n, N=entries, allow_empty=True
    )
    exact, absolute, on_device = support.in_float64(case), support.magnitudes(case), to_device(case, device)
    single = dtype == np.float32

    def check(name, run, actual):
        support.assert_calibrated(
            actual.cpu().numpy(), run(exact), dtype, f"{shape} {name}", run(case) if single else None,
            None if single else run(absolute),
        )  # fmt: skip

    check("output", lambda c: cpu_forward(oracle, "sasaw", c), hip_forward("sasaw", on_device))
    gradients = hip_vjp("sasaw", on_device)
    for key, gradient in gradients.items():
        check(f"grad_{key}", lambda c: cpu_vjp(oracle, "sasaw", c)[key], gradient)
    again = hip_vjp("sasaw", on_device)
    for key in gradients:  # the same bits twice, and alone
        assert (gradients[key] == again[key]).all(), key
        assert (gradients[key] == hip_vjp("sasaw", on_device, wanted=[key])[key]).all(), key


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize(
    "shape",
    [(2, 1, 9, 30, 16), (700, 300, 9, 60, 16), (700, 300, 4, 24, 13), (501, 200, 9, 250, 32), (300, 200, 4, 30, 33), (1999, 31, 9, 250, 40), (20001, 9000, 9, 250, 32)],
    ids=lambda s: "x".join(map(str, s)),
)  # fmt: skip
def test_edges_side_by_side(oracle, device, shape, dtype):
    """Two or four edges of a node at a time: nodes with fewer, and with any remainder; several tiles of columns."""
    test_against_the_oracle(oracle, device, shape, dtype)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize(
    "shape",
    [  # edges, nodes, components, columns: a node by a workgroup (up to 512 to 1024 nodes), a range of them by a wavefront
        (7, 3, 9, 32),
        (700, 3, 9, 33),
        (5000, 2, 4, 20),
        (1100, 512, 16, 16),
        (1030, 1024, 4, 16),
        (1030, 1025, 4, 16),
        # one launch for all gradients up to 16 384 edges, 8192 of nodes with many
        (3, 1, 4, 5),
        (4, 2, 4, 5),
        (8192, 40, 9, 32),
        (8193, 40, 9, 32),
        (16384, 400, 9, 20),
        (16385, 400, 9, 20),
        (9000, 4500, 9, 40),
        (9000, 4500, 16, 24),
    ],
    ids=lambda s: "x".join(map(str, s)),
)
def test_one_node_has_a_third_of_the_edges(oracle, device, shape, dtype):
    """The edges of one node go to several wavefronts, those of many small ones to one."""
    edges, nodes, n, columns = shape
    case = support.sasaw_case(
        sum(shape), dtype, E=edges, nA=n, L=columns, n_nodes=nodes, n2=n, n3=n, N=100, allow_empty=True
    )
    receivers = np.random.default_rng(sum(shape)).integers(0, nodes, edges)
    receivers[: edges // 3] = nodes // 2
    receivers.sort()
    case["indices_output_1"] = receivers.astype(np.int32)
    exact, absolute, on_device = support.in_float64(case), support.magnitudes(case), to_device(case, device)
    other = case if dtype == np.float32 else absolute

    def check(name, run, actual):
        same, terms = (run(other), None) if dtype == np.float32 else (None, run(other))
        support.assert_calibrated(actual.cpu().numpy(), run(exact), dtype, f"{shape} {name}", same, terms)

    check("output", lambda c: cpu_forward(oracle, "sasaw", c), hip_forward("sasaw", on_device))
    for key, gradient in hip_vjp("sasaw", on_device).items():
        check(f"grad_{key}", lambda c: cpu_vjp(oracle, "sasaw", c)[key], gradient)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize(
    "shape",
    [  # edges, nodes, components, columns, edges of one sender
        (17003, 401, 9, 16, 3000),  # a sender by a workgroup, more of its edges than fit into LDS
        (60007, 2003, 9, 32, 2500),  # two to four to a bucket
        (60007, 2003, 16, 40, 5),  # three tiles of columns and few nodes, more than three tiles
        (90001, 4503, 9, 70, 2100),
        (90001, 4503, 4, 200, 5),
        (262144, 5003, 4, 3, 40000),  # as many shares as there can be, a sender with edges in all of them
        (262145, 40009, 4, 2, 5),  # fewer, larger shares
        (150001, 70001, 4, 3, 2100),  # senders beyond 16 bits, most of them with one edge or two
    ],
    ids=lambda s: "x".join(map(str, s)),
)
def test_buckets_of_senders(oracle, device, shape, dtype):
    """The senders' edges in shares and buckets (mops_amd/csrc/sender_shares.hpp), split by the launch for the other
    gradients and by one of its own."""
    edges, nodes, n, columns, of_hub = shape
    case = support.sasaw_case(
        edges + columns, dtype, E=edges, nA=n, L=columns, n_nodes=nodes, n2=n, n3=n, N=40, allow_empty=True
    )
    hub = np.random.default_rng(3).permutation(edges)[:of_hub]
    case["indices_W_1"][hub] = nodes - 3
    exact = cpu_vjp(oracle, "sasaw", support.in_float64(case))["W"]
    other = cpu_vjp(oracle, "sasaw", case if dtype == np.float32 else support.magnitudes(case))["W"]
    on_device = to_device(case, device)
    together, alone = hip_vjp("sasaw", on_device)["W"], hip_vjp("sasaw", on_device, wanted=["W"])["W"]
    assert (together == alone).all()
    same, terms = (other, None) if dtype == np.float32 else (None, other)
    support.assert_calibrated(together.cpu().numpy(), exact, dtype, f"{shape} grad_W", same, terms)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("components", [4, 9, 16])
def test_listed_senders_shared_by_a_workgroup(oracle, device, components, dtype):
    """Lists whose entries the wavefronts of a workgroup share (more than 16 384 edges, no more nodes
    than workgroups at a time): around 64 and 128 entries, senders outside the tensor."""
    import torch

    edges, nodes, columns = 17003, 401, 16
    case = support.sasaw_case(
        components, dtype, E=edges, nA=components, L=columns, n_nodes=nodes, n2=components, n3=components, N=60,
        allow_empty=True,
    )  # fmt: skip
    rng = np.random.default_rng(components)
    # (a quarter of the index each, away from the ends of the quarters)
    quarters = [rng.permutation(np.arange(edges // 4 * q + 8, edges // 4 * (q + 1) - 8)) for q in range(4)]
    senders = rng.integers(8, nodes, edges).astype(np.int32)
    counts = {
        0: (16, 16, 16, 16), 1: (17, 16, 16, 16), 2: (32, 32, 32, 31), 3: (32, 32, 32, 32), 4: (0, 0, 32, 32),
        5: (33, 0, 0, 0), 6: (3, 30, 33, 5), 7: (0, 0, 0, 300), nodes: (9, 9, 9, 9), -1: (5, 0, 5, 0),
    }  # fmt: skip
    for q, places in enumerate(quarters):
        at = 0
        for sender, of_quarter in counts.items():
            senders[places[at : at + of_quarter[q]]] = sender
            at += of_quarter[q]
    inside = (senders >= 0) & (senders < nodes)
    assert np.bincount(senders[inside], minlength=nodes)[:8].tolist() == [sum(counts[k]) for k in range(8)]
    on_device = to_device(dict(case, indices_W_1=senders), device)
    # (for the oracle, an edge that does not count is one without B)
    case["indices_W_1"] = np.where(inside, senders, 0).astype(np.int32)
    case["B"] = np.where(inside[:, None], case["B"], 0).astype(dtype)
    exact = cpu_vjp(oracle, "sasaw", support.in_float64(case))["W"]
    other = cpu_vjp(oracle, "sasaw", case if dtype == np.float32 else support.magnitudes(case))["W"]
    beside = torch.empty(edges + 1, dtype=torch.int32, device=device)[1:]
    beside.copy_(on_device["indices_W_1"])
    for index in (on_device["indices_W_1"], beside):  # as it is, and off the 16-byte boundaries
        actual = hip_vjp("sasaw", dict(on_device, indices_W_1=index))["W"].cpu().numpy()
        same, terms = (other, None) if dtype == np.float32 else (None, other)
        support.assert_calibrated(actual, exact, dtype, f"{components} grad_W", same, terms)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_senders_outside_the_tensor_count_as_zero(oracle, device, dtype):
    case = support.sasaw_case(7, dtype, E=300, nA=9, L=20, n_nodes=12, n2=9, n3=9, N=120)
    lost = np.random.default_rng(1).integers(0, 300, 40)
    with_zero = dict(case, B=case["B"].copy())
    with_zero["B"][lost] = 0
    case["indices_W_1"] = case["indices_W_1"].copy()
    case["indices_W_1"][lost] = np.where(lost % 2 == 0, -1, 12)
    on_device = to_device(case, device)
    support.assert_close(
        hip_forward("sasaw", on_device).cpu().numpy(), cpu_forward(oracle, "sasaw", with_zero), dtype, "output"
    )
    gradients = hip_vjp("sasaw", on_device)
    expected = cpu_vjp(oracle, "sasaw", with_zero)
    support.assert_close(gradients["W"].cpu().numpy(), expected["W"], dtype, "grad_W")
    support.assert_close(gradients["A"].cpu().numpy(), expected["A"], dtype, "grad_A")
    assert (gradients["B"][lost] == 0).all()


def test_more_senders_than_the_counting_sort_counts_at_a_time(oracle, device):
    small = support.sasaw_case(9, np.float64, E=2000, nA=4, L=1, n_nodes=30, n2=4, n3=4, N=12)
    places = np.sort(np.random.default_rng(2).choice(2200000, 30, replace=False)).astype(np.int32)
    case = dict(small)
    for key in ("W", "grad_output"):
        case[key] = np.zeros((2200000, 4, 1))
        case[key][places] = small[key]
    for key in ("indices_W_1", "indices_output_1"):
        case[key] = places[small[key]]
    expected = cpu_vjp(oracle, "sasaw", small)
    actual = {key: value.cpu().numpy() for key, value in hip_vjp("sasaw", to_device(case, device)).items()}
    support.assert_close(actual["W"][places], expected["W"], np.float64, "grad_W")
    assert np.count_nonzero(actual["W"]) == np.count_nonzero(expected["W"])
    support.assert_close(actual["A"], expected["A"], np.float64, "grad_A")
