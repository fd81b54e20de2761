"""Calls on caller-owned streams: capture into a HIP graph and replay, and two host threads at once.

The library launches on the stream named with mops_amd_set_stream (per host
thread) and, in asynchronous mode, neither allocates nor synchronises once its
scratch block has its size, so a call can be captured; SASAW's vjp forks to a
side stream and joins again inside the call, which a capture has to follow.
"""
import ctypes
import threading

import numpy as np
import pytest
import torch

from tests import support
from tests.support import OPS

pytestmark = pytest.mark.gpu

CASES = {
    "hpe": lambda d: support.hpe_case(21, d, I=300, nA=20, J=150, K=3),
    "sap": lambda d: support.sap_case(22, d, I=700, nA=13, nB=7, K=300, nO=20),
    "opsa": lambda d: support.opsa_case(23, d, J=2000, K=13, L=20, n_out=70, allow_empty=True),
    "opsaw": lambda d: support.opsaw_case(24, d, E=2000, K=13, L=32, n_nodes=70, allow_empty=True),
    "sasaw": lambda d: support.sasaw_case(25, d, E=2000, nA=9, L=32, n_nodes=70, allow_empty=True),
    # paths with more than one kernel per call and with scratch memory between them:
    # segments cut into pieces and added up (OPSA forward of long segments)
    "opsa_pooling": lambda d: support.opsa_case(26, d, J=6000, K=13, L=20, n_out=8),
    # blocks of 64 columns, grad_A added to by one launch after the other
    "sasaw_many_columns": lambda d: support.sasaw_case(27, d, E=1500, nA=9, L=160, n_nodes=50, allow_empty=True),
    # more than 4000 nodes: the senders' edges listed by arrival, on counters that every replay must find at zero
    "opsaw_many_senders": lambda d: support.opsaw_case(29, d, E=30000, K=4, L=16, n_nodes=9000, allow_empty=True),
    # (components that are not all 4, 9 or 16: the others have their edges ordered without counters)
    "sasaw_many_senders_by_arrival": lambda d: support.sasaw_case(30, d, E=30000, nA=4, L=16, n_nodes=16000, n2=3, n3=4, N=30, allow_empty=True),
    "sasaw_many_senders": lambda d: support.sasaw_case(28, d, E=30000, nA=4, L=16, n_nodes=16000, n2=4, n3=4, N=30, allow_empty=True),
}


def _operation(name):
    return name.split("_")[0]


def _call(op, case):
    import mops_amd

    op = _operation(op)
    spec = OPS[op]
    forward = getattr(mops_amd, spec.function)
    backward = getattr(mops_amd, spec.function + "_vjp")
    arguments = [case[name] for name in spec.inputs]
    if op in ("sap", "opsa", "sasaw"):
        arguments.append(case["output_size"])
    output = forward(*arguments)
    gradients = backward(case["grad_output"], *[case[name] for name in spec.inputs])
    gradients = gradients if isinstance(gradients, (tuple, list)) else (gradients,)
    return [output, *gradients]


@pytest.mark.parametrize("op", list(CASES))
def test_graph_replays_match_eager_calls(device, op):
    case = support.to_device(CASES[op](np.float32), device)
    eager = [t.clone() for t in _call(op, case)]
    torch.cuda.synchronize()

    stream = torch.cuda.Stream(device=device)
    stream.wait_stream(torch.cuda.current_stream(device))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        _call(op, case)  # the scratch block takes its size outside the capture
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            captured = _call(op, case)
    torch.cuda.synchronize()
    for replay in range(3):
        for tensor in captured:
            tensor.fill_(float("nan"))
        # eager work of the program between the replays
        other = _call(op, case)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for got, want, again in zip(captured, eager, other):
            assert torch.equal(got, want), (op, replay)
            assert torch.equal(again, want), (op, replay)


@pytest.mark.parametrize("op", sorted(support.SECOND_ORDER))
def test_second_order_calls_replayed_from_a_graph(device, op):
    """With both cotangents given, the second-order functions of these shapes launch kernels only (no
    temporary from the stream's memory pool), so they can be captured; replays against eager calls."""
    from mops_amd._c_lib import device_library

    library = device_library()
    spec = OPS[op]
    case = support.to_device(support.add_cotangents(CASES[op](np.float64), op), device)

    def call():
        library.cdll.mops_amd_set_stream(torch.cuda.current_stream(device).cuda_stream)
        library.cdll.mops_amd_set_synchronous(0)
        outputs, arguments = support._vjp_vjp_arguments(
            spec, case, None, None, lambda x: torch.full_like(x, float("nan"))
        )
        library.call(spec.function + "_vjp_vjp", *arguments)
        return outputs

    try:
        eager = {key: value.clone() for key, value in call().items()}
        torch.cuda.synchronize()
        stream = torch.cuda.Stream(device=device)
        stream.wait_stream(torch.cuda.current_stream(device))
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(stream):
            call()
            torch.cuda.synchronize()
            with torch.cuda.graph(graph, stream=stream):
                captured = call()
        torch.cuda.synchronize()
        for replay in range(2):
            for tensor in captured.values():
                tensor.fill_(float("nan"))
            other = call()  # eager work between the replays
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            for key in eager:
                assert torch.equal(captured[key], eager[key]), (op, key, replay)
                assert torch.equal(other[key], eager[key]), (op, key, replay)
    finally:
        support._bind_stream(library, device)


def test_two_host_threads_on_their_own_streams(oracle, device):
    """Two host threads, each on a stream of its own, call different operations at the same time:
    the per-thread state (stream, scratch block, error message) keeps them apart, and both get
    the oracle's results."""
    results = {}
    errors = []
    ready = threading.Barrier(2)

    def worker(op):
        try:
            host_case = CASES[op](np.float32)
            case = support.to_device(host_case, device)
            stream = torch.cuda.Stream(device=device)
            ready.wait()
            with torch.cuda.stream(stream):
                first = [t.clone() for t in _call(op, case)]
                for _ in range(20):
                    again = _call(op, case)
                stream.synchronize()
            results[op] = (host_case, first, all(torch.equal(a, b) for a, b in zip(first, again)))
        except Exception as error:  # pragma: no cover - reported below
            errors.append((op, repr(error)))
            ready.abort()

    threads = [threading.Thread(target=worker, args=(op,)) for op in ("opsaw", "sasaw")]
    for thread in threads:
        thread.start()
    for thread in threads:
        thread.join()
    assert not errors, errors
    for op in ("opsaw", "sasaw"):
        host_case, first, repeatable = results[op]
        assert repeatable, op
        spec = OPS[op]
        support.assert_close(first[0].cpu().numpy(), support.cpu_forward(oracle, op, host_case), np.float32, op)
        expected = support.cpu_vjp(oracle, op, host_case)
        for name, got in zip(spec.differentiable, first[1:]):
            support.assert_close(got.cpu().numpy(), expected[name], np.float32, f"{op} grad_{name}")


def test_threads_that_end_hand_their_scratch_block_on(device):
    """A thread's scratch block goes to the next new thread instead of being lost."""
    from mops_amd._c_lib import device_library

    library = device_library()
    library.cdll.mops_amd_scratch_capacity.restype = ctypes.c_int64
    library.cdll.mops_amd_reserve_scratch.argtypes = [ctypes.c_int64]
    seen = []

    def worker(reserve):
        torch.cuda.set_device(device)
        if reserve:
            assert library.cdll.mops_amd_reserve_scratch(3 << 20) == 0
        else:
            # the first use of the state takes over what an ended thread left
            assert library.cdll.mops_amd_reserve_scratch(1) == 0
        seen.append(library.cdll.mops_amd_scratch_capacity())

    for reserve in (True, False):
        thread = threading.Thread(target=worker, args=(reserve,))
        thread.start()
        thread.join()
    assert seen[0] >= 3 << 20
    assert seen[1] == seen[0]


def test_growing_the_scratch_block_during_a_capture_is_refused(device):
    """No allocation can happen while a stream is being captured: the call fails with a message
    instead (a host-side check; nothing is launched)."""
    from mops_amd._c_lib import device_library

    library = device_library()
    library.cdll.mops_amd_scratch_capacity.restype = ctypes.c_int64
    library.cdll.mops_amd_reserve_scratch.argtypes = [ctypes.c_int64]
    torch.cuda.set_device(device)
    library.cdll.mops_amd_set_stream(torch.cuda.current_stream(device).cuda_stream)
    assert library.cdll.mops_amd_reserve_scratch(1) == 0
    capacity = library.cdll.mops_amd_scratch_capacity()
    assert capacity >= 1 << 20

    marker = torch.zeros(16, device=device)
    stream = torch.cuda.Stream(device=device)
    stream.wait_stream(torch.cuda.current_stream(device))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            library.cdll.mops_amd_set_stream(stream.cuda_stream)
            library.cdll.mops_amd_set_synchronous(0)
            marker.add_(1.0)
            within = library.cdll.mops_amd_reserve_scratch(capacity)  # fits: fine during a capture
            status = library.cdll.mops_amd_reserve_scratch(4 * capacity)
            message = library.last_error()
    library.cdll.mops_amd_set_stream(torch.cuda.current_stream(device).cuda_stream)
    assert within == 0
    assert status == 1
    assert "being captured" in message and "before capturing" in message
    assert library.cdll.mops_amd_scratch_capacity() == capacity  # untouched
    graph.replay()
    torch.cuda.synchronize()
    assert float(marker[0]) == 1.0


def test_a_block_that_a_graph_names_outlives_a_later_growth(device):
    """Eager calls with larger shapes after a capture must not free the block the graph uses."""
    from mops_amd._c_lib import device_library

    library = device_library()
    library.cdll.mops_amd_scratch_capacity.restype = ctypes.c_int64
    library.cdll.mops_amd_reserve_scratch.argtypes = [ctypes.c_int64]
    op = "opsa_pooling"  # pieces of long segments meet in scratch memory
    case = support.to_device(CASES[op](np.float32), device)
    eager = [t.clone() for t in _call(op, case)]
    torch.cuda.synchronize()
    stream = torch.cuda.Stream(device=device)
    stream.wait_stream(torch.cuda.current_stream(device))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        _call(op, case)
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            captured = _call(op, case)
    torch.cuda.synchronize()
    library.cdll.mops_amd_set_stream(torch.cuda.current_stream(device).cuda_stream)
    before = library.cdll.mops_amd_scratch_capacity()
    assert library.cdll.mops_amd_reserve_scratch(8 * before) == 0  # grows: the old block is kept
    assert library.cdll.mops_amd_scratch_capacity() >= 8 * before
    filler = torch.full((before // 4,), float("nan"), device=device)  # would land in a freed block
    for tensor in captured:
        tensor.fill_(float("nan"))
    torch.cuda.synchronize()
    graph.replay()
    torch.cuda.synchronize()
    for got, want in zip(captured, eager):
        assert torch.equal(got, want)
    del filler


@pytest.mark.parametrize(
    "op,point",
    [
        ("opsaw_many_senders", "opsaw_vjp_after_listing"),
        ("sasaw_many_senders_by_arrival", "sasaw_vjp_after_listing"),
        ("sasaw_many_senders", "sasaw_vjp_after_listing"),  # (without counters: nothing is left behind)
    ],
)
def test_a_call_that_fails_between_two_launches_does_not_spoil_the_next(device, monkeypatch, op, point):
    """The senders' edges of large graphs are listed by a launch that counts in counters which the
    launch that uses the lists sets back to zero. A call that fails on the host between the two
    leaves counts behind; the library marks its counters on the host and clears them at the start
    of the next call. The failure is requested from the host (MOPS_AMD_TEST_FAIL_AT): every
    kernel that was enqueued runs to its end."""
    from mops_amd.status import MopsError

    case = support.to_device(CASES[op](np.float32), device)
    good = [t.clone() for t in _call(op, case)]
    torch.cuda.synchronize()
    monkeypatch.setenv("MOPS_AMD_TEST_FAIL_AT", point)
    with pytest.raises(MopsError, match="failure requested by MOPS_AMD_TEST_FAIL_AT"):
        _call(op, case)
    torch.cuda.synchronize()
    monkeypatch.delenv("MOPS_AMD_TEST_FAIL_AT")
    for attempt in range(2):
        again = _call(op, case)
        torch.cuda.synchronize()
        for got, want in zip(again, good):
            assert torch.equal(got, want), (op, attempt)


def test_another_stream_waits_for_a_call_on_the_default_stream(device):
    """Nothing is recorded behind a call on the default stream; a call on another stream that takes the
    same scratch block over records there first and waits. Both streams are the library's business
    alone here: no wait is enqueued by PyTorch, and its streams do not wait for the default one by
    themselves. The call on the default stream sits behind work that takes some milliseconds."""
    from mops_amd._c_lib import device_library

    library = device_library()
    case = support.to_device(CASES["opsaw"](np.float32), device)
    expected = [t.clone() for t in _call("opsaw", case)]
    side = torch.cuda.Stream(device=device)
    busy = torch.randn((4096, 4096), device=device)
    default = torch.cuda.default_stream(device)
    assert default.cuda_stream == 0
    with torch.cuda.stream(side):  # (memory of that stream, so that the call below allocates none)
        _call("opsaw", case)
    torch.cuda.synchronize()
    first = second = None
    with torch.cuda.stream(default):
        for _ in range(20):
            busy = (busy @ busy).clamp(-1.0, 1.0)
        first = _call("opsaw", case)
        behind = torch.cuda.Event()
        behind.record(default)
    with torch.cuda.stream(side):
        second = _call("opsaw", case)
        done = torch.cuda.Event()
        done.record(side)
    assert not behind.query(), "the work on the default stream ended before the other call was enqueued"
    done.synchronize()
    assert behind.query(), "the call on the other stream did not wait for the one on the default stream"
    torch.cuda.synchronize()
    for got, again, want in zip(first, second, expected):
        assert torch.equal(got, want) and torch.equal(again, want)
    support._bind_stream(library, device)


FIRST_CALLS_CAPTURED = """
import ctypes, sys
import numpy as np
import torch
from tests import support
from mops_amd._c_lib import device_library

device = torch.device("cuda:0")
library = device_library()
library.cdll.mops_amd_scratch_capacity.restype = ctypes.c_int64
hpe, sap = support.hpe_case, support.sap_case
CASES = {  # shapes whose kernels need scratch memory; others serve them without
    "hpe_shares_of_the_monomials": (0, "hpe", np.float32, hpe(1, np.float32, I=100, nA=20, J=2100, K=1)),
    "hpe_long_table": (0, "hpe", np.float64, hpe(2, np.float64, I=700, nA=30, J=20000, K=3)),
    "hpe_gradients": (1, "hpe", np.float32, hpe(3, np.float32, I=1200, nA=40, J=3000, K=3)),
    "hpe_gradients_by_rows": (1, "hpe", np.float64, hpe(4, np.float64, I=10001, nA=12, J=50, K=3)),
    "hpe_second": (2, "hpe", np.float64, hpe(5, np.float64, I=1700, nA=40, J=5000, K=3)),
    "sap_forward": (0, "sap", np.float64, sap(6, np.float64, I=300001, nA=13, nB=7, K=900, nO=20)),
    "sap_gradients": (1, "sap", np.float32, sap(7, np.float32, I=100001, nA=13, nB=7, K=900, nO=20)),
}

def call(level, op, case):
    library.cdll.mops_amd_set_stream(ctypes.c_void_p(torch.cuda.current_stream(device).cuda_stream))
    library.cdll.mops_amd_set_synchronous(0)
    spec = support.OPS[op]
    inputs = [case[name] for name in spec.inputs]
    if level == 0:
        shape = (case["A"].shape[0],) + ((case["output_size"],) if "output_size" in case else ())
        outputs = {"output": torch.full(shape, float("nan"), dtype=case["A"].dtype, device=device)}
        library.call(spec.function, outputs["output"], *inputs)
    elif level == 1:
        outputs = {name: torch.full_like(case[name], float("nan")) for name in spec.differentiable}
        library.call(spec.function + "_vjp", *outputs.values(), case["grad_output"], *inputs)
    else:
        outputs, arguments = support._vjp_vjp_arguments(spec, case, None, None, lambda x: torch.full_like(x, float("nan")))
        library.call(spec.function + "_vjp_vjp", *arguments)
    return outputs

stream = torch.cuda.Stream(device=device)
on_device = {
    name: support.to_device(support.add_cotangents(case, op) if level == 2 else case, device)
    for name, (level, op, _, case) in CASES.items()
}
torch.cuda.synchronize()
captured = {}
for name, (level, op, dtype, _) in CASES.items():
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream), torch.cuda.graph(graph, stream=stream):
        captured[name] = graph, call(level, op, on_device[name])
    assert library.cdll.mops_amd_scratch_capacity() == 0, name
torch.cuda.synchronize()
for name, (level, op, dtype, _) in CASES.items():
    graph, got = captured[name]
    with torch.cuda.stream(stream):
        want = call(level, op, on_device[name])  # (eager: with scratch memory)
        stream.synchronize()
        for replay in range(2):
            for tensor in got.values():
                tensor.fill_(float("nan"))
            graph.replay()
            stream.synchronize()
            for key in want:
                support.assert_close(got[key].cpu().numpy(), want[key].cpu().numpy(), dtype, f"{name} {key}")
    print("ok", name, flush=True)
assert library.cdll.mops_amd_scratch_capacity() > 0
"""


def test_calls_captured_before_any_eager_call(device):
    """A thread that has no scratch memory yet and whose stream is being captured gets none: shapes that
    have kernels without scratch memory take those. In a process of its own, where nothing ran before."""
    import os
    import subprocess
    import sys

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    done = subprocess.run([sys.executable, "-c", FIRST_CALLS_CAPTURED], cwd=root, capture_output=True, text=True, timeout=100)
    assert done.returncode == 0, done.stdout + done.stderr[-3000:]
    assert done.stdout.count("ok ") == 7, done.stdout
