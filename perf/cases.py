"""The work whose speed is tracked: calls of the five operations as programs make them.

A case is one pass of a program through the public entry points, on tensors that are already on
the GPU. ``op`` names the operation (hpe, sap, opsa, opsaw, sasaw) and ``mode`` what is asked of it:

* ``forward``: the operation alone, as in inference (``torch.ops.mops.*`` under ``no_grad``, or the
  function of the ``mops_amd`` package);
* ``gradients``: forward pass and gradients with respect to every differentiable input
  (``torch.autograd`` through ``torch.ops.mops.*``, or the ``mops_amd`` functions with ``_vjp``);
* ``second``: forward pass, gradients, and the derivatives of those gradients with respect to
  everything they depend on: a model that is fitted to the derivative of its output (forces).

``api`` is ``torch`` (the PyTorch operators) or ``array`` (the functions of ``mops_amd``).
"""
import math

import torch

import mops_amd
import mops_amd.torch  # noqa: F401  (registers torch.ops.mops.*)

DTYPES = {"float32": torch.float32, "float64": torch.float64}
DIFFERENTIABLE = {"hpe": "A", "sap": "AB", "opsa": "AB", "opsaw": "ABW", "sasaw": "ABW"}
FUNCTIONS = {
    "hpe": "homogeneous_polynomial_evaluation",
    "sap": "sparse_accumulation_of_products",
    "opsa": "outer_product_scatter_add",
    "opsaw": "outer_product_scatter_add_with_weights",
    "sasaw": "sparse_accumulation_scatter_add_with_weights",
}


def _hpe(rows, features, monomials, order):
    return {"op": "hpe", "rows": rows, "features": features, "monomials": monomials, "order": order}


def _sap(rows, n_a, n_b, n_out, entries):
    return {"op": "sap", "rows": rows, "n_a": n_a, "n_b": n_b, "n_out": n_out, "entries": entries}


def _opsa(edges, nodes, k, l):
    return {"op": "opsa", "edges": edges, "nodes": nodes, "k": k, "l": l}


def _opsaw(edges, nodes, k, l):
    return {"op": "opsaw", "edges": edges, "nodes": nodes, "k": k, "l": l}


def _sasaw(edges, nodes, n_a, n_w, n_out, entries, l):
    return {
        "op": "sasaw", "edges": edges, "nodes": nodes, "n_a": n_a, "n_w": n_w, "n_out": n_out, "entries": entries, "l": l,
    }  # fmt: skip


def listed():
    def case(name, api, mode, dtype, sizes):
        return {"name": name, "api": api, "mode": mode, "dtype": dtype, **sizes}

    return [
        # one small structure, one polynomial of its features: nothing but the cost of a call
        case("hpe_one_structure", "array", "forward", "float64", _hpe(100, 10, 50, 3)),
        # a batch of 1000 atoms in training
        case("hpe_batch", "torch", "gradients", "float64", _hpe(1000, 100, 2000, 4)),
        # a large basis: thousands of features, a polynomial of a hundred thousand monomials
        case("hpe_large_basis", "torch", "gradients", "float32", _hpe(1000, 2000, 100000, 4)),
        # a layer of tensor products in training
        case("sap_batch", "torch", "gradients", "float32", _sap(32000, 13, 7, 20, 900)),
        # the same over a large data set in double, by the functions without autograd
        case("sap_dataset", "array", "gradients", "float64", _sap(1000000, 13, 7, 20, 900)),
        # descriptors fitted to forces: second derivatives, ragged sizes
        case("opsa_forces", "torch", "second", "float32", _opsa(51237, 1711, 13, 33)),
        # descriptors of a large structure, inference in double
        case("opsa_large_inference", "torch", "forward", "float64", _opsa(1000000, 33000, 13, 20)),
        # one layer of message passing in training, a batch of structures and a large one
        case("opsaw_batch", "torch", "gradients", "float32", _opsaw(60000, 2000, 13, 32)),
        case("opsaw_large", "torch", "gradients", "float32", _opsaw(1000000, 33000, 13, 32)),
        # one equivariant layer: a single small structure, a batch in double, a large structure
        case("sasaw_one_structure", "torch", "gradients", "float32", _sasaw(600, 20, 9, 9, 9, 250, 32)),
        case("sasaw_batch", "torch", "gradients", "float64", _sasaw(60000, 2000, 9, 9, 9, 250, 32)),
        case("sasaw_large", "torch", "gradients", "float32", _sasaw(1000000, 33000, 9, 9, 9, 250, 32)),
    ]


def draw(rng):
    """A case of the ranges between the listed ones: from a single structure to about a million
    rows or edges, any number of features between the smallest and the largest in use."""

    def spread(low, high):
        return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))

    def bounded(low, high, per_row, most):
        return spread(low, max(low, min(high, int(most // per_row))))

    op = rng.choice(list(FUNCTIONS))
    mode = rng.choice(["forward", "gradients", "gradients", "second"] if op in ("hpe", "sap", "opsa") else ["forward", "gradients"])
    share = 0.25 if mode == "second" else 1.0  # its four calls do several times a forward pass's work
    if op == "hpe":
        features, monomials, order = spread(10, 2000), spread(50, 100000), rng.randint(2, 4)
        sizes = _hpe(bounded(64, 100000, monomials * (order + 1), share * 2e8), features, monomials, order)
    elif op == "sap":
        # components of both operands up to l = 3, or a radial and an angular index
        n_a, n_b, n_out = rng.randint(3, 16), rng.randint(3, 16), spread(4, 100)
        entries = min(spread(30, 1500), n_a * n_b * n_out)
        sizes = _sap(bounded(100, 1000000, n_a + n_b + n_out + entries / 8, share * 1.5e8), n_a, n_b, n_out, entries)
    elif op in ("opsa", "opsaw"):
        k, l = rng.randint(4, 32), spread(8, 64)
        edges = bounded(300, 1000000, k * l, share * 4e8)
        sizes = (_opsa if op == "opsa" else _opsaw)(edges, max(8, edges // rng.randint(10, 60)), k, l)
    else:
        n = rng.choice([4, 9, 16])  # components of everything up to l = 1, 2, 3
        entries = {4: 24, 9: 250, 16: 800}[n]
        l = spread(8, 128)
        edges = bounded(300, 1000000, n * n * l, 1.5e9)
        sizes = _sasaw(edges, max(8, edges // rng.randint(10, 60)), n, n, n, entries, l)
    api = rng.choice(["torch", "torch", "array"])
    return {"api": api, "mode": mode, "dtype": rng.choice(["float32", "float64"]), **sizes}


# ------------------------------------------------------------------ inputs --
def _output_shape(case):
    if case["op"] == "hpe":
        return (case["rows"],)
    if case["op"] == "sap":
        return (case["rows"], case["n_out"])
    if case["op"] == "sasaw":
        return (case["nodes"], case["n_out"], case["l"])
    return (case["nodes"], case["k"], case["l"])


def _shapes(case):
    """Shapes of the floating-point inputs."""
    op = case["op"]
    if op == "hpe":
        return {"A": (case["rows"], case["features"]), "C": (case["monomials"],)}
    if op == "sap":
        return {"A": (case["rows"], case["n_a"]), "B": (case["rows"], case["n_b"]), "C": (case["entries"],)}
    if op == "sasaw":
        return {
            "A": (case["edges"], case["n_a"]), "B": (case["edges"], case["l"]), "C": (case["entries"],),
            "W": (case["nodes"], case["n_w"], case["l"]),
        }  # fmt: skip
    shapes = {"A": (case["edges"], case["k"]), "B": (case["edges"], case["l"])}
    if op == "opsaw":
        shapes["W"] = (case["nodes"], case["l"])
    return shapes


def _integers(case):
    """(length or shape, number of values, sorted) of the index tensors, in the order of the arguments."""
    op = case["op"]
    if op == "hpe":
        return [((case["monomials"], case["order"]), case["features"], False)]
    if op == "sap":
        n = (case["entries"],)
        return [(n, case["n_a"], False), (n, case["n_b"], False), (n, case["n_out"], True)]
    edges, nodes = (case["edges"],), case["nodes"]
    if op == "opsa":
        return [(edges, nodes, True)]
    if op == "opsaw":
        return [(edges, nodes, False), (edges, nodes, True)]
    n = (case["entries"],)
    return [(n, case["n_a"], False), (edges, nodes, False), (n, case["n_w"], False), (edges, nodes, True), (n, case["n_out"], False)]


def prepare(case, seed):
    generator = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]]

    def normal(shape):
        return torch.randn(shape, generator=generator, device="cuda", dtype=dtype)

    def integers(shape, values, is_sorted):
        drawn = torch.randint(0, values, shape, generator=generator, device="cuda", dtype=torch.int32)
        return drawn.sort().values if is_sorted else drawn

    op = case["op"]
    floats = {name: normal(shape) for name, shape in _shapes(case).items()}
    if op == "hpe":
        floats["A"] = floats["A"].clamp(-1.0, 1.0)  # features are normalised
    indices = [integers(*what) for what in _integers(case)]
    size = {"sap": case.get("n_out"), "opsa": case.get("nodes"), "sasaw": case.get("n_out")}.get(op)
    wanted = [floats[name] for name in DIFFERENTIABLE[op]]
    state = {
        "case": case,
        "arguments": [*floats.values(), *indices, *([] if size is None else [size])],
        "wanted": wanted,
        "forward": getattr(mops_amd if case["api"] == "array" else torch.ops.mops, FUNCTIONS[op]),
    }
    if case["mode"] != "forward":
        state["grad_output"] = normal(_output_shape(case))
        if case["api"] == "torch":
            for tensor in wanted:
                tensor.requires_grad_()
    if case["mode"] == "second":
        state["grad_grads"] = [normal(tensor.shape) for tensor in wanted]
        if case["api"] == "torch":
            state["grad_output"].requires_grad_()
    if case["api"] == "array":
        state["vjp"] = getattr(mops_amd, FUNCTIONS[op] + "_vjp")
        state["vjp_vjp"] = getattr(mops_amd, FUNCTIONS[op] + "_vjp_vjp")
    return state


# -------------------------------------------------------------------- pass --
def _run_array(state):
    case, arguments = state["case"], state["arguments"]
    # (the derivatives take the size of the output from grad_output)
    inputs = arguments[:-1] if isinstance(arguments[-1], int) else arguments
    outputs = [state["forward"](*arguments)]
    if case["mode"] != "forward":
        gradients = state["vjp"](state["grad_output"], *inputs)
        outputs += [gradients] if isinstance(gradients, torch.Tensor) else list(gradients)
    if case["mode"] == "second":
        outputs += state["vjp_vjp"](*state["grad_grads"], state["grad_output"], *inputs)
    return outputs


def _run_torch(state):
    case, wanted = state["case"], state["wanted"]
    if case["mode"] == "forward":
        with torch.no_grad():
            return [state["forward"](*state["arguments"])]
    second = case["mode"] == "second"
    output = state["forward"](*state["arguments"])
    gradients = torch.autograd.grad(output, wanted, state["grad_output"], create_graph=second)
    outputs = [output, *gradients]
    if second:
        outputs += torch.autograd.grad(gradients, [state["grad_output"], *wanted], state["grad_grads"])
    return [tensor.detach() for tensor in outputs]


def run(state):
    return _run_array(state) if state["case"]["api"] == "array" else _run_torch(state)


# ------------------------------------------------------------ requirements --
def _flops(case):
    """Operations of the forward pass, and of the gradients, in the cheapest formulation known."""
    op = case["op"]
    if op == "hpe":
        terms, order = case["rows"] * case["monomials"], case["order"]
        return terms * (order + 1), terms * 4 * order  # prefix and suffix products
    if op == "sap":
        terms = case["rows"] * case["entries"]
        return 3 * terms, 5 * terms
    if op == "sasaw":
        # the sum over the edges before the table: once for the output, once per gradient
        contraction = 2 * case["edges"] * case["n_a"] * case["n_w"] * case["l"]
        table = 2 * case["nodes"] * case["entries"] * case["l"]
        scaling = case["edges"] * case["n_w"] * case["l"]
        return contraction + scaling + table, 3 * contraction + 4 * scaling + 2 * table
    product = 2 * case["edges"] * case["k"] * case["l"]
    scaling = case["edges"] * case["l"] if op == "opsaw" else 0
    return product + scaling, 2 * product + 3 * scaling


def work(case):
    size = 4 if case["dtype"] == "float32" else 8
    shapes = _shapes(case)
    floats = sum(math.prod(shape) for shape in shapes.values())
    integers = sum(math.prod(shape) for shape, _, _ in _integers(case))
    output = math.prod(_output_shape(case))
    wanted = sum(math.prod(shapes[name]) for name in DIFFERENTIABLE[case["op"]])
    forward, gradients = _flops(case)
    flops, values = forward, floats + output
    if case["mode"] != "forward":
        flops, values = flops + gradients, values + output + wanted
    if case["mode"] == "second":
        # both directional derivatives of the output, and gradients along both cotangents
        flops, values = flops + 2 * forward + gradients, values + wanted + output + wanted
    return {"bytes": values * size + integers * 4, "flops": flops}


def tolerance(case):
    return {"rel": 1e-5} if case["dtype"] == "float32" else {"rel": 1e-12}
