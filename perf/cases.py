"""Performance cases of the framework: what its users run, through its public entry points.

Nine kinds of call (``op``), over the sizes of the repository's benchmark, tests and model:

* ``tp``          ``EdgeTensorProduct``: the channelwise tensor product on per-edge instances,
                  forward and gradients to features, harmonics and gates;
* ``message``     ``PackedGraphMessage`` on a periodic radius graph: forward (``order`` 0), with its
                  gradients (1), or with the mixed second derivatives of force training (2);
* ``contraction`` ``create_symmetric_contraction``: the node-wise contraction, forward, and the
                  gradients to features and weights (training);
* ``gates``       an interaction's radial network up to the message gates, forward and the gradients
                  to the edge features (forces) and to its weights (training);
* ``linear``      an interaction's message linear: forward and the gradients to input and weights;
* ``neighbors``   ``radius_graph_pbc_gpu``: the periodic neighbour list;
* ``energy``      ``energy_and_forces`` of a frozen model on new positions (structure relaxation,
                  batched evaluation);
* ``replay``      ``CapturedEnergyAndForces``: the same step captured once and replayed on new
                  positions (molecular dynamics on a fixed neighbour list);
* ``training``    energies and forces with a recorded graph, the force loss and its gradients to
                  every parameter.

Everything is float32, as the library computes.  ``exact`` restates each call in plain float64
torch; only constants (coupling tensors, harmonic polynomials, a model's parameters and U
buffers) are read from the package.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ictc-o3-hp-ascend_amd"))

import ictc_o3  # noqa: E402
import mace_hip  # noqa: E402
from ictc_o3.basis.ictd_irreps import element_path_scales, harmonics_tables, normalised_coupling, triangle_paths  # noqa: E402
from mace_hip.model import Interaction  # noqa: E402
from mace_hip.runtime import backward_to_parameters  # noqa: E402

DENSITY, CUTOFF, ELEMENTS, BASIS, HIDDEN, CUTOFF_P = 0.1, 5.0, 10, 8, 64, 5
NEIGHBORS = DENSITY * 4.0 / 3.0 * math.pi * CUTOFF ** 3          # 52.4 per atom
SILU_SCALE = 1.6791767923989418


def listed():
    return [
        # one tensor product of a small molecule's edges: launches and host work
        {"name": "tp_small_c64_l2", "op": "tp", "channels": 64, "input_lmax": 2, "edge_lmax": 2, "output_lmax": 2,
         "rows": 500, "layout": "ir_mul", "grad": True},
        # the headline tensor product workload: 131,072 instances, forward and gradients
        {"name": "tp_c128_l3", "op": "tp", "channels": 128, "input_lmax": 3, "edge_lmax": 3, "output_lmax": 3,
         "rows": 131072, "layout": "ir_mul", "grad": True},
        # a degree-4 product on a ragged number of edges
        {"name": "tp_c64_l4", "op": "tp", "channels": 64, "input_lmax": 4, "edge_lmax": 4, "output_lmax": 4,
         "rows": 20011, "layout": "ir_mul", "grad": True},
        # a large structure's message with its gradients (energies and forces of a small model)
        {"name": "message_c64_l2", "op": "message", "channels": 64, "input_lmax": 2, "lmax": 2, "atoms": 16384,
         "order": 1},
        # the second interaction's message in force training, with its second derivatives
        {"name": "message_c128_l3_force", "op": "message", "channels": 128, "input_lmax": 3, "lmax": 3, "atoms": 2048,
         "order": 2},
        # the product block's contraction in training, an odd number of nodes
        {"name": "contraction_c128_l3", "op": "contraction", "channels": 128, "lmax": 3, "target_lmax": 1,
         "correlation": 3, "nodes": 16411, "grad": True},
        # the second interaction's gates in training (edges of 2,048 atoms)
        {"name": "gates_c128_l3", "op": "gates", "channels": 128, "input_lmax": 3, "lmax": 3, "edges": 105634,
         "train": True},
        # the second interaction's message linear in training
        {"name": "message_linear_c128_l3", "op": "linear", "channels": 128, "input_lmax": 3, "lmax": 3, "atoms": 2048,
         "train": True},
        # the neighbour list of an ordinary structure, rebuilt as its atoms move
        {"name": "neighbors_4096", "op": "neighbors", "atoms": 4096, "density": 0.1, "cutoff": 5.0},
        # a small molecule or unit cell evaluated eagerly: launches and host work
        {"name": "energy_small_c64_l2", "op": "energy", "channels": 64, "lmax": 2, "atoms": 150, "structures": 1},
        # the headline model step: energies and forces of 2,048 atoms
        {"name": "replay_c128_l3", "op": "replay", "channels": 128, "lmax": 3, "atoms": 2048, "structures": 1},
        # the headline training step, as a batch of four structures
        {"name": "training_c128_l3", "op": "training", "channels": 128, "lmax": 3, "atoms": 512, "structures": 4},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    op = rng.choice(["tp", "tp", "message", "message", "contraction", "gates", "linear", "neighbors", "energy",
                     "replay", "training"])
    channels = rng.choice([24, 32, 48, 64, 96, 128])
    lmax = rng.choice([1, 2, 3])
    if op == "tp":
        lmax = rng.choice([1, 2, 3, 4])
        edge, out = rng.choice([lmax, lmax, max(lmax - 1, 1)]), rng.choice([lmax, lmax, lmax - 1])
        width = sum(2 * c + 2 for _, _, c in triangle_paths(lmax, edge, out))
        most = 131072 * 128 * 122 // (channels * width) // (4 if lmax == 4 else 1)
        return {"op": op, "channels": channels, "input_lmax": lmax, "edge_lmax": edge, "output_lmax": out,
                "rows": _log(rng, 100, min(most, 131072)), "layout": rng.choice(["ir_mul", "ir_mul", "mul_ir"]),
                "grad": rng.random() < 0.7}
    if op == "message":
        input_lmax = rng.choice([0, lmax, lmax])
        paths = len(triangle_paths(input_lmax, lmax, lmax))
        most = min(16384, 2048 * 23 * 128 // (paths * channels))
        return {"op": op, "channels": channels, "input_lmax": input_lmax, "lmax": lmax, "atoms": _log(rng, 60, most),
                "order": rng.choice([0, 1, 2])}
    if op == "contraction":
        return {"op": op, "channels": channels, "lmax": lmax, "target_lmax": rng.randint(0, lmax),
                "correlation": rng.choice([2, 3, 3]), "nodes": _log(rng, 100, 16000 if lmax < 3 else 5000),
                "grad": rng.random() < 0.6}
    if op == "gates":
        return {"op": op, "channels": channels, "input_lmax": rng.choice([0, lmax, lmax]), "lmax": lmax,
                "edges": _log(rng, 1500, 105000), "train": rng.random() < 0.5}
    if op == "linear":
        return {"op": op, "channels": channels, "input_lmax": rng.choice([0, lmax, lmax]), "lmax": lmax,
                "atoms": _log(rng, 60, 8000 if lmax < 3 else 2048), "train": rng.random() < 0.5}
    if op == "neighbors":
        return {"op": op, "atoms": _log(rng, 100, 16384), "density": rng.choice([0.05, 0.08, 0.1]),
                "cutoff": rng.choice([4.0, 5.0, 6.0])}
    structures = rng.choice([1, 1, 2, 5])
    most = 2048 if op != "training" else 1024
    return {"op": op, "channels": channels, "lmax": lmax, "atoms": max(30, _log(rng, 40, most) // structures),
            "structures": structures}


# ------------------------------------------------------------------------------------ inputs
def _gen(seed, device):
    return torch.Generator(device=device).manual_seed(int(seed) * 7919 + 13)


def _atoms(gen, n, density, device, which=0):
    """Positions in a cubic cell: a random choice of the sites of a cubic lattice, displaced by up
    to a fifth of its spacing (a dense disordered solid without overlapping atoms).  The structure
    follows from its size, so that its number of edges does; the order of its atoms and its axes
    from the seed."""
    edge = (n / density) ** (1.0 / 3.0)
    m = math.ceil(n ** (1.0 / 3.0) - 1e-9)
    own = _gen(n * 16 + which, device)
    site = torch.randperm(m ** 3, generator=own, device=device)[:n]
    grid = torch.stack([site // (m * m), site // m % m, site % m], 1).double()
    move = torch.rand(n, 3, generator=own, device=device, dtype=torch.float64) * 0.4 - 0.2
    pos = ((grid + 0.5 + move) * (edge / m)).float()
    order, axes = (torch.randperm(k, generator=gen, device=device) for k in (n, 3))
    return pos[order][:, axes].contiguous(), torch.eye(3, device=device) * edge


def _directions(gen, rows, device):
    return torch.nn.functional.normalize(torch.randn(rows, 3, generator=gen, device=device), dim=-1)


def _harmonics(directions, lmax):
    return torch.cat(ictc_o3.direction_harmonics(directions, lmax), -1).contiguous()


def _edge_features(gen, edges, device):
    """Bessel functions times the cutoff envelope at distances spread over a ball's volume."""
    r = CUTOFF * (0.03 + 0.97 * torch.rand(edges, generator=gen, device=device, dtype=torch.float64)) ** (1.0 / 3.0)
    return _radial64(r).float()


def _interaction(case, gen_seed, device):
    torch.manual_seed(int(gen_seed))
    return Interaction(channels=case["channels"], input_lmax=case["input_lmax"], edge_lmax=case["lmax"],
                       num_elements=ELEMENTS, num_basis=BASIS, avg_num_neighbors=NEIGHBORS).to(device)


def _model_inputs(case, seed, device):
    gen = _gen(seed, device)
    model = mace_hip.create_model(channels=case["channels"], lmax=case["lmax"], num_interactions=2, correlation=3,
                                  atomic_numbers=tuple(range(1, ELEMENTS + 1)), cutoff=CUTOFF,
                                  avg_num_neighbors=NEIGHBORS, device=device, seed=int(seed))
    parts, cells, count = [], [], case["atoms"]
    for b in range(case["structures"]):
        pos, cell = _atoms(gen, count, DENSITY, device, b)
        src, dst, shift = mace_hip.radius_graph_pbc_gpu(pos, CUTOFF, cell)
        parts.append((pos, src + b * count, dst + b * count, shift.float()))
        cells.append(cell)
    pos, src, dst, shift = (torch.cat(v).contiguous() for v in zip(*parts))
    species = torch.randint(0, ELEMENTS, (pos.shape[0],), generator=gen, device=device)
    graph = {"positions": pos, "atomic_numbers": species + 1,
             "batch": torch.arange(case["structures"], device=device).repeat_interleave(count),
             "edge_src": src, "edge_dst": dst, "edge_shifts": shift, "cell": torch.stack(cells)}
    return model, graph, species


def prepare(case, seed):
    device = torch.device("cuda", 0)
    gen, op = _gen(seed, device), case["op"]

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device=device)

    if op == "tp":
        c, rows = case["channels"], case["rows"]
        tp = ictc_o3.EdgeTensorProduct.create(channels=c, input_lmax=case["input_lmax"], edge_lmax=case["edge_lmax"],
                                              output_lmax=case["output_lmax"], layout=case["layout"], device=device)
        x = normal(rows, c * (case["input_lmax"] + 1) ** 2)
        y = _harmonics(_directions(gen, rows, device), case["edge_lmax"])
        g = normal(rows, tp.gate_width) / math.sqrt(len(tp.paths))
        state = {"op": op, "call": tp, "inputs": (x, y, g)}
        if case["grad"]:
            state["go"] = normal(rows, tp.output_width)
            for t in (x, y, g):
                t.requires_grad_()
        return state
    if op == "message":
        c, n = case["channels"], case["atoms"]
        call = ictc_o3.PackedGraphMessage.create(channels=c, input_lmax=case["input_lmax"], edge_lmax=case["lmax"],
                                                 output_lmax=case["lmax"], device=device)
        pos, cell = _atoms(gen, n, DENSITY, device)
        src, dst, shift = mace_hip.radius_graph_pbc_gpu(pos, CUTOFF, cell)
        vec = pos.double()[dst] - pos.double()[src] + shift @ cell.double()
        y = _harmonics(torch.nn.functional.normalize(vec, dim=-1).float(), case["lmax"])
        x = normal(n, c * (case["input_lmax"] + 1) ** 2)
        g = normal(src.numel(), call.gate_width) / math.sqrt(len(call.paths))
        state = {"op": op, "call": call, "inputs": (x, y, g), "src": src, "dst": dst, "order": case["order"]}
        if case["order"]:
            state["go"] = normal(n, call.output_width)
            for t in (x, y, g):
                t.requires_grad_()
        if case["order"] == 2:
            state["go"].requires_grad_()
            state["cotangents"] = (normal(*state["go"].shape), normal(*x.shape), normal(*y.shape), normal(*g.shape))
        return state
    if op == "contraction":
        torch.manual_seed(int(seed))
        call = ictc_o3.create_symmetric_contraction(num_elements=ELEMENTS, lmax=case["lmax"],
                                                    target_lmax=case["target_lmax"], channels=case["channels"],
                                                    correlation=case["correlation"], device=device)
        x = normal(case["nodes"], case["channels"] * (case["lmax"] + 1) ** 2)
        species = torch.randint(0, ELEMENTS, (case["nodes"],), generator=gen, device=device)
        state = {"op": op, "call": call, "inputs": (x,), "species": species}
        if case["grad"]:
            x.requires_grad_()
            state["go"] = normal(case["nodes"], case["channels"] * (case["target_lmax"] + 1) ** 2)
        else:
            call.requires_grad_(False)
        return state
    if op in ("gates", "linear"):
        call = _interaction(case, seed, device)
        if not case["train"]:
            call.requires_grad_(False)
        if op == "gates":
            x = _edge_features(gen, case["edges"], device)
            go = normal(case["edges"], call.tp.num_paths * case["channels"])
        else:
            x = normal(case["atoms"], call.message_linear.plan.in_width)
            go = normal(case["atoms"], call.message_linear.plan.out_width)
        return {"op": op, "call": call, "inputs": (x.requires_grad_(),), "go": go}
    if op == "neighbors":
        pos, cell = _atoms(gen, case["atoms"], case["density"], device)
        return {"op": op, "inputs": (pos, case["cutoff"], cell)}
    model, graph, species = _model_inputs(case, seed, device)
    state = {"op": op, "call": model, "graph": graph, "species": species}
    if op != "training":
        model.eval().requires_grad_(False)
    if op == "replay":
        state["call"] = mace_hip.CapturedEnergyAndForces(model, **graph, species=species)
        noise = torch.randn(graph["positions"].shape, generator=gen, device=device)
        state["positions"] = graph["positions"] + 0.01 * noise
    return state


# -------------------------------------------------------------------------------------- passes
def run(state):
    op, call = state["op"], state.get("call")
    if op == "tp":
        out = call(*state["inputs"])
        return [out] if "go" not in state else [out.detach(), *torch.autograd.grad(out, state["inputs"], state["go"])]
    if op == "message":
        x, y, g = state["inputs"]
        out = call(x, y, g, state["src"], state["dst"])
        if state["order"] == 0:
            return [out]
        if state["order"] == 1:
            return [out.detach(), *torch.autograd.grad(out, (x, y, g), state["go"])]
        grads = torch.autograd.grad(out, (x, y, g), state["go"], create_graph=True)
        second = torch.autograd.grad((out, *grads), (x, g, state["go"]), state["cotangents"])
        return [t.detach() for t in (out, *grads, *second)]
    if op == "contraction":
        out = call(*state["inputs"], node_type_idx=state["species"])
        if "go" not in state:
            return [out]
        return [out.detach(), *torch.autograd.grad(out, (*state["inputs"], *call.parameters()), state["go"])]
    if op in ("gates", "linear"):
        x = state["inputs"][0]
        out = call.message_gates(x) if op == "gates" else call.message_linear(x, 1.0 / call.avg_num_neighbors)
        return [out.detach(), *torch.autograd.grad(out, (x, *_layer_weights(op, call)), state["go"])]
    if op == "neighbors":
        return list(mace_hip.radius_graph_pbc_gpu(*state["inputs"]))
    if op == "energy":
        return mace_hip.energy_and_forces(call, **state["graph"], species=state["species"])
    if op == "replay":
        return call(state["positions"])
    prediction = mace_hip.energy_and_forces(call, **state["graph"], training=True, species=state["species"])
    loss = mace_hip.force_loss(prediction, state["graph"]["positions"].shape[0])
    params = [p for p in call.parameters() if p.requires_grad]
    for p in params:
        p.grad = None
    backward_to_parameters(loss, call, state["graph"]["positions"])
    return [loss.detach(), prediction["energy"].detach(), prediction["forces"].detach(), *(p.grad for p in params)]


def _layer_weights(op, interaction):
    layer = interaction.fc if op == "gates" else interaction.message_linear
    return [p for p in layer.parameters() if p.requires_grad]


# ---------------------------------------------------------------------------------------- work
def _sizes(input_lmax, edge_lmax, output_lmax):
    """(paths, path output components, bond entries, coupling entries) of a full path set."""
    paths = triangle_paths(input_lmax, edge_lmax, output_lmax)
    return (len(paths), sum(2 * c + 1 for _, _, c in paths), sum((2 * a + 1) * (2 * c + 1) for a, _, c in paths),
            sum((2 * a + 1) * (2 * b + 1) * (2 * c + 1) for a, b, c in paths))


def _tp_work(c, lin, le, lout, rows, nodes_in, nodes_out, passes):
    """Bytes and operations of a tensor product over `rows` edges with node-sized or edge-sized
    ends, for `passes` of 1 (forward), 3 (with gradients) or 9 (with second derivatives)."""
    p, o, bonds, cg = _sizes(lin, le, lout)
    x, y = c * (lin + 1) ** 2, (le + 1) ** 2
    ends, edge = nodes_in * x, rows * (y + p * c)
    out = nodes_out * o * c
    forward = 4.0 * (ends + edge + out)
    tensors = {1: forward, 3: forward + 4.0 * (2 * ends + 2 * edge + out),
               9: 4.0 * (ends + edge + out + (ends + edge) + out + 2 * (ends + edge) + out + rows * p * c)}[passes]
    return {"bytes": tensors, "flops": passes * rows * 2.0 * (cg + bonds * c + o * c)}


def _monomials(lmax, order):
    d = (lmax + 1) ** 2
    return {1: d, 2: d * (d + 1) // 2, 3: d * (d + 1) * (d + 2) // 6}[order]


def _contraction_flops(lmax, target, correlation):
    """Per node and channel: each symmetric monomial of the features once, and once into each output
    component (the smallest evaluation that does not use the couplings' structure)."""
    return 2.0 * sum(_monomials(lmax, k) for k in range(1, correlation + 1)) * (1 + (target + 1) ** 2)


def _gates_flops(edges, paths, c):
    return 2.0 * edges * (BASIS * HIDDEN + 2 * HIDDEN * HIDDEN + HIDDEN * paths * c)


def _linear_flops(atoms, out_components, c):
    return 2.0 * atoms * out_components * c * c


def work(case):
    op, c = case["op"], case.get("channels")
    if op == "tp":
        return _tp_work(c, case["input_lmax"], case["edge_lmax"], case["output_lmax"], case["rows"], case["rows"],
                        case["rows"], 3 if case["grad"] else 1)
    if op == "message":
        edges, n = int(case["atoms"] * NEIGHBORS), case["atoms"]
        w = _tp_work(c, case["input_lmax"], case["lmax"], case["lmax"], edges, n, n, (1, 3, 9)[case["order"]])
        return {"bytes": w["bytes"] + 16.0 * edges, "flops": w["flops"]}
    if op == "contraction":
        d, o, n = c * (case["lmax"] + 1) ** 2, c * (case["target_lmax"] + 1) ** 2, case["nodes"]
        flops = n * c * _contraction_flops(case["lmax"], case["target_lmax"], case["correlation"])
        return {"bytes": n * (4.0 * ((d + o) + (d + o if case["grad"] else 0)) + 8),
                "flops": flops * (3 if case["grad"] else 1)}
    if op == "gates":
        e, p = case["edges"], _sizes(case["input_lmax"], case["lmax"], case["lmax"])[0]
        return {"bytes": 4.0 * e * (2 * BASIS + 2 * p * c) + 4.0 * HIDDEN * p * c,
                "flops": _gates_flops(e, p, c) * (3 if case["train"] else 2)}
    if op == "linear":
        n, o = case["atoms"], _sizes(case["input_lmax"], case["lmax"], case["lmax"])[1]
        return {"bytes": 4.0 * n * 2 * (o * c + c * (case["lmax"] + 1) ** 2),
                "flops": _linear_flops(n, o, c) * (3 if case["train"] else 2)}
    if op == "neighbors":
        per_atom = case["density"] * 4.0 / 3.0 * math.pi * case["cutoff"] ** 3
        # each pair within the cells around an atom is tried once, each edge written once
        return {"bytes": case["atoms"] * (12.0 + 40.0 * per_atom),
                "flops": case["atoms"] * 8.0 * 27.0 * case["density"] * case["cutoff"] ** 3}
    n, lmax = case["atoms"] * case["structures"], case["lmax"]
    edges, flops, nbytes = n * NEIGHBORS, 0.0, n * (12.0 + 8 + 8 + 12 + 4) + n * NEIGHBORS * (16 + 12)
    times = 2 if op != "training" else 6
    for lin, target in ((0, lmax), (lmax, 0)):
        p, o, bonds, cg = _sizes(lin, lmax, lmax)
        flops += times * (_gates_flops(edges, p, c) + _linear_flops(n, o + (lin + 1) ** 2 + (target + 1) ** 2 + 1, c)
                          + edges * 2.0 * (cg + bonds * c + o * c) + n * c * _contraction_flops(lmax, target, 3))
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the largest relative error against ``exact`` measured over the listed cases
    and a dozen drawn ones (products 1.6e-7, contraction and linear 5e-7, gates 1.5e-6, forces and
    parameter gradients 1.6e-6)."""
    if case["op"] == "neighbors":
        return "exact"
    rel = {"tp": 8e-7, "message": 8e-7, "contraction": 2e-6, "linear": 2e-6, "gates": 6e-6, "energy": 7e-6,
           "replay": 7e-6, "training": 7e-6}[case["op"]]
    return {"rel": rel, "max": 100 * rel}


# ------------------------------------------------------------------------------ float64 values
def _couplings(paths, device):
    return [torch.from_numpy(normalised_coupling(*p) * s).to(device) for p, s in zip(paths, element_path_scales(paths))]


def _tp64(paths, cgs, c, lmax, x, y, g):
    """[E, C (L+1)^2] ir_mul features, harmonics, gates [E, P C] -> [E, out] (per output degree, per
    path: 2l+1 rows of C)."""
    rows, parts = x.shape[0], {}
    for k, ((l1, l2, l3), cg) in enumerate(zip(paths, cgs)):
        xb = x[:, c * l1 * l1:c * (l1 + 1) ** 2].reshape(rows, 2 * l1 + 1, c)
        bond = y[:, l2 * l2:(l2 + 1) ** 2] @ cg.permute(1, 2, 0).reshape(2 * l2 + 1, -1)
        value = bond.reshape(rows, 2 * l3 + 1, 2 * l1 + 1) @ xb
        parts.setdefault(l3, []).append((value * g[:, None, k * c:(k + 1) * c]).reshape(rows, -1))
    return torch.cat([t for l in range(lmax + 1) for t in parts.get(l, [])], 1)


def _transposed(t, c, counts, to_ir):
    """Rows of per-degree [count][C][2l+1] blocks to [count][2l+1][C] blocks, or back."""
    parts, at = [], 0
    for l, k in enumerate(counts):
        w = k * c * (2 * l + 1)
        shape = (t.shape[0], k, c, 2 * l + 1) if to_ir else (t.shape[0], k, 2 * l + 1, c)
        parts.append(t[:, at:at + w].reshape(shape).transpose(2, 3).reshape(t.shape[0], w))
        at += w
    return torch.cat(parts, 1)


def _exact_tp(case, state):
    c, device = case["channels"], state["inputs"][0].device
    lin, lmax = case["input_lmax"], max(case["input_lmax"], case["edge_lmax"], case["output_lmax"])
    paths = triangle_paths(lin, case["edge_lmax"], case["output_lmax"])
    counts = [sum(p[2] == l for p in paths) for l in range(lmax + 1)]
    cgs, mul = _couplings(paths, device), case["layout"] == "mul_ir"
    outs, step = None, 4096
    for at in range(0, case["rows"], step):
        x, y, g = (t[at:at + step].detach().double().requires_grad_(case["grad"]) for t in state["inputs"])
        out = _tp64(paths, cgs, c, lmax, _transposed(x, c, [1] * (lin + 1), True) if mul else x, y, g)
        out = _transposed(out, c, counts, False) if mul else out
        got = [out.detach()]
        if case["grad"]:
            got += torch.autograd.grad(out, (x, y, g), state["go"][at:at + step].double())
        if outs is None:
            outs = [torch.empty(case["rows"], t.shape[1], dtype=torch.float64, device=device) for t in got]
        for o, t in zip(outs, got):
            o[at:at + step] = t
    return outs


def _exact_message(case, state):
    c, order, device = case["channels"], case["order"], state["src"].device
    paths = triangle_paths(case["input_lmax"], case["lmax"], case["lmax"])
    cgs = _couplings(paths, device)
    src, dst = state["src"], state["dst"]
    nodes = state["inputs"][0].shape[0]
    x, y, g = (t.detach().double() for t in state["inputs"])
    go = state["go"].detach().double() if order else None
    cot = [t.double() for t in state["cotangents"]] if order == 2 else None
    out = dx = dy = dg = ggo = gx = gg = None
    dy, dg, gg = (torch.empty_like(t) if order else None for t in (y, g, g))
    step = 8192
    for at in range(0, src.numel(), step):
        s, d = src[at:at + step], dst[at:at + step]
        leaves = [t.requires_grad_(order > 0) for t in (x.detach(), y[at:at + step].clone(), g[at:at + step].clone())]
        value = _tp64(paths, cgs, c, case["lmax"], leaves[0].index_select(0, s), leaves[1], leaves[2])
        part = torch.zeros(nodes, value.shape[1], dtype=torch.float64, device=device).index_add(0, d, value)
        out = part.detach() if out is None else out.add_(part.detach())
        if not order:
            continue
        gl = go.detach().requires_grad_(order == 2)
        grads = torch.autograd.grad((value * gl.index_select(0, d)).sum(), leaves, create_graph=order == 2)
        dx = grads[0].detach().clone() if dx is None else dx.add_(grads[0].detach())
        dy[at:at + step], dg[at:at + step] = grads[1].detach(), grads[2].detach()
        if order == 2:
            total = ((value * cot[0].index_select(0, d)).sum() + (grads[0] * cot[1]).sum()
                     + (grads[1] * cot[2][at:at + step]).sum() + (grads[2] * cot[3][at:at + step]).sum())
            a, b, o = torch.autograd.grad(total, (leaves[0], leaves[2], gl))
            gx = a.clone() if gx is None else gx.add_(a)
            ggo = o.clone() if ggo is None else ggo.add_(o)
            gg[at:at + step] = b
    return [out] if not order else [out, dx, dy, dg] if order == 1 else [out, dx, dy, dg, gx, gg, ggo]


def _contraction64(module, x, species):
    """x flat mul_ir [N, C (L+1)^2] -> [N, C (T+1)^2] with the module's own U buffers, each compressed
    to its symmetric part over i <= j <= k; weights in the order of module.parameters()."""
    c, lmax, top = module.channels, module.lmax, module.correlation
    d, n = (lmax + 1) ** 2, x.shape[0]
    feats, at = [], 0
    for l in range(lmax + 1):
        feats.append(x[:, at:at + c * (2 * l + 1)].reshape(n, c, 2 * l + 1))
        at += c * (2 * l + 1)
    feats, mono = torch.cat(feats, -1).reshape(n * c, d), {}
    for order in range(1, top + 1):
        full = np.stack(np.meshgrid(*[np.arange(d)] * order, indexing="ij"), -1).reshape(-1, order)
        keep, where = np.unique(np.sort(full, 1), axis=0, return_inverse=True)
        value = feats[:, torch.from_numpy(keep[:, 0].copy()).to(x.device)]
        for q in range(1, order):
            value = value * feats[:, torch.from_numpy(keep[:, q].copy()).to(x.device)]
        mono[order] = (value, torch.from_numpy(where.reshape(-1).copy()).to(x.device), len(keep))
    outs = []
    for l, block in enumerate(module.symmetric_contractions.contractions):
        total = 0.0
        for order, weight in zip(range(top, 0, -1), [block.weights_max, *block.weights]):
            u = getattr(block, "U_matrix_%d" % order).double()
            u = u.reshape(2 * l + 1, d ** order, u.shape[-1])
            value, where, count = mono[order]
            sym = torch.zeros(2 * l + 1, count, u.shape[-1], dtype=torch.float64, device=x.device).index_add(1, where, u)
            chains = torch.stack([value @ s for s in sym], -1).reshape(n, c, u.shape[-1], 2 * l + 1)
            total = total + (chains * weight.index_select(0, species).transpose(1, 2).unsqueeze(-1)).sum(2)
        outs.append(total.reshape(n, -1))
    return torch.cat(outs, 1)


class _Double:
    """A module's parameters in float64 under their own names (leaves that record gradients)."""

    def __init__(self, module, grad):
        self.of = {id(p): p.detach().double().requires_grad_(grad and p.requires_grad) for p in module.parameters()}

    def __call__(self, p):
        return self.of[id(p)]


class _Contraction64:
    """The contraction module's constants with its weights replaced by float64 ones."""

    def __init__(self, module, weights):
        self.channels, self.lmax, self.correlation = module.channels, module.lmax, module.correlation
        self.symmetric_contractions = self
        self.contractions = []
        for block in module.symmetric_contractions.contractions:
            new = type("Block", (), {})()
            new.weights_max, new.weights = weights(block.weights_max), [weights(w) for w in block.weights]
            for order in range(1, module.correlation + 1):
                setattr(new, "U_matrix_%d" % order, getattr(block, "U_matrix_%d" % order))
            self.contractions.append(new)


def _exact_contraction(case, state):
    module, grad = state["call"], case["grad"]
    weights = _Double(module, grad)
    plain = _Contraction64(module, weights)
    params = [weights(p) for p in module.parameters()]
    outs, dxs, dws, step = [], [], None, 512
    for at in range(0, case["nodes"], step):
        x = state["inputs"][0][at:at + step].detach().double().requires_grad_(grad)
        out = _contraction64(plain, x, state["species"][at:at + step])
        outs.append(out.detach())
        if grad:
            dx, *dw = torch.autograd.grad(out, (x, *params), state["go"][at:at + step].double())
            dxs.append(dx)
            dws = dw if dws is None else [a + b for a, b in zip(dws, dw)]
    return [torch.cat(outs)] if not grad else [torch.cat(outs), torch.cat(dxs), *dws]


def _radial64(r):
    n = torch.arange(1, BASIS + 1, dtype=torch.float64, device=r.device)
    x, p = (r / CUTOFF)[:, None], float(CUTOFF_P)
    envelope = 1.0 - (p + 1) * (p + 2) / 2 * x ** p + p * (p + 2) * x ** (p + 1) - p * (p + 1) / 2 * x ** (p + 2)
    wave = math.sqrt(2.0 / CUTOFF) * torch.sin(n * math.pi * r[:, None] / CUTOFF) / r[:, None]
    return wave * envelope * (r < CUTOFF).double()[:, None]


def _silu64(x):
    return torch.nn.functional.silu(x) * SILU_SCALE


def _gates64(interaction, weights, feats):
    layers = [m for m in interaction.fc if hasattr(m, "weight")]
    for lin in layers[:-1]:
        feats = _silu64(feats @ weights(lin.weight).t())
    return feats @ (weights(layers[-1].weight) * weights(interaction.tp.weight).reshape(-1, 1)).t()


def _linear64(linear, weights, m, alpha):
    """[N, sum_l count_l (2l+1) C] -> [N, C (L+1)^2] (per degree [C][2l+1])."""
    n, c, at, parts = m.shape[0], linear.channels, 0, []
    for l, count in enumerate(linear.counts):
        w = count * (2 * l + 1) * c
        rows = m[:, at:at + w].reshape(n, count, 2 * l + 1, c).permute(0, 2, 1, 3).reshape(n, 2 * l + 1, count * c)
        parts.append((rows @ weights(linear.weights[l]).t()).transpose(1, 2).reshape(n, -1) * alpha)
        at += w
    return torch.cat(parts, 1)


def _exact_layer(case, state):
    call, op = state["call"], case["op"]
    weights = _Double(call, True)
    params = [weights(p) for p in _layer_weights(op, call)]
    x, go = state["inputs"][0].detach().double(), state["go"]
    outs, dxs, dws, step = [], [], None, 16384 if op == "gates" else 512
    for at in range(0, x.shape[0], step):
        part = x[at:at + step].clone().requires_grad_()
        out = (_gates64(call, weights, part) if op == "gates"
               else _linear64(call.message_linear, weights, part, 1.0 / call.avg_num_neighbors))
        dx, *dw = torch.autograd.grad(out, (part, *params), go[at:at + step].double())
        outs.append(out.detach())
        dxs.append(dx)
        dws = dw if dws is None else [a + b for a, b in zip(dws, dw)]
    return [torch.cat(outs), torch.cat(dxs), *dws]


def _exact_neighbors(case, state):
    """Every pair over every lattice image in reach, ordered by (dst, src, shift)."""
    pos, cutoff, cell = state["inputs"]
    pos, cell, n = pos.double(), cell.double(), pos.shape[0]
    reach = math.ceil(cutoff / float(cell[0, 0]))
    found = []
    images = [(i, j, k) for i in range(-reach, reach + 1) for j in range(-reach, reach + 1)
              for k in range(-reach, reach + 1)]
    for q, image in enumerate(images):
        shift = torch.tensor(image, dtype=torch.float64, device=pos.device) @ cell
        for at in range(0, n, 4096):
            there = pos[at:at + 4096, None, :] - pos[None, :, :] + shift
            d, s = ((there * there).sum(-1) < cutoff * cutoff).nonzero(as_tuple=True)
            d = d + at
            keep = d != s
            found.append(((d[keep] * n + s[keep]) * len(images) + q))
    key = torch.cat(found).sort().values
    shifts = torch.tensor(images, dtype=torch.float64, device=pos.device)[key % len(images)]
    pair = key // len(images)
    return [pair % n, pair // n, shifts]


def _harmonics64(n, lmax):
    parts = []
    for l in range(lmax + 1):
        monomials, table, scale = harmonics_tables(l)
        mono = torch.stack([n[:, 0] ** a * n[:, 1] ** b * n[:, 2] ** k for a, b, k in monomials], 1)
        parts.append(scale * (mono @ torch.from_numpy(np.ascontiguousarray(table)).to(n.device)))
    return torch.cat(parts, 1)


def _model64(model, weights, graph, species, pos):
    c, lmax, n = model.channels, model.lmax, pos.shape[0]
    src, dst = graph["edge_src"], graph["edge_dst"]
    cell = graph["cell"].double()[graph["batch"][src]]
    vec = pos.index_select(0, dst) - pos.index_select(0, src) + (graph["edge_shifts"].double()[:, :, None] * cell).sum(1)
    r = vec.norm(dim=1)
    y, feats = _harmonics64(vec / r[:, None], lmax), _radial64(r)
    h, energy = weights(model.node_embedding.weight).t()[species], 0.0
    for t, (interaction, product) in enumerate(zip(model.interactions, model.products)):
        lin = interaction.input_lmax
        parts, at = [], 0
        for l in range(lin + 1):
            block = h[:, at:at + c * (2 * l + 1)].reshape(n, c, 2 * l + 1).transpose(1, 2)
            parts.append((block @ weights(interaction.linear_up.weights[l]).t()).reshape(n, -1))
            at += c * (2 * l + 1)
        paths = triangle_paths(lin, lmax, lmax)
        value = _tp64(paths, _couplings(paths, pos.device), c, lmax, torch.cat(parts, 1).index_select(0, src), y,
                      _gates64(interaction, weights, feats))
        m = torch.zeros(n, value.shape[1], dtype=torch.float64, device=pos.device).index_add(0, dst, value)
        message = _linear64(interaction.message_linear, weights, m, 1.0 / interaction.avg_num_neighbors)
        kept = (weights(interaction.self_connection.weight)[species] @ h[:, :c, None]).squeeze(-1)
        out = _contraction64(_Contraction64(product.symmetric_contractions, weights), message, species)
        parts, at = [], 0
        for l in range(product.target_lmax + 1):
            block = out[:, at:at + c * (2 * l + 1)].reshape(n, c, 2 * l + 1)
            block = (weights(product.linear.weights[l]) @ block).reshape(n, -1) / math.sqrt(c)
            parts.append(block + kept if l == 0 else block)
            at += c * (2 * l + 1)
        h = torch.cat(parts, 1)
        if t < len(model.interactions) - 1:
            energy = energy + h[:, :c] @ weights(model.layer_readouts[t].weight).t()
    first, _, last = model.last_readout
    energy = energy + _silu64(h @ weights(first.weight).t()) @ weights(last.weight).t()
    return energy.reshape(-1)


def _exact_model(case, state):
    model = state["call"].model if case["op"] == "replay" else state["call"]
    graph, training = state["graph"], case["op"] == "training"
    weights = _Double(model, training)
    pos = state.get("positions", graph["positions"]).double().requires_grad_()
    atomic = _model64(model, weights, graph, state["species"], pos)
    structures = case["structures"]
    energy = torch.zeros(structures, dtype=torch.float64, device=pos.device).index_add(0, graph["batch"], atomic)
    forces = -torch.autograd.grad(energy.sum(), pos, create_graph=training)[0]
    if not training:
        return {"energy": energy.detach(), "forces": forces.detach(), "atomic_energy": atomic.detach()}
    loss = (energy / pos.shape[0]).square().mean() + forces.square().mean()
    grads = torch.autograd.grad(loss, [weights(p) for p in model.parameters() if p.requires_grad])
    return [loss.detach(), energy.detach(), forces.detach(), *grads]


def exact(case, seed):
    state = prepare(case, seed)
    how = {"tp": _exact_tp, "message": _exact_message, "contraction": _exact_contraction, "gates": _exact_layer,
           "linear": _exact_layer, "neighbors": _exact_neighbors}.get(case["op"], _exact_model)
    return how(case, state)
