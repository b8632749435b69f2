"""The workloads this library's speed is judged by: its two operators, ``TensorProduct`` and ``TensorProductConv``,
called as a model's program calls them, over the range of problems, sizes, directions and data types they are used at.

A case is a dict of plain values:

* ``op``      ``tp`` (a product per row of a batch) or ``conv`` (gather - product - scatter over the edges of a graph)
* ``mode``    ``uvu`` (channel-wise) or ``uvw`` (fully connected)
* ``in1``, ``in2``, ``out``  the irreps; every path they allow is in use
* ``shared``  one weight vector for all rows (True) or one per row / edge (False)
* ``dtype``   ``f32`` or ``f64``
* ``rows``    batch rows or edges; ``nodes`` and ``sorted`` (edges sorted by receiver, deterministic operator) for ``conv``
* ``what``    ``forward`` (inference without gradients), ``train`` (forward and the gradients of all three operands: a
  training step, and equally the energy and forces of a molecular-dynamics step), ``forces`` (training on forces:
  the gradients of the first derivatives too, i.e. forward, backward and double backward)
"""
import math

import numpy as np
import torch

import openequivariance_amd as oeq
from openequivariance_amd.sh import random_unit_vectors, spherical_harmonics

DTYPES = {"f32": (np.float32, torch.float32, 4), "f64": (np.float64, torch.float64, 8)}


def listed():
    return [
        # the README's one-path product: the smallest call, nothing but call overhead and one short launch
        dict(name="readme_forward", op="tp", mode="uvu", in1="1x2e", in2="1x3e", out="1x2e", shared=False, dtype="f32",
             rows=1000, what="forward"),
        # the 17-path, 128-channel product of a MACE interaction over the edges of a training batch
        dict(name="mace_train", op="tp", mode="uvu", in1="128x0e+128x1o+128x2e", in2="1x0e+1x1o+1x2e+1x3o",
             out="128x0e+128x1o+128x2e+128x3o", shared=False, dtype="f32", rows=50000, what="train"),
        # the smaller MACE interaction (8 paths) trained on forces; an odd number of edges
        dict(name="mace_medium_forces", op="tp", mode="uvu", in1="128x0e+128x1o", in2="1x0e+1x1o+1x2e+1x3o",
             out="128x0e+128x1o+128x2e", shared=False, dtype="f32", rows=20011, what="forces"),
        # a channel-wise product whose weights belong to the layer and not to the edge
        dict(name="shared_uvu_train", op="tp", mode="uvu", in1="64x0e+64x1o+64x2e", in2="1x0e+1x1o+1x2e",
             out="64x0e+64x1o+64x2e", shared=True, dtype="f32", rows=30001, what="train"),
        # one molecular-dynamics step of a small cell: energy and forces, neighbour list as it comes
        dict(name="md_step", op="conv", mode="uvu", in1="64x0e+64x1o", in2="1x0e+1x1o", out="64x0e+64x1o",
             shared=False, dtype="f32", rows=5183, nodes=192, sorted=False, what="train"),
        # NequIP-style convolution over a large batch of graphs, edges in no order
        dict(name="nequip_conv_train", op="conv", mode="uvu", in1="32x0e+32x1o+32x2e", in2="1x0e+1x1o+1x2e",
             out="32x0e+32x1o+32x2e", shared=False, dtype="f32", rows=150000, nodes=5000, sorted=False, what="train"),
        # the same layer trained on forces, a small batch, deterministic
        dict(name="nequip_conv_forces", op="conv", mode="uvu", in1="32x0e+32x1o+32x2e", in2="1x0e+1x1o+1x2e",
             out="32x0e+32x1o+32x2e", shared=False, dtype="f32", rows=30000, nodes=1001, sorted=True, what="forces"),
        # the MACE interaction as a fused convolution in double precision
        dict(name="mace_conv_train_f64", op="conv", mode="uvu", in1="128x0e+128x1o+128x2e", in2="1x0e+1x1o+1x2e+1x3o",
             out="128x0e+128x1o+128x2e+128x3o", shared=False, dtype="f64", rows=300000, nodes=10000, sorted=True,
             what="train"),
        # the largest: 256 channels on 800 000 edges, deterministic
        dict(name="large_conv_train", op="conv", mode="uvu", in1="256x0e+256x1o+256x2e", in2="1x0e+1x1o+1x2e+1x3o",
             out="256x0e+256x1o+256x2e", shared=False, dtype="f32", rows=800000, nodes=20000, sorted=True, what="train"),
        # a dense fully connected layer with shared weights on a large batch
        dict(name="dense_uvw_train", op="tp", mode="uvw", in1="64x0e+64x1o+64x2e", in2="1x0e+1x1o+1x2e",
             out="64x0e+64x1o+64x2e", shared=True, dtype="f32", rows=100000, what="train"),
        # a hidden layer of the tetris classifier: multiplicities of 50, both parities, small batch, double precision
        dict(name="tetris_uvw_train_f64", op="tp", mode="uvw", in1="50x0e+50x1o+50x1e+50x2o+50x2e", in2="1x0e",
             out="50x0e+50x1o+50x1e+50x2o+50x2e", shared=True, dtype="f64", rows=4097, what="train"),
        # DiffDock's fully connected product with a weight vector per edge
        dict(name="diffdock_train", op="tp", mode="uvw", in1="10x1o+10x1e+48x0e+48x0o", in2="1x0e+1x1o+1x2e",
             out="10x1o+10x1e+48x0e+48x0o", shared=False, dtype="f32", rows=50000, what="train"),
    ]


def _spread(rng, lo, hi):
    """A whole number, spread over the logarithm of the range, odd as often as even."""
    return min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def _natural(mul, lmax):
    return "+".join(f"{mul}x{l}{'eo'[l % 2]}" for l in range(lmax + 1))


def _both(mul, lmax):
    return "+".join(f"{mul}x{l}{p}" for l in range(lmax + 1) for p in "eo")


def draw(rng):
    """One more case: channel-wise products and convolutions of 8 to 128 channels, fully connected layers with shared
    weights and with weights per row; graphs of 64 to 10 000 nodes and batches of 500 to 50 000 rows."""
    family = rng.choice(["uvu", "uvu", "uvu", "conv", "conv", "conv", "conv", "uvw", "uvw", "uvw_rows", "uvu_shared"])
    case = dict(op="tp", mode="uvu", shared=False, dtype="f64" if rng.random() < 0.25 else "f32")
    if family in ("uvu", "conv", "uvu_shared"):
        mul = rng.choice([16, 32, 64, 128]) if rng.random() < 0.5 else _spread(rng, 8, 128)
        lmax = rng.choice([1, 2])
        irreps = _both if rng.random() < 0.25 and mul <= 64 else _natural
        case.update(in1=irreps(mul, lmax), in2=_natural(1, rng.choice([lmax, 3])), out=irreps(mul, lmax),
                    what=rng.choice(["forward", "train", "train", "forces"]), shared=(family == "uvu_shared"))
        if family == "conv":
            nodes = _spread(rng, 64, 10000)
            case.update(op="conv", nodes=nodes, rows=int(nodes * rng.uniform(8, 40)), sorted=rng.random() < 0.5)
        else:
            case.update(rows=_spread(rng, 500, 50000))
    elif family == "uvw":
        a, b = _spread(rng, 8, 100), _spread(rng, 8, 100)
        case.update(mode="uvw", shared=True, in1=_natural(a, rng.choice([1, 2])), in2=_natural(1, rng.choice([0, 1, 2])),
                    out=_natural(b, rng.choice([1, 2])), rows=_spread(rng, 500, 50000),
                    what=rng.choice(["forward", "train", "train"]))
    else:
        a = _spread(rng, 4, 48)
        case.update(mode="uvw", in1=_natural(a, rng.choice([1, 2])), in2=_natural(1, rng.choice([1, 2])),
                    out=_natural(a, rng.choice([1, 2])), rows=_spread(rng, 500, 20000),
                    what=rng.choice(["forward", "train", "train"]))
    while work(case)["bytes"] > 6e9:
        case["rows"] = case["rows"] * 2 // 3
    return case


def _problem(case):
    kw = dict(irrep_dtype=DTYPES[case["dtype"]][0], weight_dtype=DTYPES[case["dtype"]][0])
    irreps = (case["in1"], case["in2"], case["out"])
    if case["mode"] == "uvw":
        return oeq.FullyConnectedTPProblem(*irreps, shared_weights=case["shared"], internal_weights=False, **kw)
    if irreps == ("1x2e", "1x3e", "1x2e"):
        return oeq.TPProblem(*irreps, [(0, 0, 0, "uvu", True)], shared_weights=False, internal_weights=False, **kw)
    p = oeq.ChannelwiseTPP(*irreps, **kw)
    if not case["shared"]:
        return p
    paths = [(i.i_in1, i.i_in2, i.i_out, "uvu", True) for i in p.instructions]
    return oeq.TPProblem(p.irreps_in1, p.irreps_in2, p.irreps_out, paths, shared_weights=True, internal_weights=False, **kw)


def prepare(case, seed):
    problem = _problem(case)
    _, dtype, _ = DTYPES[case["dtype"]]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, device="cuda", dtype=dtype, generator=gen)

    n = case["rows"]
    d1, d2, d3 = problem.irreps_in1.dim, problem.irreps_in2.dim, problem.irreps_out.dim
    # second operand: spherical harmonics of edge directions (a pool of random directions, one of them per row)
    lmax = max(ir.l for _, ir in problem.irreps_in2)
    pool = spherical_harmonics(lmax, random_unit_vectors(4096, np.random.default_rng(seed)))[:, -d2:]
    pool = torch.tensor(pool, device="cuda", dtype=dtype)
    y = pool[torch.randint(0, pool.shape[0], (n,), device="cuda", generator=gen)]
    x = normal(case["nodes"] if case["op"] == "conv" else n, d1)
    w = normal(problem.weight_numel) if case["shared"] else normal(n, problem.weight_numel)
    index = ()
    if case["op"] == "conv":
        nodes = case["nodes"]
        receivers = torch.randint(0, nodes, (n,), device="cuda", generator=gen)
        senders = torch.randint(0, nodes - 1, (n,), device="cuda", generator=gen)
        senders = senders + (senders >= receivers)                       # no self-loops
        index = (receivers, senders)
        if case["sorted"]:
            receivers, senders, _, transpose_perm = oeq.sort_by_receiver(receivers, senders, nodes)
            index = (receivers, senders, transpose_perm)
        op = oeq.TensorProductConv(problem, torch_op=True, deterministic=case["sorted"])
    else:
        op = oeq.TensorProduct(problem, torch_op=True)
    state = dict(op=op, index=index, what=case["what"], args=(x, y, w))
    if case["what"] != "forward":
        state["args"] = tuple(t.requires_grad_() for t in state["args"])
        state["g"] = normal(x.shape[0], d3)                              # gradient arriving from the rest of the model
    if case["what"] == "forces":
        state["g"].requires_grad_()
        state["probes"] = (normal(*x.shape), normal(*y.shape), normal(*w.shape))     # gradient of the loss on the forces
    return state


def run(state):
    op, args, index = state["op"], state["args"], state["index"]
    if state["what"] == "forward":
        with torch.no_grad():
            return [op(*args, *index)]
    z = op(*args, *index)
    if state["what"] == "train":
        return [z.detach(), *torch.autograd.grad(z, args, state["g"])]
    first = torch.autograd.grad(z, args, state["g"], create_graph=True)
    second = torch.autograd.grad(first, (*args, state["g"]), state["probes"])
    return [z.detach(), *(t.detach() for t in first), *second]


def work(case):
    problem = _problem(case)
    n, size = case["rows"], DTYPES[case["dtype"]][2]
    nodes = case["nodes"] if case["op"] == "conv" else n
    x, y, z = nodes * problem.irreps_in1.dim, n * problem.irreps_in2.dim, nodes * problem.irreps_out.dim
    w = problem.weight_numel * (1 if case["shared"] else n)
    words = {"forward": x + y + w + z,                                   # read x, y, w; write z
             "train": 2 * (x + y + w + z),                               # ... read dz; write dx, dy, dw
             "forces": 4 * (x + y + w) + 3 * z}[case["what"]]            # ... read the probes; write four second gradients
    index = 16 * n * (1.5 if case.get("sorted") else 1) if case["op"] == "conv" else 0
    if case["mode"] == "uvw":
        flops = sum(2 * math.prod(i.path_shape) * problem.irreps_out[i.i_out].ir.dim for i in problem.instructions)
        passes = {"forward": 1, "train": 3, "forces": 10}
    else:
        flops = 0
        for i in problem.instructions:
            l1, l2, l3 = problem.irreps_in1[i.i_in1].ir.l, problem.irreps_in2[i.i_in2].ir.l, problem.irreps_out[i.i_out].ir.l
            flops += 3 * int(np.count_nonzero(np.abs(oeq.wigner_3j(l1, l2, l3)) > 1e-14)) * math.prod(i.path_shape)
        passes = {"forward": 1, "train": 4, "forces": 16}
    return {"bytes": float(words * size + index), "flops": float(flops * n * passes[case["what"]])}


def tolerance(case):
    """About four times what fp32 outputs were seen to differ by from the same call in fp64 on the same inputs: at most
    7.5e-7 in the 2-norm and 4e-6 in a value (the weight gradient of a dense layer, summed over 100 000 rows); for fp64 the
    same, scaled by the ratio of the two types' precisions."""
    return {"rel": 3e-6, "max": 2e-5} if case["dtype"] == "f32" else {"rel": 6e-15, "max": 4e-14}
