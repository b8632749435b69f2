"""Double backward of the uvu batch product in one launch: the generated source on the host (tests/host_emu) and the
operator on the GPU against the second derivatives of the fp64 oracle, at the edges of the schedule: one to sixteen rows
per wavefront, ragged multiplicities, one to three 64-channel chunks, copies of the second operand, blocks no path
touches, operands requested one output block ahead or all at once."""
import os
import tempfile

import numpy as np
import pytest

import common
import openequivariance_amd as oeq
from common import rel_err
from host_emu import emu
from openequivariance_amd.codegen.uvu_double import UVUDoubleGenerator
from oracle import spec, torch_cpu, weights as ow

CASES = {   # irreps, batch sizes
    "two_rows_per_wavefront": (common.NEQUIP, (1, 5)),
    "sixteen_rows": (("3x0e+3x1o", "1x0e+1x1o", "3x0e+3x1o"), (1, 19)),
    "ragged_two_chunks": (("5x0e+3x1o+70x2e", "1x0e+1x1o+1x2e", "5x0e+3x1o+70x2e+7x3o"), (2,)),
    "three_chunks": (("192x0e+192x1o", "1x0e+1x1o", "192x0e+192x1o"), (2,)),
    "blocks_no_path_touches": (("1x0e+1x1o+16x3o", "1x0e+1x1o", "16x0e+16x0o+16x1e+16x1o"), (3,)),
    "copies_of_the_second_operand": (("12x0e+12x1o", "3x0e+2x1o", "12x0e+12x1o"), (7,)),
}
MAIN = r"""
int main(int argc, char** argv) {
    const std::string d = argv[1];
    FILE* job = fopen((d + "/job.txt").c_str(), "r");
    unsigned long long n, d1, d2, d3, wn; unsigned grid;
    if (fscanf(job, "%llu %llu %llu %llu %llu %u", &n, &d1, &d2, &d3, &wn, &grid) != 6) return 3;
    auto in = [&](const char* name, unsigned long long w) { return emu_read(d + "/" + name + ".bin", n * w * sizeof(T)); };
    auto X = in("X", d1), Y = in("Y", d2), W = in("W", wn), G = in("G", d3), A = in("A", d1), B = in("B", d2), V = in("V", wn);
    std::vector<char> Xg(n * d1 * sizeof(T), (char)0x7f), Yg(n * d2 * sizeof(T), (char)0x7f), Wg(n * wn * sizeof(T), (char)0x7f),
        Gg(n * d3 * sizeof(T), (char)0x7f);
    emu_run(grid, 1, 64, [&] { double_backward(n, (const T*)X.data(), (const T*)Y.data(), (const T*)W.data(), (const T*)G.data(),
        (const T*)A.data(), (const T*)B.data(), (const T*)V.data(), (T*)Xg.data(), (T*)Yg.data(), (T*)Wg.data(), (T*)Gg.data()); });
    emu_write(d + "/Xg.bin", Xg); emu_write(d + "/Yg.bin", Yg); emu_write(d + "/Wg.bin", Wg); emu_write(d + "/Gg.bin", Gg);
    return 0;
}
"""


def _problems(case, dtype=np.float32):
    a = CASES[case][0]
    if case == "copies_of_the_second_operand":
        ins = [(0, 0, 0, "uvu", True), (1, 1, 0, "uvu", True), (1, 0, 1, "uvu", True)]
        return (oeq.TPProblem(*a, ins, shared_weights=False, internal_weights=False, irrep_dtype=dtype, weight_dtype=dtype),
                spec.Problem(*a, ins, shared_weights=False))
    return common.channelwise(a, dtype)


def _inputs(prob, n, seed, dtype):
    X, Y, W, G = common.tp_inputs(prob, n, seed, dtype)
    A, B, V, _ = common.tp_inputs(prob, n, seed + 1, dtype)
    return X, Y, W, G, A, B, V


def _reference(oprob, X, Y, We, G, A, B, Ve):
    """fp64 second derivatives (weights and their cotangents in e3nn order)."""
    import torch
    x, y, w, g = (torch.tensor(a.astype(np.float64), requires_grad=True) for a in (X, Y, We, G))
    z = torch_cpu.TorchTP(oprob, dtype=torch.float64).forward(x, y, w)
    first = torch.autograd.grad(z, (x, y, w), g, create_graph=True)
    return [t.numpy() for t in torch.autograd.grad(first, (x, y, w, g), [torch.tensor(a.astype(np.float64)) for a in (A, B, Ve)])]


@pytest.mark.parametrize("case", sorted(CASES))
def test_generated_source_without_vector_stores(case, monkeypatch):
    test_generated_source(case, None, monkeypatch, vector_stores=False)


@pytest.mark.parametrize("ahead", [False, True])
@pytest.mark.parametrize("case", sorted(CASES))
def test_generated_source(case, ahead, monkeypatch, vector_stores=True):
    prob, oprob = _problems(case)
    monkeypatch.setattr(UVUDoubleGenerator, "ONE_BLOCK_AHEAD", ahead)
    g = UVUDoubleGenerator(prob, vector_stores=vector_stores)
    exe = emu.build(g.render(prelude=emu.emu_prelude(g.T)), MAIN)
    for n in CASES[case][1]:
        X, Y, We, G, A, B, Ve = _inputs(prob, n, 5, np.float32)
        arrays = dict(X=X, Y=Y, W=ow.e3nn_to_oeq(oprob, We), G=G, A=A, B=B, V=ow.e3nn_to_oeq(oprob, Ve))
        with tempfile.TemporaryDirectory() as d:
            for k, a in arrays.items():
                np.ascontiguousarray(a, dtype=np.float32).tofile(os.path.join(d, k + ".bin"))
            with open(os.path.join(d, "job.txt"), "w") as f:
                f.write(f"{n} {g.D1} {g.D2} {g.D3} {g.WN} {emu.grid_of(g.plan()[0], n, 0)}\n")
            emu._run(exe, d)
            got = [np.fromfile(os.path.join(d, k + ".bin"), dtype=np.float32).reshape(a.shape)
                   for k, a in (("Xg", X), ("Yg", Y), ("Wg", We), ("Gg", G))]
        got[2] = ow.oeq_to_e3nn(oprob, got[2])
        for a, b in zip(got, _reference(oprob, X, Y, We, G, A, B, Ve)):
            assert rel_err(a, b) < 4e-6       # twice the terms of a first derivative, fp32 against fp64


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("case", sorted(CASES))
def test_operator(cuda, case, dtype):
    import torch
    prob, oprob = _problems(case, dtype)
    tol = 2e-5 if dtype == np.float32 else 2e-12       # two chained kernels' worth of the first-order tolerances
    tp = oeq.TensorProduct(prob, torch_op=True)
    for n in (*CASES[case][1], 333):
        X, Y, We, G, A, B, Ve = _inputs(prob, n, 6, dtype)
        x, y, w, g = (torch.tensor(a, device=cuda, requires_grad=True) for a in (X, Y, ow.e3nn_to_oeq(oprob, We), G))
        cots = [torch.tensor(a, device=cuda) for a in (A, B, ow.e3nn_to_oeq(oprob, Ve))]
        first = torch.autograd.grad(tp(x, y, w), (x, y, w), g, create_graph=True)
        second = torch.autograd.grad(first, (x, y, w, g), cots, retain_graph=True)
        assert tp._double, "the second derivatives did not come from the fused kernel"
        torch.cuda.synchronize()
        got = [t.cpu().numpy() for t in second]
        got[2] = ow.oeq_to_e3nn(oprob, got[2])
        for a, b in zip(got, _reference(oprob, X, Y, We, G, A, B, Ve)):
            assert rel_err(a, b) <= tol
        # a graph of the second derivatives is built from first-order calls: the same numbers, differentiable again
        again = torch.autograd.grad(first, (x, y, w, g), cots, create_graph=True)
        for a, b in zip(again, second):
            assert rel_err(a.detach().cpu().numpy(), b.cpu().numpy()) <= tol
        third = torch.autograd.grad(again[0].square().sum(), (y, w))
        assert all(bool(torch.isfinite(t).all()) for t in third)


@pytest.mark.gpu
def test_loss_on_one_of_the_gradients_and_misaligned_operands(cuda):
    """Forces usually come from dY alone: the other two cotangents do not exist.  A dZ at an odd storage offset changes
    nothing: the operator's outputs, which 16-byte stores go to, are its own."""
    import torch
    prob, oprob = common.channelwise(common.NEQUIP)
    tp = oeq.TensorProduct(prob, torch_op=True)
    X, Y, W, G, A, B, V = _inputs(prob, 41, 7, np.float32)
    x, y, w = (torch.tensor(a, device=cuda, requires_grad=True) for a in (X, Y, W))
    g = torch.zeros(G.size + 1, device=cuda)[1:].view(G.shape).copy_(torch.tensor(G)).requires_grad_()
    first = torch.autograd.grad(tp(x, y, w), (x, y, w), g, create_graph=True)
    got = torch.autograd.grad(first[1], (x, y, w, g), torch.tensor(B, device=cuda), allow_unused=True)
    ref = _reference(oprob, X, Y, W, G, 0 * A, B, 0 * V)
    for a, b in zip(got, ref):
        if a is not None and np.abs(b).max() > 0:
            assert rel_err(a.cpu().numpy(), b) <= 2e-5


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_misaligned_outputs(cuda, dtype):
    """Raw outputs that are not 16-byte aligned take the kernels without 16-byte stores; nothing beside them is written."""
    import torch
    prob, oprob = common.channelwise(common.NEQUIP, dtype)
    tp = oeq.TensorProduct(prob, torch_op=False)
    X, Y, W, G, A, B, V = _inputs(prob, 41, 8, dtype)
    ops = [torch.tensor(a, device=cuda) for a in (X, Y, W, G, A, B, V)]
    for offset in (0, 1):
        pads = [torch.full((t.numel() + 8,), 7.0, dtype=t.dtype, device=cuda) for t in ops[:4]]
        outs = [p[offset:offset + t.numel()].view(t.shape) for p, t in zip(pads, ops)]
        tp.double_backward_raw(41, *(t.data_ptr() for t in (*ops, *outs)))
        torch.cuda.synchronize()
        assert (offset == 0) in tp._double
        for p, t in zip(pads, ops):
            assert bool((p[:offset] == 7).all()) and bool((p[offset + t.numel():] == 7).all())
        for a, b in zip(outs, _reference(oprob, X, Y, W, G, A, B, V)):
            assert rel_err(a.cpu().numpy(), b) <= (2e-5 if dtype == np.float32 else 2e-12)


@pytest.mark.gpu
def test_capture_before_the_first_call(cuda):
    """The kernels are loaded with the operator: a stream capture records them without an eager call before it."""
    import torch
    prob, oprob = common.channelwise(common.NEQUIP)
    X, Y, W, G, A, B, V = _inputs(prob, 70, 9, np.float32)
    x, y, w, g = (torch.tensor(a, device=cuda, requires_grad=True) for a in (X, Y, W, G))
    cots = [torch.tensor(a, device=cuda) for a in (A, B, V)]

    def step(tp):
        first = torch.autograd.grad(tp(x, y, w), (x, y, w), g, create_graph=True)
        return torch.autograd.grad(first, (x, y, w, g), cots)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        eager = step(oeq.TensorProduct(prob, torch_op=True))             # (torch's own first use, by another operator)
    side.synchronize()
    tp = oeq.TensorProduct(prob, torch_op=True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = step(tp)
    for _ in range(3):
        for t in out:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, eager))
        assert all(torch.equal(a, b) for a, b in zip(step(tp), eager))
    for a, b in zip(out, _reference(oprob, X, Y, W, G, A, B, V)):
        assert rel_err(a.cpu().numpy(), b) <= 2e-5
