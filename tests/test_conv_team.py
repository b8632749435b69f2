"""Convolutions of few nodes, whose edges are walked by a team of wavefronts: the generated source on the host (tests/host_emu) at
the edges of the schedule - nodes with fewer edges than the team has wavefronts, one and two row groups per wavefront,
LDS-staged and register loops, several chunks and launches, long nodes walked in pieces, edges naming no node."""
import numpy as np
import pytest

import common
from common import rel_err
from host_emu import emu
from openequivariance_amd.codegen.uvu_det import UVUDetGenerator
from openequivariance_amd.codegen.uvu_recv import UVURecvGenerator
from openequivariance_amd.codegen.uvu_sorted import UVUSortedGenerator
from oracle import tp as otp

CASES = {   # irreps, dtype, nodes, edges, hub?, generator arguments
    "two_row_groups_staged": (common.NEQUIP, np.float32, 9, 60, False, {}),
    "two_row_groups_registers": (common.NEQUIP, np.float32, 9, 60, False, dict(lds=False)),
    "hubs": (("16x0e+16x1o", "1x0e+1x1o", "16x0e+16x1o"), np.float32, 12, 400, True, {}),
    "chunks_and_launches_fp64": (("5x0e+3x1o+70x2e", "1x0e+1x1o+1x2e", "5x0e+3x1o+70x2e+7x3o"), np.float64, 6, 40, False, {}),
}
TOL = {np.float32: 5e-6, np.float64: 1e-13}       # some hundred roundings a value


def graph(case):
    _, _, nodes, nnz, hub, _ = CASES[case]
    if hub:
        return *common.hub_graph(nodes, nnz, 3, hub_in=3, hub_out=5, in_edges=150, out_edges=130), np.ones(nnz, bool)
    return common.with_invalid_edges(*common.random_graph(nodes - 1, nnz, 3), nodes, 4)        # the last node has no edges


def check(g, case, rows, cols, tperm, valid, **kw):
    irreps, dtype, nodes, nnz, _, _ = CASES[case]
    prob, oprob = common.channelwise(irreps, dtype=dtype)
    X, Y, W, G = common.conv_inputs(prob, nodes, nnz, 5, dtype=dtype)
    want = common.conv_reference_on_valid_edges(otp, oprob, X, Y, W, G, rows, cols, valid)
    fwd, bwd, ws = g.plan()
    out = emu.run_conv(g, fwd, X, Y, W, rows, cols, tperm=tperm, ws_bytes=ws(nnz, nodes))
    assert rel_err(out["Z"], want[0]) < TOL[dtype]
    out = emu.run_conv(g, bwd, X, Y, W, rows, cols, G=G, tperm=tperm, ws_bytes=ws(nnz, nodes))
    for got, ref in zip((out["Xg"], out["Yg"], out["Wg"]), want[1:]):
        assert rel_err(got, ref) < TOL[dtype]


@pytest.mark.parametrize("team", [2, 4])
@pytest.mark.parametrize("case", sorted(CASES))
def test_sorted_edges(case, team):
    irreps, dtype, nodes, _, hub, kw = CASES[case]
    rows, cols, valid = graph(case)
    rows, cols, tperm, order = otp.coord_graph(rows, cols)
    check(UVUDetGenerator(common.channelwise(irreps, dtype=dtype)[0], **kw).team_twin(team), case, rows, cols, tperm,
          (rows >= 0) & (rows < nodes) & (cols >= 0) & (cols < nodes))


@pytest.mark.parametrize("cls", [UVUSortedGenerator, UVURecvGenerator])
@pytest.mark.parametrize("case", ["two_row_groups_staged", "hubs"])
def test_unsorted_edges_and_receiver_order(case, cls):
    irreps, dtype, nodes, _, _, _ = CASES[case]
    rows, cols, valid = graph(case)
    tperm = None
    if cls is UVURecvGenerator:
        rows, cols, tperm, _ = otp.coord_graph(rows, cols)
        valid = (rows >= 0) & (rows < nodes) & (cols >= 0) & (cols < nodes)
        g = cls(common.channelwise(irreps, dtype=dtype)[0]).team_twin()
    else:
        g = cls(common.channelwise(irreps, dtype=dtype)[0], grouped_backward=True)
        g.fwd, g.bwd = g.fwd.team_twin(), g.bwd.team_twin()
    check(g, case, rows, cols, tperm, valid)


@pytest.mark.gpu
@pytest.mark.parametrize("deterministic", [False, True])
@pytest.mark.parametrize("irreps,dtype", [(common.NEQUIP, np.float32), (("16x0e+16x1o", "1x0e+1x1o", "16x0e+16x1o"), np.float32),
                                          (common.MACE, np.float32), (("64x0e+64x1o+64x2e", "1x0e+1x1o+1x2e", "64x0e+64x1o+64x2e"), np.float64)],
                         ids=["staged", "four_row_groups", "receiver_order", "fp64"])
def test_on_the_gpu(cuda, irreps, dtype, deterministic, monkeypatch):
    """At both sides of the size rule, and on a small graph with hubs: forward, backward and double backward against single
    wavefronts' (same products, another order of the sums), the deterministic operator bit for bit twice."""
    import torch
    import openequivariance_amd as oeq
    prob, _ = common.channelwise(irreps, dtype=dtype)
    conv = oeq.TensorProductConv(prob, torch_op=True, deterministic=deterministic)
    monkeypatch.setattr(UVUDetGenerator, "TEAMS", ())
    single = oeq.TensorProductConv(prob, torch_op=True, deterministic=deterministic)
    assert "forward_few" in conv.jit_kernel and "forward_few" not in single.jit_kernel
    for c in (conv, single):
        if not deterministic:
            c._bwd_choice = type("Grouped", (dict,), dict(__contains__=lambda s, k: True, __getitem__=lambda s, k: "grouped"))()
    monkeypatch.undo()
    g = getattr(conv.generator, "fwd", conv.generator)
    (_, _, four), (_, beyond, two) = g.few_teams("forward")
    each = 2 * g.R
    assert beyond == four < two
    for n, nnz, graph in ((four, four * each, common.random_graph), (four + 1, 5 * four, common.random_graph),
                          (two, two * each, common.random_graph), (two, two * each - 1, common.random_graph),
                          (two + 1, 5 * two, common.random_graph), (1, 2 * each, lambda n, nnz, seed: (np.zeros(nnz, np.int64),) * 2),
                          (40, 900, lambda n, nnz, seed: common.hub_graph(n, nnz, seed, 3, 5, 300, 200))):
        print(n, nnz, flush=True)
        rows, cols, tperm, _ = otp.coord_graph(*graph(n, nnz, 7))
        index = [torch.tensor(a, device=cuda) for a in ((rows, cols, tperm) if deterministic else (rows, cols))]
        t = [torch.tensor(a, device=cuda) for a in (*common.conv_inputs(prob, n, nnz, 8, dtype), *common.conv_inputs(prob, n, nnz, 9, dtype)[:3])]

        def run(c):
            x, y, w, g = (a.clone().requires_grad_() for a in t[:4])
            z = c(x, y, w, *index)
            first = torch.autograd.grad(z, (x, y, w), g, create_graph=True)
            return [z, *first, *torch.autograd.grad(first, (x, y, w, g), t[4:])]
        got, again, want = run(conv), run(conv), run(single)
        for a, b, c in zip(got, again, want):
            assert rel_err(a.detach().cpu().numpy(), c.detach().cpu().numpy()) < TOL[dtype]
            assert not deterministic or torch.equal(a, b)
