"""The counting sort that groups an unsorted edge list: ranges of nodes, the scan in LDS and in memory, several workgroups."""
import numpy as np
import pytest
import torch

import common
import openequivariance_amd as oeq
from host_emu import emu
from openequivariance_amd.codegen.uvu_sorted import UVUSortedGenerator
from oracle import tp as otp


@pytest.mark.parametrize("range_nodes,nodes", [(64, 150), (64, 64), (64, 63), (256, 150)])
def test_groups_of_several_ranges_and_workgroups(range_nodes, nodes, monkeypatch):
    """1300 edges in workgroups of 1024, a hub, edges naming no node; counters walked in LDS (fewer nodes
    than a range) and in memory, called twice on one workspace as the counters are left zero."""
    monkeypatch.setattr(UVUSortedGenerator, "GROUP_NODES", range_nodes)
    monkeypatch.setattr(UVUSortedGenerator, "GROUP_EDGES", 1)
    prob, oprob = common.channelwise(("2x0e+2x1o", "1x0e+1x1o", "2x0e+2x1o"))
    g = UVUSortedGenerator(prob, grouped_backward=True)
    nnz = 1300
    rng = np.random.default_rng(nodes)
    rows, cols = rng.integers(0, nodes, nnz), rng.integers(0, nodes, nnz)
    rows[100:400], cols[700:900] = 5, nodes - 1
    rows[1000:1003], cols[1010:1012] = (-1, nodes, nodes + 40), (nodes, -7)
    valid = (rows >= 0) & (rows < nodes) & (cols >= 0) & (cols < nodes)
    X, Y, W, G = common.conv_inputs(prob, nodes, nnz, 3)
    Z, dX, dY, dW = common.conv_reference_on_valid_edges(otp, oprob, X, Y, W, G, rows, cols, valid)
    fwd, bwd, ws = g.plan()
    again = [s for s in fwd if not s.get("counter_clear")], [s for s in bwd if not s.get("counter_clear")]
    out = emu.run_conv(g, fwd + again[0], X, Y, W, rows, cols, ws_bytes=ws(nnz, nodes))
    assert common.rel_err(out["Z"], Z) < 2e-6
    out = emu.run_conv(g, bwd + again[1], X, Y, W, rows, cols, G=G, ws_bytes=ws(nnz, nodes))
    for got, ref in zip((out["Xg"], out["Yg"], out["Wg"]), (dX, dY, dW)):
        assert common.rel_err(got, ref) < 2e-6


def test_edge_positions_hold_32_bits():
    """The grouping kernels keep positions in 32 bits: longer edge lists are refused before anything is launched (tensors
    without storage)."""
    class Conv(oeq.TensorProductConv):
        def __init__(self, generator):
            self.generator, self.deterministic, self._dims = generator, False, (8, 4, 8, 4)
            self._torch_dtype, self._torch_idx = torch.float32, torch.int64
    conv = Conv(UVUSortedGenerator(common.channelwise(("2x0e+2x1o", "1x0e+1x1o", "2x0e+2x1o"))[0]))
    for edges, message in ((2 ** 32, "edge count"), (2 ** 32 - 1, "must be on the GPU")):
        x, y, w = (torch.empty(n, d, device="meta") for n, d in ((10, 8), (edges, 4), (edges, 4)))
        rows, cols = (torch.empty(edges, dtype=torch.int64, device="meta") for _ in range(2))
        with pytest.raises(ValueError, match=message):
            conv._check(x, y, w, rows, cols)
