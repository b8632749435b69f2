"""The counting sort that groups an unsorted edge list: ranges of nodes, the scan in LDS and in memory, several workgroups."""
import subprocess

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


SHAPES = {"keys over more ranges than a workgroup walks": dict(GROUP_RANGES=1, GROUP_NODES=16, GROUP_EDGES=1),
          "... with runs of equal keys": dict(GROUP_RANGES=1, GROUP_NODES=16, GROUP_FEW_EDGES=0),
          "one workgroup, several turns of its threads": dict(GROUP_WORKGROUPS=1, GROUP_FEW_EDGES=0, GROUP_EDGES=1),
          "ranges from the first node named, runs": dict(GROUP_NODES=16, GROUP_FEW_EDGES=0)}


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("order", ["random", "by receiver"])
def test_shares_and_spans_of_workgroups(shape, order, monkeypatch):
    """275 edges in workgroups of 128 threads, a hub, edges naming no node among them."""
    for name, value in dict(SHAPES[shape], SCAN_THREADS=128).items():
        monkeypatch.setattr(UVUSortedGenerator, name, value)
    prob, oprob = common.channelwise(("2x0e+2x1o", "1x0e+1x1o", "2x0e+2x1o"))
    g = UVUSortedGenerator(prob, grouped_backward=False)
    nnz, nodes = 275, 60
    rng = np.random.default_rng(7)
    rows, cols = rng.integers(5, nodes, nnz), rng.integers(0, nodes, nnz)
    rows[50:150] = 50
    if order == "by receiver":
        rows.sort()
    rows[200:203], cols[205:207] = (-1, nodes, 2 ** 40), (nodes, -7)
    valid = (rows >= 0) & (rows < nodes) & (cols >= 0) & (cols < nodes)
    X, Y, W, G = common.conv_inputs(prob, nodes, nnz, 3)
    Z = common.conv_reference_on_valid_edges(otp, oprob, X, Y, W, G, rows, cols, valid)[0]
    fwd, _, ws = g.plan()
    out = emu.run_conv(g, fwd, X, Y, W, rows, cols, ws_bytes=ws(nnz, nodes))
    assert common.rel_err(out["Z"], Z) < 2e-6


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


def test_shares_cover_every_edge_list():
    """A workgroup's share of the edges times the workgroups launched, up to the longest list that is taken."""
    g = UVUSortedGenerator(common.channelwise(("2x0e+2x1o", "1x0e+1x1o", "2x0e+2x1o"))[0])
    edges = [1, 1024, 1025, 32768, 32769, 4096 * 128, 4096 * 128 + 1, 2 ** 31, 2 ** 32 - 128, 2 ** 32 - 127, 2 ** 32 - 1]
    main = "int main() { for (u64 n : {" + ", ".join(f"{n}ull" for n in edges) + '}) printf("%llu\\n", (unsigned long long)oeq_group_share(n)); }'
    shares = subprocess.run([emu.build(g.render(prelude=emu.emu_prelude("float")), main)], capture_output=True, text=True, check=True).stdout.split()
    step = next(s for s in g.plan()[0] if s["kernel"] == "group_count")
    for n, share in zip(edges, map(int, shares)):
        assert share % step["num_threads"] == 0 and share * emu.grid_of(step, n, 1) >= n


@pytest.mark.gpu
@pytest.mark.parametrize("nodes", [1023, 16383, 16384, 16385, 100_001])
@pytest.mark.parametrize("order", ["random", "by receiver", "hub"])
def test_gpu_against_sorted_edges(nodes, order):
    """Edges of the ranges in LDS, of keys over more nodes than a workgroup walks, and of lists long enough for four per thread;
    the deterministic operator on the sorted list sums the same edges of a node in its own order."""
    prob, _ = common.channelwise(("4x0e+4x1o", "1x0e+1x1o", "4x0e+4x1o"))
    free, fixed = oeq.TensorProductConv(prob, torch_op=True), oeq.TensorProductConv(prob, torch_op=True, deterministic=True)
    nnz = 150_001
    gen = torch.Generator(device="cuda").manual_seed(nodes)
    rows, cols = (torch.randint(0, nodes, (nnz,), device="cuda", generator=gen) for _ in range(2))
    if order == "hub":
        rows[torch.randperm(nnz, device="cuda", generator=gen)[:nnz // 2]] = nodes - 1
    if order == "by receiver":
        rows = rows.sort().values
    x, y, w = (torch.randn(n, d, device="cuda", generator=gen)
               for n, d in ((nodes, prob.irreps_in1.dim), (nnz, prob.irreps_in2.dim), (nnz, prob.weight_numel)))
    g = torch.randn(nodes, prob.irreps_out.dim, device="cuda", generator=gen)
    r, c, perm, tperm = oeq.sort_by_receiver(rows, cols, nodes)
    want = [fixed.forward(x, y[perm], w[perm], r, c, tperm)]
    dx, dy, dw = fixed.backward_helper(x, y[perm], w[perm], g, r, c, tperm)
    back = torch.empty_like(perm)
    back[perm] = torch.arange(nnz, device="cuda")
    want += [dx, dy[back], dw[back]]
    for _ in range(2):
        got = (free.forward(x, y, w, rows, cols), *free.backward_helper(x, y, w, g, rows, cols))
        for a, b in zip(got, want):
            assert float((a - b).norm() / b.norm()) < 2e-6     # (a hub's 75 000 edges summed in another order)
