"""Dense uvw products on operands split into three bf16 numbers: generated source on the host, choice of kernels, and (on the
GPU) both against the fp64 oracle, with infinities and NaN among the operands too."""
import re

import numpy as np
import pytest

import common
import openequivariance_amd as oeq
from host_emu import emu
from openequivariance_amd.codegen.uvw import UVWGenerator
from openequivariance_amd.codegen.uvw_split import UVWSplitGenerator
from openequivariance_amd.tensor_product import few_rows_generator
from oracle import tp as otp
from oracle import weights as ow


def natural(mul, lmax):
    return "+".join(f"{mul}x{l}{'eo'[l % 2]}" for l in range(lmax + 1))


def both(mul, lmax):
    return "+".join(f"{mul}x{l}{p}" for l in range(lmax + 1) for p in "eo")


def worst(got, ref):
    """Largest error among the rows whose reference is finite, and whether finite values are where the reference has them."""
    rows = np.isfinite(ref).reshape(ref.shape[0], -1).all(1)
    return float(np.abs(got[rows] - ref[rows]).max() / np.abs(ref[rows]).max()), bool((np.isfinite(got) == np.isfinite(ref)).all())


EMULATED = {
    "whole rows through LDS, two tiles a workgroup": ("20x0e+24x1o", "1x0e+1x1o+1x2e", "36x0e+12x1o+5x1e+8x2e", 3, 37),
    "records stored directly, odd channels": ("5x0e+21x1o", "1x0e+1x1o+1x2e", "18x0e+7x1o+3x2e", 3, 37),
    "second operand in another order, a block no path reads, an output no path writes": ("33x0e+2x3o", "1x2e+1x0e", "34x0e+33x2e+4x1o", 2, 19),
    "several tiles for a dW workgroup, two of its kinds": ("70x0e+20x1o", "1x0e+1x1o", "68x0e+16x1o", 2, 150),
    "eight K blocks: the smaller products of dX summed apart, and not": ("18x0e+17x1o", "1x0e+1x1o", "226x0e+18x1o", 4, 37),
}


@pytest.mark.parametrize("name", EMULATED)
def test_generated_source(name, monkeypatch):
    """Every direction forced onto the split kernels.  37, 19 and 150 rows: whole tiles and a ragged one.  The tolerance is that
    of the fp32 kernels' emulation; the split itself holds 24 bits, the products left out are 2^-26 of the largest."""
    a1, a2, a3, groups, n = EMULATED[name]
    monkeypatch.setattr(UVWSplitGenerator, "DW_WORKGROUPS", groups)
    monkeypatch.setattr(UVWSplitGenerator, "_pays", lambda *args: True)
    prob, oprob = common.fully_connected((a1, a2, a3), shared=True, dtype=np.float32)
    g = UVWSplitGenerator(prob)
    assert g.split_forward and g.split_dx and g.dw_kinds and len(g.dw_kinds) <= groups
    X, Y, We, G = common.tp_inputs(prob, n, 9, np.float32, w_scale=0.3)
    W = ow.e3nn_to_oeq(oprob, We)
    fwd, bwd, ws = g.plan()
    for special in (False, True):
        if special:                                          # the part of a wavefront that meets them is computed in fp32
            X[3, 1], G[n - 2, 2] = np.inf, np.nan
        with np.errstate(invalid="ignore"):
            refs = (otp.forward(oprob, X, Y, We), *otp.backward(oprob, X, Y, We, G))
        out = emu.run_tp(g, fwd, X, Y, W, ws_bytes=ws())
        back = emu.run_tp(g, bwd, X, Y, W, G, ws_bytes=ws())
        got = (out["Z"], back["Xg"], back["Yg"], ow.oeq_to_e3nn(oprob, back["Wg"])[:, None])
        for value, ref in zip(got, (*refs[:3], refs[3][:, None])):
            error, finite = worst(value, ref)
            assert error < 2e-6 and finite


# X, W and dZ times these: what bf16 holds of a small number ends at 2^-133, 16 bits above the last bit of fp32
SCALES = {"small rows": (1e-36, 1, 1), "small gradients": (1, 1, 1e-36), "small weights": (1, 1e-36, 1), "denormal rows": (1e-41, 1e8, 1e8),
          "large rows": (1e30, 1, 1), "largest rows": (3e36, 1e-3, 1e-3)}      # (M x of 4100 rows: up to 40 times 3e36, finite in fp32)


@pytest.mark.parametrize("name", SCALES)
def test_small_and_large_operands(name, monkeypatch):
    """No direction loses bits of operands that fp32 holds (tolerance as above)."""
    monkeypatch.setattr(UVWSplitGenerator, "DW_WORKGROUPS", 2)
    monkeypatch.setattr(UVWSplitGenerator, "_pays", lambda *args: True)
    prob, oprob = common.fully_connected(("5x0e+21x1o", "1x0e+1x1o", "18x0e+7x1o"), shared=True, dtype=np.float32)
    g = UVWSplitGenerator(prob)
    X, Y, We, G = (t * np.float32(f) for t, f in zip(common.tp_inputs(prob, 37, 9, np.float32, w_scale=0.3), np.insert(SCALES[name], 1, 1.0)))
    fwd, bwd, ws = g.plan()
    W = ow.e3nn_to_oeq(oprob, We)
    out, back = emu.run_tp(g, fwd, X, Y, W, ws_bytes=ws()), emu.run_tp(g, bwd, X, Y, W, G, ws_bytes=ws())
    refs = (otp.forward(oprob, X, Y, We), *otp.backward(oprob, X, Y, We, G))
    for value, ref in zip((out["Z"], back["Xg"], back["Yg"], ow.oeq_to_e3nn(oprob, back["Wg"])), refs):
        assert np.isfinite(value).all() and np.abs(value - ref).max() < 2e-6 * np.abs(ref).max()


def test_directions_and_rows():
    """Which kernels serve a problem: padding and wavefronts without a tile decide per direction, other types take the fp32 or
    fp64 kernels altogether, and the kernels for few rows keep only the backward's smallest batches."""
    def made(a, b, in2=natural(1, 2), dtype=np.float32):
        return UVWSplitGenerator.create(common.fully_connected((natural(a, 2), in2, natural(b, 2)), shared=True, dtype=dtype)[0])
    g = made(64, 64)
    assert g.split_forward and g.split_dx and len(g.dw_kinds) == 1 and g.few_rows((8192, 5120)) == (0, 2048)
    g = made(20, 72)
    assert g.split_forward and not g.split_dx and g.few_rows((8192, 5120)) == (0, 5120)
    g = made(96, 9)
    assert not g.split_forward and not g.split_dx
    assert made(64, 64, dtype=np.float64) is None and made(16, 16) is None and made(17, 16) is not None
    for a, b in ((64, 64), (100, 100), (8, 100), (100, 8), (33, 50)):
        g = made(a, b)
        assert g.ws_elems >= UVWGenerator(g.problem).ws_elems
        for kernel in g.render().split("__global__")[1:]:
            arrays = re.findall(r"__shared__ (\w+) \w+\[([\d* +]+)\]", kernel)
            assert sum({"T": 4, "VT": 16, "U4": 16}[t] * eval(size) for t, size in arrays) <= UVWSplitGenerator.LDS_BYTES


def test_operators_of_one_problem_share_a_source(monkeypatch):
    """Written once for equal problems, and for no more than a few of them kept."""
    monkeypatch.setattr(UVWSplitGenerator, "_SOURCES", type(UVWSplitGenerator._SOURCES)())
    monkeypatch.setattr(UVWSplitGenerator, "_SOURCES_MAX", 2)
    def generator(mul):
        return UVWSplitGenerator(common.fully_connected((f"{mul}x0e", "1x0e", f"{mul}x0e"), shared=True, dtype=np.float32)[0])
    first = generator(64).render()
    assert generator(64).render() is first and generator(72).render() != first
    generator(80).render()
    assert len(UVWSplitGenerator._SOURCES) == 2 and generator(64).render() == first


# Few wavefronts on a compute unit beside long rows: what was slower than the fp32 kernels (40 000 rows, both sides with the rules);
# forward, dX / dY, dW on split operands
DIRECTIONS = {
    "four wavefronts": (natural(64, 3), natural(1, 1), natural(64, 3), False, False, True),
    "four wavefronts, both parities": (both(50, 2), "1x0e", both(50, 2), False, False, True),
    "three wavefronts, both parities": (both(33, 2), natural(1, 2), both(33, 2), False, False, True),
    "two workgroups of four": (both(50, 1), "1x0e", both(50, 1), True, True, True),
    "five, several paths a block": (natural(65, 2), natural(1, 2), natural(65, 2), True, True, True),
    "five, one path a block": (natural(65, 2), "1x0e", natural(65, 2), False, True, False),
    "six, one path a block": (natural(48, 2), "1x0e", natural(48, 2), False, True, True),
    "seven, one path a block": (natural(100, 2), "1x0e", natural(100, 2), True, True, True),
    "narrow outputs": (natural(64, 2), natural(1, 2), natural(16, 2), False, True, False),
    "narrow outputs of few paths": (natural(64, 2), "1x0e", natural(16, 2), False, True, True),
}


@pytest.mark.parametrize("name", DIRECTIONS)
def test_directions_that_pay(name):
    *irreps, forward, dx, dw = DIRECTIONS[name]
    g = UVWSplitGenerator.create(common.fully_connected(irreps, shared=True, dtype=np.float32)[0])
    assert (g.split_forward, g.split_dx, bool(g.dw_kinds)) == (forward, dx, dw)


@pytest.mark.parametrize("irreps,kept", [
    ((natural(48, 2), natural(1, 2), natural(48, 2)), (0, 4096)), ((natural(25, 1), natural(1, 2), natural(25, 1)), (0, 5120)),
    ((natural(65, 2), natural(1, 2), natural(65, 2)), (0, 0)), ((natural(64, 2), "1x0e", natural(64, 2)), (0, 1024)),
    ((both(50, 1), "1x0e", both(50, 1)), (2048, 8192)), ((natural(100, 2), "1x0e", natural(100, 2)), (1024, 0)),
    ((natural(20, 2), "1x0e", natural(64, 2)), (2048, 65536)), ((both(50, 2), "1x0e", both(50, 2)), (8192, 65536))])
def test_rows_left_to_the_kernels_for_few(irreps, kept):
    g = UVWSplitGenerator.create(common.fully_connected(irreps, shared=True, dtype=np.float32)[0])
    assert g.few_rows((8192, 65536)) == kept and g.few_rows((0, 0)) == (0, 0)
    few, limits = few_rows_generator(g.problem, g)
    assert (few is None) == (not any(limits)) and all(a <= b for a, b in zip(limits, kept))
    if few is not None:
        assert ("void forward(" in few.render()) == bool(few.plan()[0]) == (limits[0] > 0)


# dW workgroups of several kinds: the one that stages most of dZ is not the one with most entries of the M table, and the two
# together would exceed a compute unit; both parities, degrees up to 5, uneven multiplicities
KINDS = {
    "64 -> 96, both parities": (natural(64, 2), natural(1, 2), "96x0e+96x0o+96x1e+96x1o+96x2e+96x2o"),
    "64x4e": ("64x4e", natural(1, 4), "100x5o+32x5o+20x4e"),
    "scalars": ("109x0o+79x0e", natural(1, 3), "68x0e+86x0o+75x1e+96x1o+68x2e+90x2o"),
    "17 and 38 -> 94": ("17x0e+38x1o+17x2e", natural(1, 2), "94x0e+94x0o+94x1e+94x1o+94x2e+94x2o"),
    "92 and 40 -> 98": ("92x0e+40x1o", natural(1, 4), "98x0e+98x0o+77x1e+4x1o+98x2e+98x2o"),
    "127 and 40 -> 72": ("127x0e+40x1o+40x2e+40x3o", natural(1, 4), "72x0e+72x1o+72x2e+72x3o+17x4e"),
    "85 -> 10, 4 and 76": ("85x0e+85x0o+85x1e+85x1o", natural(1, 4), "10x2e+4x0e+76x4e+76x1o+76x3o"),
    **{f"{mul}, both parities": (both(mul, 2), natural(1, 2), both(mul, 2)) for mul in (20, 33, 72, 128)},
    **{f"{mul}, l <= {lmax}": (natural(mul, lmax), natural(1, lmax), natural(mul, lmax)) for mul in (24, 65, 128) for lmax in (1, 3, 4)},
}


@pytest.mark.parametrize("name", KINDS)
def test_arrays_fit_lds_together(name):
    """A kernel's arrays as emitted, not one kind of workgroup or one array at a time: what exceeds 160 KB does not compile."""
    g = UVWSplitGenerator.create(common.fully_connected(KINDS[name], shared=True, dtype=np.float32)[0])
    used = common.lds_bytes(g.render(), 4) if g is not None else {}
    assert all(size <= 160 * 1024 for size in used.values()), used
    if g is not None and g.dw_kinds:
        assert used["backward_dw"] == max(kind.lds_bytes() for kind in g.dw_kinds)


def test_source_whose_dw_kinds_nearly_fill_lds_builds():
    from openequivariance_amd import runtime as rt
    g = UVWSplitGenerator.create(common.fully_connected(KINDS["scalars"], shared=True, dtype=np.float32)[0])
    used = rt.kernel_metadata(rt.compile_source(g.render()))["backward_dw"][".group_segment_fixed_size"]
    assert 150 * 1024 < used <= 160 * 1024


GPU = {"64": (natural(64, 2), natural(1, 2), natural(64, 2)), "100": (natural(100, 2), natural(1, 1), natural(100, 1)),
       "20 -> 72": (natural(20, 2), natural(1, 2), natural(72, 2)), "50, both parities": ("50x0e+50x1o+50x1e", "1x0e", "50x0e+50x1o+50x1e"),
       "33 -> 47": (natural(33, 1), natural(1, 1), natural(47, 2)), "132": (natural(132, 1), "1x0e", natural(132, 1)),
       "three kinds of dW workgroups that nearly fill LDS": KINDS["scalars"]}


@pytest.mark.gpu
@pytest.mark.parametrize("name", GPU)
@pytest.mark.parametrize("n", [1, 16, 2049, 6001])
def test_gpu_against_oracle(name, n):
    import torch
    prob, _ = common.fully_connected(GPU[name], shared=True, dtype=np.float32)
    p64, _ = common.fully_connected(GPU[name], shared=True, dtype=np.float64)
    op, ref = oeq.TensorProduct(prob), oeq.TensorProduct(p64)
    assert type(op.generator) is UVWSplitGenerator
    X, Y, W, G = (torch.tensor(t, device="cuda") for t in common.tp_inputs(prob, n, 5, np.float32))
    refs = (ref.forward(X.double(), Y.double(), W.double()), *ref.backward_helper(X.double(), Y.double(), W.double(), G.double()))
    got = (op.forward(X, Y, W), *op.backward_helper(X, Y, W, G))
    # fp32 sums of at most 11 x 132 products, dW of 6001 rows: 2-norm errors of a few 1e-7 (fp32 matrix instructions: 1 to 4e-7)
    for a, b in zip(got, refs):
        assert float((a.double() - b).norm() / b.norm()) < 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("name", SCALES)
def test_gpu_small_and_large_operands(name):
    import torch
    prob, _ = common.fully_connected(GPU["64"], shared=True, dtype=np.float32)
    p64, _ = common.fully_connected(GPU["64"], shared=True, dtype=np.float64)
    op, ref = oeq.TensorProduct(prob), oeq.TensorProduct(p64)
    assert op.generator.split_forward and op.generator.split_dx and op.generator.dw_kinds
    X, Y, W, G = (torch.tensor(t * np.float32(f), device="cuda")
                  for t, f in zip(common.tp_inputs(prob, 4100, 5, np.float32), np.insert(SCALES[name], 1, 1.0)))
    refs = (ref.forward(X.double(), Y.double(), W.double()), *ref.backward_helper(X.double(), Y.double(), W.double(), G.double()))
    for a, b in zip((op.forward(X, Y, W), *op.backward_helper(X, Y, W, G)), refs):
        # (dW: a denormal T = M x of 1e-41 is rounded at 2^-149 in fp32 arithmetic of any kind, here at 2^-150; measured 2.5e-6)
        tol = 2.0 ** -149 / 1e-41 if b.ndim == 1 and name == "denormal rows" else 1e-6
        assert float((a.double() - b).norm() / b.norm()) < tol


# operands of one sign: all channels of a row meet the same roundings, and dY adds them up
ONE_SIGN = {"64": (GPU["64"], True), "200, l <= 1": ((natural(200, 1), natural(1, 1), natural(200, 1)), True),
            "256 scalars": (("256x0e", "1x0e", "256x0e"), True), "512 scalars": (("512x0e", "1x0e", "512x0e"), False)}


@pytest.mark.gpu
@pytest.mark.parametrize("name", ONE_SIGN)
def test_gpu_operands_of_one_sign(name):
    import torch
    irreps, dw_kinds = ONE_SIGN[name]
    prob, p64 = (common.fully_connected(irreps, shared=True, dtype=t)[0] for t in (np.float32, np.float64))
    op, ref = oeq.TensorProduct(prob), oeq.TensorProduct(p64)
    assert op.generator.split_forward and op.generator.split_dx and bool(op.generator.dw_kinds) == dw_kinds
    gen = torch.Generator(device="cuda").manual_seed(3)
    X, Y, W, G = (torch.rand(*s, device="cuda", generator=gen) + 0.5
                  for s in ((4100, prob.irreps_in1.dim), (4100, prob.irreps_in2.dim), (prob.weight_numel,), (4100, prob.irreps_out.dim)))
    refs = (ref.forward(X.double(), Y.double(), W.double()), *ref.backward_helper(X.double(), Y.double(), W.double(), G.double()))
    # fp32 matrix instructions: Z, dX up to 3.2e-7, dW 2.5e-7; dY up to 6e-8 - one rounding of a result is 3.4e-8
    for a, b, tol in zip((op.forward(X, Y, W), *op.backward_helper(X, Y, W, G)), refs, (3.2e-7, 3.2e-7, 2.0 ** -24, 2.5e-7)):
        assert float((a.double() - b).norm() / b.norm()) < tol


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["64", "33 -> 47", "50, both parities"])
def test_gpu_misaligned_and_strided_rows(name):
    """Views that start at any word and rows cut from wider ones, in every operand: as for contiguous copies, bit for bit."""
    import torch
    prob, _ = common.fully_connected(GPU[name], shared=True, dtype=np.float32)
    op = oeq.TensorProduct(prob, torch_op=True)
    op._few_rows_limits = (0, 0)
    operands = [torch.tensor(t, device="cuda") for t in common.tp_inputs(prob, 4099, 5, np.float32)]
    def run(x, y, w, g):
        x, y, w = (t.detach().requires_grad_() for t in (x, y, w))
        z = op(x, y, w)
        return [z.detach(), *torch.autograd.grad(z, (x, y, w), g)]
    want = run(*operands)
    for off in (1, 2, 3):
        def shifted(t):
            out = torch.empty(t.numel() + off, device="cuda")[off:].view(t.shape)
            return out.copy_(t)
        def cut(t):
            wide = torch.full((*t.shape[:-1], t.shape[-1] + off + 2), float("nan"), device="cuda")
            return wide[..., off:off + t.shape[-1]].copy_(t)
        for view in (shifted, cut):
            assert all(torch.equal(a, b) for a, b in zip(run(*map(view, operands)), want))
    # results at any word, through the raw entry points
    n, off = operands[0].shape[0], 3
    x, y, w, g = (torch.empty(t.numel() + off, device="cuda")[off:].copy_(t.reshape(-1)) for t in operands)
    dx, dy, dw = (torch.empty(t.numel() + 1, device="cuda")[1:] for t in operands[:3])
    z = torch.empty(operands[3].numel() + 1, device="cuda")[1:]
    op.forward_raw(n, x.data_ptr(), y.data_ptr(), z.data_ptr(), w.data_ptr())
    op.backward_raw(n, x.data_ptr(), dx.data_ptr(), y.data_ptr(), dy.data_ptr(), w.data_ptr(), dw.data_ptr(), g.data_ptr())
    torch.cuda.synchronize()
    assert all(torch.equal(a, b.reshape(-1)) for a, b in zip((z, dx, dy, dw), want))


@pytest.mark.gpu
def test_gpu_streams_of_one_operator():
    """Packed weights and partial sums lie in a workspace per stream: calls with weights of their own on four streams at once."""
    import torch
    prob, _ = common.fully_connected(GPU["64"], shared=True, dtype=np.float32)
    op = oeq.TensorProduct(prob)
    sets = [[torch.tensor(t, device="cuda") for t in common.tp_inputs(prob, 6001, seed, np.float32)] for seed in range(4)]
    want = [[op.forward(*s[:3]), *op.backward_helper(*s)] for s in sets]
    streams = [torch.cuda.Stream() for _ in sets]
    torch.cuda.synchronize()
    got = [[] for _ in sets]
    for _ in range(3):
        for q, (stream, s) in enumerate(zip(streams, sets)):
            with torch.cuda.stream(stream):
                got[q].append([op.forward(*s[:3]), *op.backward_helper(*s)])
    torch.cuda.synchronize()
    for q in range(len(sets)):
        for out in got[q]:
            assert all(torch.equal(a, b) for a, b in zip(out, want[q]))


@pytest.mark.gpu
def test_gpu_infinities_and_large_values():
    """Rows with an infinity, a NaN and values whose bf16 rounding is infinite; the other rows keep their accuracy."""
    import torch
    prob, oprob = common.fully_connected((natural(64, 1), natural(1, 1), natural(64, 1)), shared=True, dtype=np.float32)
    op = oeq.TensorProduct(prob)
    assert op.generator.split_forward and op.generator.split_dx and op.generator.dw_kinds
    n = 4100
    X, Y, We, G = common.tp_inputs(prob, n, 6, np.float32, w_scale=1e-3)
    X[5, 3], G[40, 7], X[70, 9], G[n - 1, 0] = np.inf, np.nan, 3.4e38, -np.inf
    x, y, w, g = (torch.tensor(t, device="cuda") for t in (X, Y, ow.e3nn_to_oeq(oprob, We), G))
    z = op.forward(x, y, w)
    dx, dy, dw = op.backward_helper(x, y, w, g)
    with np.errstate(invalid="ignore", over="ignore"):
        ref = (otp.forward(oprob, X, Y, We), *otp.backward(oprob, X, Y, We, G))
    big = np.arange(n) == 70                                 # (fp32 may overflow there where the oracle does not)
    for value, r in zip((z, dx, dy), ref):
        error, _ = worst(value.cpu().numpy()[~big], r[~big])
        assert error < 2e-6
        assert (np.isfinite(value.cpu().numpy()[~big]) == np.isfinite(r[~big])).all()
    zb, rb = z.cpu().numpy()[big], ref[0][big]
    assert np.isfinite(zb).all() and np.abs(zb - rb).max() <= 2e-6 * np.abs(rb).max()
    got = ow.oeq_to_e3nn(oprob, dw.cpu().numpy())
    assert (~np.isfinite(got))[~np.isfinite(ref[3])].all()
    # (entries that the 3.4e38 takes part in may overflow in fp32; of the others every one that is finite is computed)
    X[70, 9] = 0
    with np.errstate(invalid="ignore", over="ignore"):
        without = otp.backward(oprob, X, Y, We, G)[2]
    plain = np.isfinite(ref[3]) & (without == ref[3])
    assert 0.5 < plain.mean() < 1 and np.isfinite(got[plain]).all()
    assert np.abs(got[plain] - ref[3][plain]).max() < 2e-6 * np.abs(ref[3][plain]).max()
