"""Ahead-of-time hipRTC compilation of the benchmark configurations' kernels.

hipRTC cross-compiles for gfx950 without a GPU, so the code objects of the benchmark
problems can be produced where the package is built and picked up from the in-tree cache on the
GPU machine.  Problems outside this list are compiled on first construction as usual.
"""
from __future__ import annotations

import time

import numpy as np

from . import runtime as rt
from .codegen.uvu_conv_double import conv_double_generator
from .codegen.uvu_double import UVUDoubleGenerator
from .codegen.uvw import UVWGenerator
from .codegen.uvw_batched import UVWBatchedGenerator
from .codegen.uvw_split import UVWSplitGenerator
from .conv import select_conv_generator, with_few_nodes
from .problem import ChannelwiseTPP, FullyConnectedTPProblem, TPProblem
from .tensor_product import few_rows_generator, select_generator
from .workloads import get as get_workload
from .workloads import DENSE, DIFFDOCK_L2, LARGE, MACE, MACE_ALL, NEQUIP, TETRIS_POLY


def benchmark_generators():
    """(label, generator) for every kernel set the operators of the benchmark workloads and of the smoke test are
    constructed with, chosen by the same selection functions."""
    readme = TPProblem("1x2e", "1x3e", "1x2e", [(0, 0, 0, "uvu", True)], shared_weights=False, internal_weights=False)
    gens = []

    def tp(label, problem):
        g = select_generator(problem)
        gens.append((label, g))
        if type(g) in (UVWGenerator, UVWSplitGenerator, UVWBatchedGenerator):
            few, _ = few_rows_generator(problem, g)
            if few is not None:
                gens.append((label + " few rows", few))
        elif problem.instructions[0].connection_mode == "uvu" and UVUDoubleGenerator.suits(problem):
            gens.append((label + " double backward", UVUDoubleGenerator(problem)))

    def conv(label, problem, deterministic):
        gens.append((label, with_few_nodes(select_conv_generator(problem, deterministic))))
        gens.append((label + " double backward", with_few_nodes(conv_double_generator(problem, deterministic))))

    tp("readme/tp", readme)
    tp("mace/tp", ChannelwiseTPP(*MACE))
    tp("mace-all-parities/tp", ChannelwiseTPP(*MACE_ALL))
    tp("nequip/tp", ChannelwiseTPP(*NEQUIP))
    for label, irreps in (("nequip", NEQUIP), ("large", LARGE), ("mace", MACE)):
        for det in (False, True):
            conv(f"{label}/conv_{'det' if det else 'atomic'}", ChannelwiseTPP(*irreps), det)
    for det in (False, True):
        p = ChannelwiseTPP(*MACE, irrep_dtype=np.float64, weight_dtype=np.float64)
        conv(f"mace/conv_{'det' if det else 'atomic'}/float64", p, det)
    conv("benzene/conv_det", get_workload("benzene_conv_det").problem(), True)
    for dt in (np.float32, np.float64):
        p = FullyConnectedTPProblem(*DENSE, shared_weights=True, internal_weights=False, irrep_dtype=dt, weight_dtype=dt)
        tp(f"dense/uvw/{np.dtype(dt).name}", p)
        p = FullyConnectedTPProblem(*DIFFDOCK_L2, shared_weights=False, internal_weights=False, irrep_dtype=dt, weight_dtype=dt)
        tp(f"diffdock/uvw per-row weights/{np.dtype(dt).name}", p)
        for which, irreps in TETRIS_POLY.items():
            p = FullyConnectedTPProblem(*irreps, shared_weights=True, internal_weights=False, irrep_dtype=dt, weight_dtype=dt)
            tp(f"tetris-poly-{which}/uvw few weights/{np.dtype(dt).name}", p)
    return gens


def compile_benchmark_kernels(verbose: bool = False, refresh: bool = False) -> None:
    """``refresh``: compile every kernel set again even where the cache already holds its code object."""
    for name, g in benchmark_generators():
        t = time.time()
        code = rt.compile_source(g.render(), refresh=refresh)
        if verbose:
            print(f"hipRTC gfx950 {name}: {len(code) // 1024} KiB ({time.time() - t:.1f}s)", flush=True)
