"""The launches of a call on a workspace stay together when several threads use one operator on one stream.  The runtime
(csrc/oeq_hip.cpp) is built for the host over a HIP of a few lines whose launches are written down and take a millisecond."""
import ctypes as C
import pathlib
import shutil
import subprocess
import threading

import pytest

from openequivariance_amd import runtime as rt

ROOT = pathlib.Path(__file__).resolve().parent.parent
HIP = r"""
#pragma once
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <cstdlib>
#include <mutex>
#include <unistd.h>
#include <vector>
#define __device__
#define __align__(n) __attribute__((aligned(n)))
typedef int hipError_t;
enum { hipSuccess = 0 };
typedef void *hipModule_t, *hipFunction_t, *hipStream_t, *hipEvent_t;
struct hipDeviceProp_t { char name[256], gcnArchName[256]; int warpSize, major, minor, multiProcessorCount, clockRate, memoryClockRate,
    memoryBusWidth, l2CacheSize; size_t sharedMemPerBlock, totalGlobalMem; };
enum { hipDeviceAttributeMaxSharedMemoryPerBlock, hipFuncAttributeMaxDynamicSharedMemorySize, hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
#define OK(name) template <class... A> int name(A...) { return 0; }
OK(hipModuleUnload) OK(hipFuncSetAttribute) OK(hipGetLastError) OK(hipGetDeviceCount) OK(hipGetDeviceProperties)
OK(hipDeviceGetAttribute) OK(hipEventCreate) OK(hipEventDestroy) OK(hipEventRecord) OK(hipEventSynchronize)
OK(hipEventElapsedTime) OK(hipFree) OK(hipMalloc) OK(hipMemsetAsync) OK(hipMemcpy) OK(hipStreamSynchronize)
inline const char* hipGetErrorString(int) { return "error"; }
inline int hipGetDevice(int* d) { *d = 0; return 0; }
inline int hipModuleLoadData(hipModule_t* m, const void*) { *m = (void*)1; return 0; }
inline int hipModuleGetFunction(hipFunction_t* f, hipModule_t, const char* name) { *f = strdup(name); return 0; }
#define HIP_SYMBOL(x) (&x)
template <class T> int hipGetSymbolAddress(void** p, T* symbol) { *p = (void*)symbol; return 0; }
inline std::mutex g_log_mutex;
inline std::vector<std::pair<const char*, const void*>> g_log;           // kernel, first argument
inline int hipModuleLaunchKernel(hipFunction_t f, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, hipStream_t,
                                 void** args, void**) {
    { std::lock_guard<std::mutex> lock(g_log_mutex); g_log.push_back({(const char*)f, *(void**)args[0]}); }
    usleep(1000);
    return 0;
}
extern "C" inline __attribute__((used)) size_t log_size() { return g_log.size(); }
extern "C" inline __attribute__((used)) const char* log_kernel(size_t i) { return g_log[i].first; }
extern "C" inline __attribute__((used)) const void* log_caller(size_t i) { return g_log[i].second; }
extern "C" inline __attribute__((used)) void log_clear() { g_log.clear(); }
"""
HIPRTC = r"""
#pragma once
typedef int hiprtcResult;
typedef void* hiprtcProgram;
enum { HIPRTC_SUCCESS = 0 };
template <class... A> int hiprtcVersion(A...) { return 0; }
template <class... A> int hiprtcCreateProgram(A...) { return 0; }
template <class... A> int hiprtcCompileProgram(A...) { return 0; }
template <class... A> int hiprtcGetProgramLogSize(A...) { return 0; }
template <class... A> int hiprtcGetProgramLog(A...) { return 0; }
template <class... A> int hiprtcDestroyProgram(A...) { return 0; }
template <class... A> int hiprtcGetCodeSize(A...) { return 0; }
template <class... A> int hiprtcGetCode(A...) { return 0; }
inline const char* hiprtcGetErrorString(int) { return "error"; }
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    """The runtime over the HIP above."""
    d = tmp_path_factory.mktemp("host_hip")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(HIP)
    (d / "hip" / "hiprtc.h").write_text(HIPRTC)
    subprocess.run([shutil.which("g++"), "-std=c++17", "-O1", "-fPIC", "-shared", "-pthread", f"-I{d}", str(ROOT / "openequivariance_amd/csrc/oeq_hip.cpp"),
                    "-o", str(d / "host.so")], check=True)
    L = C.CDLL(str(d / "host.so"))
    L.log_kernel.restype, L.log_caller.restype, L.log_size.restype = C.c_char_p, C.c_void_p, C.c_size_t
    return L


def handle(L, kind, n):
    """An operator whose plans are ``n`` kernels each."""
    steps = [(rt.Step * n)(*(rt.Step.make(f"{kind}_{d}_{i}", 64, flags=rt.STEP_NEEDS_WORKSPACE) for i in range(n))) for d in "fb"]
    h = C.c_void_p()
    assert getattr(L, f"oeq_{kind}_create")(b"code", C.c_size_t(4), steps[0], n, steps[1], n, C.byref(h)) == 0
    return h


def runs(L):
    """The launches as written down: (caller, its kernels in a row)."""
    out = []
    for i in range(L.log_size()):
        caller, kernel = L.log_caller(i), L.log_kernel(i).decode()
        if kernel.endswith("_0"):
            out.append((caller, [kernel]))
        else:
            assert out and out[-1][0] == caller, f"{kernel} of one caller among the launches of another"
            out[-1][1].append(kernel)
    return [k for _, k in out]


P, U = C.c_void_p, C.c_uint64
WS = 1 << 21
CALLS = {
    # (the first argument, which the log names the caller by, is the batch or the first operand)
    "tp_forward": ("tp", "f", lambda L, h, me: L.oeq_tp_forward(h, U(me), *[P(8)] * 4, P(WS), None)),
    "tp_backward": ("tp", "b", lambda L, h, me: L.oeq_tp_backward(h, U(me), *[P(8)] * 7, P(WS), None)),
    "conv_forward": ("conv", "f", lambda L, h, me: L.oeq_conv_forward_ex(h, P(me), *[P(8)] * 5, U(9), U(9), P(WS), P(8), None, 0)),
    "conv_backward": ("conv", "b", lambda L, h, me: L.oeq_conv_backward_ex(h, P(me), *[P(8)] * 8, U(9), U(9), P(WS), P(8), None, 0)),
    "conv_double": ("conv", "b", lambda L, h, me: L.oeq_conv_double_backward_ex(h, P(me), *[P(8)] * 12, U(9), U(9), P(WS), P(8), None, 0)),
}


@pytest.mark.parametrize("a, b", [("tp_forward", "tp_forward"), ("tp_forward", "tp_backward"), ("tp_backward", "tp_backward"),
                                  ("conv_forward", "conv_forward"), ("conv_forward", "conv_backward"), ("conv_backward", "conv_double")])
def test_launches_of_a_call_stay_together(host, a, b):
    host.log_clear()
    kinds = [CALLS[n] for n in (a, b)]
    handles = [handle(host, kind, 3) for kind, _, _ in kinds]                   # two kernel sets, one workspace
    status = []

    def work(k):
        _, _, call = kinds[k]
        status.extend(call(host, handles[k], 1000 + k) for _ in range(10))
    threads = [threading.Thread(target=work, args=(k,)) for k in (0, 1)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert status == [0] * 20
    want = sorted([f"{kind}_{d}_{i}" for i in range(3)] for kind, d, _ in kinds for _ in range(10))
    assert sorted(runs(host)) == want


def counted(L):
    """A convolution whose plans are a step that clears counters, and two more."""
    flags = (rt.STEP_NEEDS_WORKSPACE | rt.STEP_COUNTER_CLEAR, rt.STEP_NEEDS_WORKSPACE, rt.STEP_NEEDS_WORKSPACE)
    steps = [(rt.Step * 3)(*(rt.Step.make(f"{d}_{i}", 64, flags=f) for i, f in enumerate(flags))) for d in "fb"]
    h = C.c_void_p()
    assert L.oeq_conv_create(b"code", C.c_size_t(4), steps[0], 3, steps[1], 3, C.byref(h)) == 0
    return h


def clears(L, call):
    L.log_clear()
    assert call() == 0
    names = [L.log_kernel(i).decode() for i in range(L.log_size())]
    assert [n[-1] for n in names] in (["0", "1", "2"], ["1", "2"])
    return len(names) == 3


def on(L, h, counters, kind, which, nnz, nodes, me=8):
    call = {"f": L.oeq_conv_forward_on, "b": L.oeq_conv_backward_on, "d": L.oeq_conv_double_backward_on}[which]
    return call(h, P(me), *[P(8)] * {"f": 5, "b": 8, "d": 12}[which], U(nnz), U(nodes), P(WS), P(8), None, 0, C.byref(counters), U(kind))


def test_record_of_the_counters(host):
    """The step that clears them is left out exactly where a completed call of the same sizes and kind left them zero, and no call
    of other sizes, no unknown one and no capture came between."""
    h, c = counted(host), rt.ConvCounters()
    for which, nnz, nodes, kind, cleared in (
            ("f", 9, 5, 1, True), ("f", 9, 5, 1, False), ("b", 9, 5, 2, True), ("f", 9, 5, 1, False), ("b", 9, 5, 2, False),
            ("b", 9, 5, 3, True), ("f", 9, 5, 1, False),                            # another kernel set's backward
            ("f", 8, 5, 1, True), ("b", 9, 5, 3, True), ("f", 8, 5, 1, True), ("f", 8, 5, 1, False),      # other sizes
            ("d", 8, 5, 0, True), ("f", 8, 5, 1, True), ("f", 8, 5, 0, True), ("f", 8, 5, 1, True), ("f", 8, 5, 1, False)):
        assert clears(host, lambda: on(host, h, c, kind, which, nnz, nodes)) == cleared, (which, nnz, nodes, kind)
    c.captured = 1
    assert clears(host, lambda: on(host, h, c, 1, "f", 8, 5)) and clears(host, lambda: on(host, h, c, 1, "f", 8, 5))


def test_record_of_the_counters_by_two_threads(host):
    """Calls of two sizes on one workspace: a call that follows one of the other size clears, however the threads take turns."""
    h, c = counted(host), rt.ConvCounters()
    host.log_clear()

    def work(me):
        for _ in range(20):
            assert on(host, h, c, 1, "f", me, 5, me) == 0
    threads = [threading.Thread(target=work, args=(me,)) for me in (1000, 1001)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    last, calls = None, 0
    for i in range(host.log_size()):
        caller, step = host.log_caller(i), host.log_kernel(i).decode()[-1]
        assert step != "1" or caller == last or host.log_kernel(i - 1).decode()[-1] == "0"
        if step == "2":
            last, calls = caller, calls + 1
    assert calls == 40


def test_a_lease_knows_nothing_of_its_counters():
    """A buffer put in another's place: what a call in the old one left in the record meanwhile says nothing about the new one."""
    import torch
    from openequivariance_amd import autograd_glue
    autograd_glue._operators()
    ops = torch.ops.openequivariance_amd
    id = ops.native_operator([0] * 16, [0] * 9, [])
    c = rt.ConvCounters()
    ops.native_lease(id, torch.empty(256, dtype=torch.uint8), 0, 0, C.addressof(c))
    c.forward[:], c.backward[:] = (900, 70, 1), (900, 70, 3)
    ops.native_lease(id, torch.empty(512, dtype=torch.uint8), 0, 0, C.addressof(c))
    assert c.forward[2] == c.backward[2] == 0


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["uvw", "conv", "conv_sorted"])
def test_two_threads_on_one_stream(cuda, case):
    """One operator, two threads with operands (a graph, weights) of their own, one of them with operands that the general
    implementation takes: every pass gives what it gives by itself."""
    import numpy as np
    import torch
    import common
    import openequivariance_amd as oeq
    from oracle import tp as otp
    if case == "uvw":
        prob = common.fully_connected(common.DENSE, shared=True)[0]
        op = oeq.TensorProduct(prob, torch_op=True)
    else:
        prob = common.channelwise(common.NEQUIP)[0]
        op = oeq.TensorProductConv(prob, torch_op=True, deterministic=case == "conv_sorted")

    def operands(k):
        if case == "uvw":
            return [torch.tensor(a, device=cuda) for a in common.tp_inputs(prob, 2000 + 300 * k, k, np.float32)], []
        nodes, nnz = 70 + 9 * k, 900 + 100 * k
        rows, cols, tperm, _ = otp.coord_graph(*common.random_graph(nodes, nnz, k))
        return ([torch.tensor(a, device=cuda) for a in common.conv_inputs(prob, nodes, nnz, k, np.float32)],
                [torch.tensor(a, device=cuda) for a in ((rows, cols, tperm) if case == "conv_sorted" else (rows, cols))])

    def step(t, index):
        x, y, w = (a.detach().requires_grad_() for a in t[:3])
        z = op(x, y, w, *index)
        return [z.detach(), *torch.autograd.grad(z, (x, y, w), t[3])]
    jobs = [operands(k) for k in (0, 1)]
    for t, index in jobs:                                                   # (workspace, and the choice of the backward)
        step(t, index)
    want = [step(*job) for job in jobs]
    jobs[1][0][1] = torch.stack([jobs[1][0][1]] * 2, -1)[..., 0]            # strided: not for the C++ kernels
    wrong = []

    def work(k):
        for i in range(40):
            for a, b in zip(step(*jobs[k]), want[k]):
                # (an unsorted edge list's sums take the order in which integer atomics land)
                if not (torch.equal(a, b) if case != "conv" else float((a - b).abs().max()) <= 1e-5 * float(b.abs().max())):
                    wrong.append((k, i))
    threads = [threading.Thread(target=work, args=(k,)) for k in (0, 1)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not wrong
