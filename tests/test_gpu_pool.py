"""Graphs built, fitted and released again and again on several threads and
streams share freed device memory: results stay right, the memory is given
back on trim, and a release is safe while a stream is captured."""

import ctypes
import threading

import numpy as np
import pytest
import torch

from oracle import c_oracle as C
from commonnnclustering_amd import _lib, engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(900, 4000, 900, 2500), (3000, 3000, 3000, 3000)])
def test_reuse_across_threads_and_streams(cuda, sizes):
    rng = np.random.default_rng(1)
    data = [rng.normal(size=(n, 3)) for n in sizes]
    want = [[C.fit(x, r, 4, member_cutoff=3) for r in (0.3, 0.2)] for x in data]
    errors = []

    def work(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for rep in range(6):
                    i = (k + rep) % len(data)
                    X = torch.from_numpy(data[i]).cuda()
                    g = engine.build_graph(X, 0.09, "f32_band")
                    h = g.rethreshold(0.04)
                    g_lab = g.fit(6, 5, member_cutoff=3)[0].cpu().numpy()
                    g.release()
                    h_lab = h.fit(6, 5, member_cutoff=3)[0].cpu().numpy()
                    h.release()
                    assert (g_lab == want[i][0]).all() and (h_lab == want[i][1]).all()
        except BaseException as e:  # noqa: BLE001 (reported by the test thread)
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[0]


def test_trim_gives_the_memory_back(cuda):
    ctx = _lib.get_context(torch.device("cuda", 0))
    X = torch.from_numpy(np.random.default_rng(2).normal(size=(100_000, 3))).cuda()
    engine.build_graph(X, 0.01).release()
    ctx.trim()
    before = torch.cuda.mem_get_info()[0]
    engine.build_graph(X, 0.04).release()
    ctx.trim()
    assert torch.cuda.mem_get_info()[0] >= before - (64 << 20)


@pytest.mark.parametrize("mode", [0, 1])
def test_release_while_a_stream_is_captured(cuda, mode):
    """A thread that captures a stream (globally, or for itself) may not wait for the
    device.  A graph released then is freed: it must not enter the pool unwaited.
    (The refused wait invalidates the capture, as documented for HIP.)"""
    hip = ctypes.CDLL("libamdhip64.so")
    hip.hipStreamBeginCapture.argtypes = [ctypes.c_void_p, ctypes.c_int]
    hip.hipStreamEndCapture.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_void_p)]
    hip.hipGraphDestroy.argtypes = [ctypes.c_void_p]
    ctx = _lib.get_context(torch.device("cuda", 0))
    X = torch.from_numpy(np.random.default_rng(3).normal(size=(200_000, 3))).cuda()
    engine.build_graph(X, 0.04).release()
    ctx.trim()
    graph = engine.build_graph(X, 0.04)
    ctx.trim()
    size = graph.nbytes
    assert size > 64 << 20
    stream, recorded = torch.cuda.Stream(), ctypes.c_void_p()
    torch.cuda.synchronize()
    held = torch.cuda.mem_get_info()[0]
    assert hip.hipStreamBeginCapture(stream.cuda_stream, mode) == 0
    graph.release()
    if hip.hipStreamEndCapture(stream.cuda_stream, ctypes.byref(recorded)) == 0:
        hip.hipGraphDestroy(recorded)
    hip.hipGetLastError()
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] > held + size // 2
    want = engine.fit(X, 0.04, 5, 4)[0]
    assert (engine.build_graph(X, 0.04).fit(5, 4)[0] == want).all()
