"""A graph captured around a dispatch on a plain backend keeps its split-K scratch
when later eager calls outgrow it: its replays give the eager bits, and memory
allocated since is left alone."""
import numpy as np
import pytest

from conftest import to_dev
from hologram_amd import DTYPE_BF16, BufferRef, DeviceWorkspace, HipBackend, KernelCall, MatMulCall

pytestmark = pytest.mark.gpu


def product(torch, rng, m, k, n):
    ws = DeviceWorkspace()
    a, b = ((rng.standard_normal(x).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
            for x in (m * k, k * n))
    for s, x in enumerate((a, b)):
        ws.bind(s, to_dev(torch, x))
    out = torch.zeros(m * n, dtype=torch.int16, device="cuda")
    ws.bind(2, out)
    return ws, out, KernelCall.MatMul(MatMulCall(BufferRef(0), BufferRef(1), BufferRef(2), m, k, n, DTYPE_BF16))


def test_scratch_outgrown_after_a_capture_stays_with_the_graph(torch_cuda):
    torch, rng = torch_cuda, np.random.default_rng(1)
    small, sout, scall = product(torch, rng, 8, 2048, 1024)
    stream = torch.cuda.Stream()
    be = HipBackend(stream=stream.cuda_stream)
    torch.cuda.synchronize()
    be.dispatch(scall, small)
    be.synchronize()
    want = sout.cpu()
    assert want.any()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        be.dispatch(scall, small)
    for m, k, n in ((16, 8192, 4096), (64, 8192, 8192)):      # each needs more than the one before
        ws, out, call = product(torch, rng, m, k, n)
        be.dispatch(call, ws)
        be.synchronize()
        first = out.cpu()
        new = [torch.full((1 << 18,), 7, dtype=torch.int32, device="cuda") for _ in range(16)]
        for _ in range(2):
            sout.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(sout.cpu(), want)
            assert all(bool((x == 7).all()) for x in new)
        be.dispatch(call, ws)
        be.synchronize()
        assert torch.equal(out.cpu(), first)
    del graph
    be.close()
