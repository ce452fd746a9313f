"""Per-stream library staging of the reference-layout entry points is
released with its stream (dlm_scratch_release) and does not accumulate a
set per stream (GPU).

The reference's launch_* wrappers cudaMalloc / cudaFree their temporaries
per call (src/kernels/conv2d.cu:362-448, attention.cu); this library keeps
grow-only staging per (device, stream) instead.  A caller that cycles through
streams (a stream per request, a stream pool) gets every byte back by
releasing each stream before destroying it, and results do not depend on
whether a stream's staging was freed and re-created in between.
"""
import ctypes

import pytest
import torch

from dollama_amd import _lib, ops
from tests._util import randn, to_gpu

pytestmark = pytest.mark.gpu


def _held():
    n = ctypes.c_size_t(0)
    fn = _lib.hip_lib().dlm_scratch_bytes
    fn.restype = ctypes.c_int
    assert fn(ctypes.byref(n)) == 0
    return n.value


def _release(stream):
    fn = _lib.hip_lib().dlm_scratch_release
    fn.restype = ctypes.c_int
    assert fn(ctypes.c_void_p(stream.cuda_stream)) == 0, _lib.last_error()


def test_streams_cycled_through_reference_entries_give_memory_back(gpu):
    print("[case] 6 streams x (NCHW conv 320@64x64, [B,H,S,Dh] attention 2x10x1024x64)", flush=True)
    x = to_gpu(randn((1, 320, 64, 64), 1))
    w = to_gpu(randn((320, 320, 3, 3), 2, std=0.02))
    b = to_gpu(randn((320,), 3, std=0.01))
    q, k, v = (to_gpu(randn((2, 10, 1024, 64), s)) for s in (4, 5, 6))
    torch.cuda.synchronize()
    _release(torch.cuda.current_stream())
    base = _held()  # what earlier tests' streams still hold
    outs = []
    streams = [torch.cuda.Stream() for _ in range(6)]
    for st in streams:
        with torch.cuda.stream(st):
            y = torch.empty(1, 320, 64, 64, dtype=torch.float16, device=gpu)
            o = torch.empty(2, 10, 1024, 64, dtype=torch.float16, device=gpu)
            ops.launch_conv2d(x, w, b, y, 1, 320, 64, 64, 320, 3, 3, 1, 1, 1, 1)
            ops.launch_attention(q, k, v, o, 2, 10, 1024, 1024, 64, 0.125)
            outs.append((y, o))
    torch.cuda.synchronize()
    grown = _held()
    assert grown > base, "the calls staged nothing per stream"
    per_stream = (grown - base) / len(streams)
    for st in streams:
        _release(st)
    # (<=: staging of other, older streams may have been dropped at the cap)
    assert _held() <= base, "released streams left staging behind"
    # results are the same on every stream, and again after release
    for y, o in outs[1:]:
        assert torch.equal(y, outs[0][0]) and torch.equal(o, outs[0][1])
    with torch.cuda.stream(streams[0]):
        y = torch.empty_like(outs[0][0])
        ops.launch_conv2d(x, w, b, y, 1, 320, 64, 64, 320, 3, 3, 1, 1, 1, 1)
    torch.cuda.synchronize()
    assert torch.equal(y, outs[0][0])
    _release(streams[0])
    assert _held() <= base
    print(f"[scratch] {per_stream / 2**20:.1f} MiB per stream, all returned", flush=True)


def test_split_workspace_that_cannot_be_had(gpu):
    """A GEMM whose plan splits K runs unsplit when its stream's workspace cannot be allocated: no
    error of the failed allocation is left for the launch to report, and once the stream's state is
    released the split form's bits come back."""
    M, N, K = 144, 1280, 5120
    print(f"[case] linear {M}x{N}x{K} on a stream without a split-K workspace", flush=True)
    x, w = to_gpu(randn((M, K), 7)), to_gpu(randn((N, K), 8, std=K ** -0.5))
    want = ops.linear(x, w)
    torch.cuda.synchronize()
    st = torch.cuda.Stream()
    _release(st)
    try:
        with torch.cuda.stream(st):
            _lib.call("dlm_gemm_set_variant", 1)
            unsplit = ops.linear(x, w)
            _lib.call("dlm_gemm_set_variant", 2)
            held = _held()
            for _ in range(3):
                assert torch.equal(ops.linear(x, w), unsplit)
            assert _held() == held
            st.synchronize()
            _release(st)
            _lib.call("dlm_gemm_set_variant", 0)
            assert torch.equal(ops.linear(x, w), want)
            assert _held() > held
            st.synchronize()
    finally:
        _lib.call("dlm_gemm_set_variant", 0)
        _release(st)


def test_split_workspace_during_another_streams_capture(gpu):
    """A stream gets its split-K workspace while another stream is captured, without disturbing the
    capture; the captured stream itself, which has none, runs unsplit."""
    M, N, K = 144, 1280, 5120
    print(f"[case] linear {M}x{N}x{K} while another stream is captured", flush=True)
    x, w = to_gpu(randn((M, K), 9)), to_gpu(randn((N, K), 10, std=K ** -0.5))
    want = ops.linear(x, w)
    try:
        _lib.call("dlm_gemm_set_variant", 1)
        unsplit = ops.linear(x, w)
    finally:
        _lib.call("dlm_gemm_set_variant", 0)
    ya, yb = torch.empty_like(want), torch.empty_like(want)
    torch.cuda.synchronize()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    _release(a)
    _release(b)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=a):
        ops.linear(x, w, out=ya)
        with torch.cuda.stream(b):
            ops.linear(x, w, out=yb)
    b.synchronize()
    assert torch.equal(yb, want)
    for _ in range(3):
        ya.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(ya, unsplit)
        assert torch.equal(ops.linear(x, w), want)
    _release(b)
