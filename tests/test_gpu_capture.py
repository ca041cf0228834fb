"""Graph capture and the context's per-stream scratch: a graph keeps the address of the scratch that its calls
used, so that memory stays allocated when a later call needs more, and every replay gives the eager result."""
from __future__ import annotations

import pytest
import torch

from cellm_amd import HipOps
from cellm_amd._lib import CellmHipError

pytestmark = pytest.mark.gpu


@pytest.fixture
def own():
    """A context of its own: no scratch of other tests."""
    o = HipOps(0)
    yield o
    torch.cuda.synchronize()
    o.close()


def _i8(n, k, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randint(-128, 128, (n, k), generator=g, device="cuda", dtype=torch.int8),
            torch.rand(n, generator=g, device="cuda") * 0.01 + 1e-3)


def _q4(n, k, seed, dtype=torch.float16):
    g = torch.Generator(device="cuda").manual_seed(seed)
    w = torch.randint(-2**31, 2**31, (n, k // 8), generator=g, device="cuda", dtype=torch.int64).to(torch.int32)
    s = (torch.rand(n, k // 64, generator=g, device="cuda") * 0.01 + 1e-3).to(dtype)
    return w, s, (s.float() * -7.5).to(dtype)


def _x(m, k, seed, dtype=torch.float32):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(m, k, generator=g, device="cuda").to(dtype)


def _capture(stream, call):
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        call(torch.cuda.current_stream())
    return graph


def _replays(graph, y, ref, between=lambda: None):
    for _ in range(3):
        y.zero_()
        between()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ref)


def test_scratch_of_a_graph_outlives_a_grow(own):
    """A split q4 qGEMM is captured; an eager f32 call on that stream then needs more scratch.  The grow takes new
    memory and keeps the old: the free memory tells, before a replay could write to it."""
    side = torch.cuda.Stream()
    (w8, s8), (wq, s, b) = _i8(64, 8192, 1), _q4(896, 4864, 2)
    x = _x(128, 4864, 3, torch.float16)
    small, large = _x(1024, 8192, 4), _x(2048, 8192, 5)
    y, y8 = torch.zeros(128, 896, device="cuda"), torch.zeros(2048, 64, device="cuda")
    gemm = lambda st: own.encode_qgemm_q4_affine(wq, s, b, x, y, stream=st)
    rows = lambda v, st: own.encode_qgemv_i8(w8, s8, v, y8[:v.shape[0]], stream=st)
    rows(large, torch.cuda.current_stream())  # the kernels' modules are loaded, another stream's scratch taken
    rows(small, side)                         # 1024 rows of two f16 parts: 32 MiB on this stream
    gemm(side)
    torch.cuda.synchronize()
    ref = y.clone()
    graph = _capture(side, gemm)
    before = torch.cuda.mem_get_info()[0]
    rows(large, side)                         # 64 MiB
    torch.cuda.synchronize()
    assert before - torch.cuda.mem_get_info()[0] >= 60 * 2**20  # 32 MiB where the old scratch was freed
    _replays(graph, y, ref, lambda: rows(large, side))


def test_call_short_of_scratch_is_refused_and_the_capture_goes_on(own):
    side = torch.cuda.Stream()
    wq, s, b = _q4(896, 4864, 2)
    x, y = _x(128, 4864, 3, torch.float16), torch.zeros(128, 896, device="cuda")
    g, up = _x(16, 64, 6), _x(16, 64, 7)
    own.encode_qgemm_q4_affine(wq, s, b, x, y)  # the scratch of another stream
    h = g.clone()
    own.encode_silu_mul(h, up)
    ref = h.clone()

    def calls(st):
        with pytest.raises(CellmHipError, match="scratch"):
            own.encode_qgemm_q4_affine(wq, s, b, x, y, stream=st)
        h.copy_(g)
        own.encode_silu_mul(h, up, stream=st)

    _replays(_capture(side, calls), h, ref)


def _i4(n, k, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randint(0, 256, (n, k // 2), generator=g, device="cuda", dtype=torch.uint8),
            (torch.rand(n, 1, generator=g, device="cuda") * 0.01 + 1e-3).half())


M, N, K = 77, 200, 960  # k % 128 == 64: q4 over f16 rows takes the GEMM that needs scratch


def _gate_up_i8(ops, x, y):
    g, u = _i8(N, K, 1), _i8(N, K, 2)
    return lambda st: ops.encode_gate_up_silu_i8(*g, *u, x, y, stream=st)


def _gate_up_q4(ops, x, y):
    g, u = _q4(N, K, 1, x.dtype), _q4(N, K, 2, x.dtype)
    return lambda st: ops.encode_gate_up_silu_q4_affine(*g, *u, x, y, stream=st)


def _gate_up_i4(ops, x, y):
    g, u = _i4(N, K, 1), _i4(N, K, 2)
    return lambda st: ops.encode_gate_up_gelu_i4_sym(*g, *u, K, x, y, K, stream=st)


def _qkv_q4(ops, x, y):
    w = [t for i, n in enumerate((N - 80, 40, 40)) for t in _q4(n, K, 3 + i, x.dtype)]
    q, k, v = (t.view(M, -1) for t in y.view(-1).split([M * (N - 80), M * 40, M * 40]))
    return lambda st: ops.encode_qkv_q4_affine(*w, x, q, k, v, stream=st)


def _qkv_i8(ops, x, y):
    w = [t for i, n in enumerate((N - 80, 40, 40)) for t in _i8(n, K, 3 + i)]
    q, k, v = (t.view(M, -1) for t in y.view(-1).split([M * (N - 80), M * 40, M * 40]))
    return lambda st: ops.encode_qkv_i8(*w, x, q, k, v, stream=st)


def _one_i8(ops, x, y):
    w = _i8(N, K, 9)
    return lambda st: ops.encode_qgemv_i8(*w, x, y, stream=st)


def _one_i4(ops, x, y):
    w = _i4(N, K, 9)
    return lambda st: ops.encode_qgemv_i4_sym(*w, K, x, y, K, stream=st)


def _one_f16(ops, x, y):
    w = _x(N, K, 9, torch.float16)
    return lambda st: ops.encode_qgemv_f16(w, x, y, stream=st)


@pytest.mark.parametrize("make,dtype", [(_gate_up_i8, torch.float32), (_gate_up_q4, torch.float32),
                                        (_gate_up_i4, torch.float32), (_gate_up_q4, torch.float16),
                                        (_gate_up_i8, torch.float16), (_qkv_q4, torch.float16),
                                        (_qkv_q4, torch.float32), (_qkv_i8, torch.float32),
                                        (_one_i8, torch.float32), (_one_i4, torch.float32),
                                        (_one_f16, torch.float32)])
def test_one_eager_call_makes_the_capture_possible_and_equal(own, make, dtype):
    """The scratch of one eager call on the capture stream is all that the capture of that call needs, and the
    graph runs the same launches."""
    y = torch.zeros(M, N, device="cuda")
    call, side = make(own, _x(M, K, 5, dtype) * 0.1, y), torch.cuda.Stream()
    torch.cuda.synchronize()
    call(side)
    torch.cuda.synchronize()
    ref = y.clone()
    assert bool(ref.any())
    _replays(_capture(side, call), y, ref)


@pytest.mark.parametrize("warm", [False, True])  # first scratch of the stream; a grow
def test_scratch_grows_beside_the_capture_of_another_stream(own, warm):
    """An eager call that needs scratch runs while another stream is captured in torch's (global) mode, and the
    capture goes on."""
    w, s = _i8(64, 512, 1)
    x, y = _x(64, 512, 2), torch.zeros(64, 64, device="cuda")
    h, up = _x(16, 64, 6), _x(16, 64, 7)
    src, other = h.clone(), torch.cuda.Stream()
    own.encode_silu_mul(h, up)
    ref = h.clone()
    own.encode_qgemv_i8(w, s, x, y)  # scratch of the current stream
    expected = y.clone()
    if warm:
        own.encode_qgemv_i8(w, s, x[:32], y[:32], stream=other)
    y.zero_()

    def calls(st):
        h.copy_(src)
        own.encode_qgemv_i8(w, s, x, y, stream=other)
        own.encode_silu_mul(h, up, stream=st)

    graph = _capture(torch.cuda.Stream(), calls)
    torch.cuda.synchronize()
    assert torch.equal(y, expected)
    _replays(graph, h, ref)
