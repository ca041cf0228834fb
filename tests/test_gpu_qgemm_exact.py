"""The multi-row GEMM over f32 activations (qgemm_exact.hip) against 64-bit results.

The bar: x is carried to 2^-23 of each element (the smallest to 2^-38 of their
row's largest) and every sum is f32 over chains of at most 16 MFMA roundings plus
one add per 64 k, so the 2-norm error stays within a few 2^-24 (6e-8) times the
square root of the number of roundings: 1e-6 holds up to K = 8192 with a wide
margin (the one-wave-per-row kernels show 1e-7 to 2e-7 at these sizes)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 1e-6


def _x(m, k, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(m, k, generator=g)
    return x * torch.where(torch.rand(k, generator=g) < 0.02, 30.0, 1.0)  # a few large channels


def _i8(n, k, seed):
    g = torch.Generator().manual_seed(seed)
    w = torch.randint(-128, 128, (n, k), generator=g, dtype=torch.int8)
    return w, (torch.rand(n, generator=g) * 0.01 + 1e-3)


def _rel(got, ref):
    got, ref = got.double(), ref.double()
    return float((got - ref).norm() / ref.norm())


# edges of the 32 / 64 / 128-row and 128 / 256-column tiles, K not a multiple of 64 and of one step,
# split and unsplit K, the forms of xg_plan (small, middle, wide)
SIZES = [(440, 16, 16), (110, 1, 64), (5, 150000, 48), (5, 33, 1408), (6, 70, 4096), (31, 127, 80), (32, 128, 128), (33, 129, 960), (64, 257, 2560), (65, 384, 1056),
         (77, 40, 4864), (200, 1000, 1024), (512, 960, 960), (513, 4100, 208), (1030, 6000, 320)]


@pytest.mark.parametrize("m,n,k", SIZES)
@pytest.mark.parametrize("sdt", [torch.float32, torch.float16])
def test_i8_f32_rows(ops, m, n, k, sdt):
    x = _x(m, k, m * 7 + k)
    w, s = _i8(n, k, n * 3 + k)
    s = s.to(sdt)
    bias = torch.randn(n, generator=torch.Generator().manual_seed(n))
    ref = x.double() @ w.double().t() * s.double() + bias.double()
    y = torch.full((m, n), float("nan"), device="cuda")
    ops.encode_qgemv_i8(w.cuda(), s.cuda(), x.cuda(), y, bias=bias.cuda())
    torch.cuda.synchronize()
    assert _rel(y.cpu(), ref) <= TOL


@pytest.mark.parametrize("m,n,k", [s for s in SIZES if s[2] % 32 == 0])
@pytest.mark.parametrize("spr", [1, 3])  # scales per row; the first one holds for the whole row
def test_i4_f32_rows(ops, m, n, k, spr):
    g = torch.Generator().manual_seed(m + n + k)
    w = torch.randint(0, 256, (n, k // 2), generator=g, dtype=torch.uint8)
    s = (torch.rand(n, spr, generator=g) * 0.01 + 1e-3).half()
    q = torch.stack([w & 15, w >> 4], 2).reshape(n, k).double() - 8
    x = _x(m, k, m + k)
    y = torch.full((m, n), float("nan"), device="cuda")
    ops.encode_qgemv_i4_sym(w.cuda(), s.cuda(), k, x.cuda(), y, k)
    torch.cuda.synchronize()
    assert _rel(y.cpu(), x.double() @ q.t() * s[:, 0].double()) <= TOL


@pytest.mark.parametrize("m,n,k", [s for s in SIZES if s[2] % 32 == 0])
@pytest.mark.parametrize("sdt,group", [(torch.float32, 64), (torch.float16, 64), (torch.bfloat16, 64),
                                       (torch.float32, 128), (torch.float16, 256)])
def test_q4_affine_f32_rows(ops, m, n, k, sdt, group):
    """Group scales and biases in each dtype, groups of one and of several K steps, a last group cut short."""
    g = torch.Generator().manual_seed(m + n + k)
    w = torch.randint(-2**31, 2**31, (n, k // 8), generator=g, dtype=torch.int64).to(torch.int32)
    s = (torch.rand(n, -(-k // group), generator=g) * 0.01 + 1e-3).to(sdt)
    b = (s.float() * (-7.5 + torch.randn(s.shape, generator=g))).to(sdt)
    q = ((w[:, :, None] >> torch.arange(0, 32, 4)) & 15).reshape(n, k).double()
    wide = lambda t: t.double().repeat_interleave(group, 1)[:, :k]
    x = _x(m, k, m + k)
    y = torch.full((m, n), float("nan"), device="cuda")
    ops.encode_qgemv_q4_affine(w.cuda(), s.cuda(), b.cuda(), x.cuda(), y, group=group)
    torch.cuda.synchronize()
    assert _rel(y.cpu(), x.double() @ (q * wide(s) + wide(b)).t()) <= TOL


@pytest.mark.parametrize("m,n,k,gs", [(40, 130, 192, 64), (65, 257, 1056, 192), (300, 384, 2560, 640)])
def test_i4_grouped_f32_rows(ops, m, n, k, gs):
    g = torch.Generator().manual_seed(m + n + k)
    w = torch.randint(0, 256, (n, k // 2), generator=g, dtype=torch.uint8)
    s = (torch.rand(n, -(-k // gs), generator=g) * 0.01 + 1e-3).half()
    q = torch.stack([w & 15, w >> 4], 2).reshape(n, k).double() - 8
    x = _x(m, k, m + k)
    y = torch.full((m, n), float("nan"), device="cuda")
    ops.encode_qgemv_i4_sym(w.cuda(), s.cuda(), gs, x.cuda(), y, k)
    torch.cuda.synchronize()
    assert _rel(y.cpu(), x.double() @ (q * s.double().repeat_interleave(gs, 1)[:, :k]).t()) <= TOL


def test_q4_affine_non_finite(ops):
    """inf and NaN in x, in a group's scale and in its bias reach the outputs of a plain f32 sum."""
    m, n, k = 100, 96, 256
    g = torch.Generator().manual_seed(1)
    w = torch.randint(-2**31, 2**31, (n, k // 8), generator=g, dtype=torch.int64).to(torch.int32)
    s, b = torch.rand(n, 4, generator=g) * 0.01 + 1e-3, torch.randn(n, 4, generator=g) * 0.01
    s[5, 1], b[6, 2], b[7, 0] = float("inf"), float("-inf"), float("nan")
    x = _x(m, k, 2)
    x[3, 77], x[4, 200] = float("inf"), float("nan")
    q = ((w[:, :, None] >> torch.arange(0, 32, 4)) & 15).reshape(n, k).float()
    ref = x @ (q * s.repeat_interleave(64, 1) + b.repeat_interleave(64, 1)).t()
    y = torch.empty(m, n, device="cuda")
    ops.encode_qgemv_q4_affine(w.cuda(), s.cuda(), b.cuda(), x.cuda(), y)
    torch.cuda.synchronize()
    got = y.cpu()
    assert np.array_equal(torch.isnan(got).numpy(), torch.isnan(ref).numpy())
    assert np.array_equal(torch.isposinf(got).numpy(), torch.isposinf(ref).numpy())
    fine = torch.isfinite(ref)
    assert _rel(got[fine], ref[fine]) <= TOL


@pytest.mark.parametrize("m,n,k", SIZES + [(300, 70, 8), (64, 130, 904)])
def test_f16_weights_f32_rows(ops, m, n, k):
    g = torch.Generator().manual_seed(m + n + k)
    w = (torch.randn(n, k, generator=g) * 0.02).half()
    w[0, 0] = 6e-8  # a subnormal weight
    x = _x(m, k, m + k)
    y = torch.full((m, n), float("nan"), device="cuda")
    ops.encode_qgemv_f16(w.cuda(), x.cuda(), y)
    torch.cuda.synchronize()
    assert _rel(y.cpu(), x.double() @ w.double().t()) <= TOL


@pytest.mark.parametrize("k", [840, 2560])  # a ragged last step; split over k
def test_f16_non_finite_weights(ops, k):
    """An infinite weight gives the infinities (and 0 * inf its NaN) of a plain f32 sum, in its own column only."""
    m, n = 10, 70
    x = _x(m, k, 2)
    w = (torch.randn(n, k, generator=torch.Generator().manual_seed(3)) * 0.02).half()
    w[3, k - 1], w[4, 0], w[5, 1], w[5, 2] = float("inf"), float("nan"), float("inf"), float("-inf")
    x[2, k - 1] = 0.0
    x[1, 1], x[1, 2] = 1.0, 1.0
    y = torch.empty(m, n, device="cuda")
    ops.encode_qgemv_f16(w.cuda(), x.cuda(), y)
    torch.cuda.synchronize()
    got, ref = y.cpu(), x @ w.float().t()
    assert np.array_equal(torch.isnan(got).numpy(), torch.isnan(ref).numpy())
    assert np.array_equal(torch.isinf(got).numpy(), torch.isinf(ref).numpy())
    assert torch.equal(torch.sign(got[:, 3]).nan_to_num(), torch.sign(ref[:, 3]).nan_to_num())
    fine = [c for c in range(n) if c not in (3, 4, 5)]
    assert _rel(got[:, fine], x.double() @ w[fine].double().t()) <= TOL


def test_i8_per_tensor_scale_and_row_spread(ops):
    """Rows whose magnitudes lie 2^80 apart (zero and subnormal rows among them) keep their own precision."""
    m, n, k = 40, 130, 192
    x = _x(m, k, 5)
    x *= torch.pow(2.0, torch.linspace(-60, 20, m))[:, None].float()
    x[3] = 0.0
    x[4] = x[4] * 0.0 + 1e-41  # subnormal
    w, _ = _i8(n, k, 6)
    s = torch.tensor([0.0625])
    y = torch.empty(m, n, device="cuda")
    ops.encode_qgemv_i8(w.cuda(), s.cuda(), x.cuda(), y)
    torch.cuda.synchronize()
    ref = x.double() @ w.double().t() * 0.0625
    got = y.cpu().double()
    assert torch.equal(got[3], torch.zeros(n, dtype=torch.float64))
    for r in range(m):
        if r not in (3, 4):
            assert _rel(got[r], ref[r]) <= TOL, r
    assert _rel(got[4], ref[4]) <= 1e-3  # a subnormal has few bits of its own


@pytest.mark.parametrize("k", [832, 2560])  # unsplit and split over k
def test_i8_non_finite_activations(ops, k):
    """inf and NaN reach exactly the outputs they reach in a plain f32 sum, and overflow is an infinity."""
    m, n = 9, 70
    x = _x(m, k, 8)
    x[1, 5], x[2, 7], x[3, 0], x[3, 1] = float("inf"), float("nan"), float("inf"), float("-inf")
    x[4] = 3e38
    w, s = _i8(n, k, 9)
    w[::3, 5] = 0  # inf * 0 = nan
    y = torch.empty(m, n, device="cuda")
    ops.encode_qgemv_i8(w.cuda(), s.cuda(), x.cuda(), y)
    torch.cuda.synchronize()
    ref = (x[:4] @ w.float().t()) * s
    got = y.cpu()
    assert np.array_equal(torch.isnan(got[:4]).numpy(), torch.isnan(ref).numpy())
    assert np.array_equal(torch.isposinf(got[:4]).numpy(), torch.isposinf(ref).numpy())
    assert np.array_equal(torch.isneginf(got[:4]).numpy(), torch.isneginf(ref).numpy())
    big = torch.full((k,), 3e38).double() @ w.double().t()
    far = (big.abs() > 2.0**129)  # overflows f32 in any order of the sum
    assert torch.equal(torch.isfinite(got[4])[far], torch.zeros(int(far.sum()), dtype=torch.bool))
    assert _rel(got[5:], x[5:].double() @ w.double().t() * s.double()) <= TOL


def test_captured_calls_use_no_scratch(ops):
    """Under capture the call takes the kernels without scratch: a replay stays right after later eager calls
    with larger shapes have regrown the workspace."""
    m, n, k = 32, 96, 256
    x, (w, s) = _x(m, k, 1).cuda(), _i8(n, k, 2)
    w, s = w.cuda(), s.cuda()
    y = torch.zeros(m, n, device="cuda")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        ops.encode_qgemv_i8(w, s, x, y, stream=torch.cuda.current_stream())
    big = torch.empty(600, 4096, device="cuda")
    bx, (bw, bs) = _x(600, 512, 3).cuda(), _i8(4096, 512, 4)
    ref = x.cpu().double() @ w.cpu().double().t() * s.cpu().double()
    for _ in range(3):
        y.zero_()
        ops.encode_qgemv_i8(bw.cuda(), bs.cuda(), bx, big, stream=side)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert _rel(y.cpu(), ref) <= TOL


def test_captured_f16_rows_on_a_fresh_stream(ops):
    """int8 over f16 rows whose eager form splits K: a capture on a stream without a workspace allocates none and
    runs unsplit.  One f32 chain of 2560 / 16 MFMA roundings stays within TOL."""
    m, n, k = 129, 200, 2560
    x, (w, s) = _x(m, k, 1).half(), _i8(n, k, 2)
    ref = x.double() @ w.double().t() * s.double()
    wd, sd, xd, y = w.cuda(), s.cuda(), x.cuda(), torch.zeros(m, n, device="cuda")
    ops.encode_qgemm_i8(wd, sd, xd, y)  # the kernels' modules are loaded
    torch.cuda.synchronize()
    assert _rel(y.cpu(), ref) <= TOL
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        ops.encode_qgemm_i8(wd, sd, xd, y, stream=torch.cuda.current_stream())
    for _ in range(3):
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert _rel(y.cpu(), ref) <= TOL


def _q4(n, k, seed, sdt=torch.float32):
    g = torch.Generator().manual_seed(seed)
    w = torch.randint(-2**31, 2**31, (n, k // 8), generator=g, dtype=torch.int64).to(torch.int32)
    s = (torch.rand(n, -(-k // 64), generator=g) * 0.01 + 1e-3).to(sdt)
    b = (s.float() * (-7.5 + torch.randn(s.shape, generator=g))).to(sdt)
    q = ((w[:, :, None] >> torch.arange(0, 32, 4)) & 15).reshape(n, k).double()
    wide = lambda t: t.double().repeat_interleave(64, 1)[:, :k]
    return w.cuda(), s.cuda(), b.cuda(), q * wide(s) + wide(b)


def _i4(n, k, gs, seed):
    g = torch.Generator().manual_seed(seed)
    w = torch.randint(0, 256, (n, k // 2), generator=g, dtype=torch.uint8)
    s = (torch.rand(n, -(-k // gs), generator=g) * 0.01 + 1e-3).half()
    q = torch.stack([w & 15, w >> 4], 2).reshape(n, k).double() - 8
    return w.cuda(), s.cuda(), q * s.double().repeat_interleave(gs, 1)[:, :k]


def _act(g, u, act):
    if act == "silu":
        return g / (1 + torch.exp(-g)) * u
    return 0.5 * g * (1 + torch.tanh(0.7978846 * (g + 0.044715 * g * g * g))) * u


# segments that end inside a tile, one far smaller than a tile; unsplit, split over k, and the wide form
QKV = [(40, 130, 33, 224), (77, 896, 128, 896), (512, 300, 260, 2560), (1030, 2500, 520, 320)]


@pytest.mark.parametrize("m,rq,rkv,k", QKV)
def test_qkv_f32_rows(ops, m, rq, rkv, k):
    x = _x(m, k, m + k)
    rows, xc = (rq, rkv, rkv), x.cuda()
    bias = [torch.randn(r, generator=torch.Generator().manual_seed(r)) for r in rows]
    w = [_i8(r, k, 7 + i) for i, r in enumerate(rows)]
    y = [torch.full((m, r), float("nan"), device="cuda") for r in rows]
    dev = [t.cuda() for ws in w for t in ws]
    ops.encode_qkv_i8(*dev, xc, *y, bq=bias[0].cuda(), bk=None, bv=bias[2].cuda())
    torch.cuda.synchronize()
    for i in range(3):
        ref = x.double() @ w[i][0].double().t() * w[i][1].double() + (bias[i].double() if i != 1 else 0)
        assert _rel(y[i].cpu(), ref) <= TOL, i
    q = [_q4(r, k, 17 + i) for i, r in enumerate(rows)]
    for t in y:
        t.fill_(float("nan"))
    ops.encode_qkv_q4_affine(*q[0][:3], *q[1][:3], *q[2][:3], xc, *y, biasq=bias[0].cuda(), biasv=bias[2].cuda())
    torch.cuda.synchronize()
    for i in range(3):
        assert _rel(y[i].cpu(), x.double() @ q[i][3].t() + (bias[i].double() if i != 1 else 0)) <= TOL, i


@pytest.mark.parametrize("act", ["silu", "gelu"])
@pytest.mark.parametrize("m,n,k", [(40, 70, 224), (77, 33, 896), (200, 4096, 1024), (300, 100, 2560), (1100, 2500, 320)])
def test_gate_up_f32_rows(ops, m, n, k, act):
    """One launch of gate and up with the activation, against the 64-bit sums: act(g) * u carries both sums' errors."""
    x = _x(m, k, m + k) * 0.3
    xc, h = x.cuda(), torch.full((m, n), float("nan"), device="cuda")
    (wg, sg), (wu, su) = _i8(n, k, 1), _i8(n, k, 2)
    sg, su = sg * 0.02, su * 0.02  # sums near 1, where the activation bends
    bg, bu = (torch.randn(n, generator=torch.Generator().manual_seed(i)) for i in (3, 4))
    fn = ops.encode_gate_up_silu_i8 if act == "silu" else ops.encode_gate_up_gelu_i8
    fn(wg.cuda(), sg.cuda(), wu.cuda(), su.cuda(), xc, h, bg=bg.cuda(), bu=bu.cuda())
    torch.cuda.synchronize()
    one = lambda w, s, b: x.double() @ w.double().t() * s.double() + b.double()
    assert _rel(h.cpu(), _act(one(wg, sg, bg), one(wu, su, bu), act)) <= 2 * TOL
    g, u = _q4(n, k, 5), _q4(n, k, 6)
    h.fill_(float("nan"))
    fn = ops.encode_gate_up_silu_q4_affine if act == "silu" else ops.encode_gate_up_gelu_q4_affine
    fn(*g[:3], *u[:3], xc, h)
    torch.cuda.synchronize()
    assert _rel(h.cpu(), _act(x.double() @ g[3].t(), x.double() @ u[3].t(), act)) <= 2 * TOL
    if act == "gelu":
        for gs in (k, 64):
            if gs != k and k % 64:
                continue
            g, u = _i4(n, k, gs, 8), _i4(n, k, gs, 9)
            h.fill_(float("nan"))
            ops.encode_gate_up_gelu_i4_sym(*g[:2], *u[:2], gs, xc, h, k)
            torch.cuda.synchronize()
            assert _rel(h.cpu(), _act(x.double() @ g[2].t(), x.double() @ u[2].t(), act)) <= 2 * TOL, gs


@pytest.mark.parametrize("k", [832, 2560])  # unsplit and split over k
def test_gate_up_non_finite(ops, k):
    m, n = 9, 70
    x = _x(m, k, 8) * 0.3
    x[1, 5], x[2, 7], x[3, 0] = float("inf"), float("nan"), float("-inf")
    (wg, sg), (wu, su) = _i8(n, k, 1), _i8(n, k, 2)
    h = torch.empty(m, n, device="cuda")
    ops.encode_gate_up_silu_i8(wg.cuda(), (sg * 0.02).cuda(), wu.cuda(), (su * 0.02).cuda(), x.cuda(), h)
    torch.cuda.synchronize()
    g, u = ((x @ w.float().t()) * (s * 0.02) for w, s in ((wg, sg), (wu, su)))
    ref, got = g * (1 / (1 + torch.exp(-g))) * u, h.cpu()
    assert np.array_equal(torch.isnan(got).numpy(), torch.isnan(ref).numpy())
    assert np.array_equal(torch.isposinf(got).numpy(), torch.isposinf(ref).numpy())
    assert np.array_equal(torch.isneginf(got).numpy(), torch.isneginf(ref).numpy())
    assert _rel(got[4:], _act(g[4:].double(), u[4:].double(), "silu")) <= 1e-5  # against f32 sums


# f16 activations over int8: products are exact, one f32 chain over K (a rounding per 8 or 16 products):
# sqrt(K / 8) * 2^-24 is 1.9e-6 at K = 8192
@pytest.mark.parametrize("m,n,k", SIZES + [(70, 300, 8192), (2049, 6200, 192), (129, 64, 64)])
@pytest.mark.parametrize("sdt", [torch.float32, torch.bfloat16])
def test_i8_f16_rows(ops, m, n, k, sdt):
    x = _x(m, k, m * 7 + k).half()
    w, s = _i8(n, k, n * 3 + k)
    s = s.to(sdt)
    bias = torch.randn(n, generator=torch.Generator().manual_seed(n))
    ref = x.double() @ w.double().t() * s.double() + bias.double()
    y = torch.full((m, n), float("nan"), device="cuda")
    ops.encode_qgemv_i8(w.cuda(), s.cuda(), x.cuda(), y, bias=bias.cuda())
    torch.cuda.synchronize()
    assert _rel(y.cpu(), ref) <= 2e-6
    if k % 64 == 0:  # the qGEMM entry point takes any number of rows
        for rows in (1, m):
            y.fill_(float("nan"))
            ops.encode_qgemm_i8(w.cuda(), s.cuda(), x[:rows].cuda(), y[:rows], bias=bias.cuda())
            torch.cuda.synchronize()
            assert _rel(y[:rows].cpu(), ref[:rows]) <= 2e-6


@pytest.mark.parametrize("m,rq,rkv,k", [s for s in QKV if s[0] > 64])
def test_qkv_and_gate_up_f16_rows(ops, m, rq, rkv, k):
    x = _x(m, k, m + k).half()
    rows = (rq, rkv, rkv)
    w = [_i8(r, k, 7 + i) for i, r in enumerate(rows)]
    y = [torch.full((m, r), float("nan"), device="cuda") for r in rows]
    ops.encode_qkv_i8(*[t.cuda() for ws in w for t in ws], x.cuda(), *y)
    torch.cuda.synchronize()
    for i in range(3):
        assert _rel(y[i].cpu(), x.double() @ w[i][0].double().t() * w[i][1].double()) <= 2e-6, i
    x = (x * 0.3).half()
    (wg, sg), (wu, su) = _i8(rq, k, 1), _i8(rq, k, 2)
    sg, su = sg * 0.02, su * 0.02
    h = torch.full((m, rq), float("nan"), device="cuda")
    ops.encode_gate_up_silu_i8(wg.cuda(), sg.cuda(), wu.cuda(), su.cuda(), x.cuda(), h)
    torch.cuda.synchronize()
    g, u = (x.double() @ t.double().t() * s.double() for t, s in ((wg, sg), (wu, su)))
    assert _rel(h.cpu(), _act(g, u, "silu")) <= 4e-6


# f16 activations over MLX q4 at more than 64 rows: k % 128 == 0 runs f16 weight tiles (2^-11 per weight, 2e-4 in
# the sum; f32, f16 and bf16 scales), other k the exact nibbles
@pytest.mark.parametrize("m,rq,rkv,k", [(65, 130, 33, 128), (77, 896, 128, 896), (300, 300, 260, 2560), (513, 2500, 520, 384),
                                        (128, 1000, 64, 6400), (77, 896, 128, 960), (200, 300, 40, 1056), (40, 300, 40, 1056)])
@pytest.mark.parametrize("sdt", [torch.float16, torch.float32, torch.bfloat16])
def test_q4_qkv_and_gate_up_f16_rows(ops, m, rq, rkv, k, sdt):
    tol = 5e-4 if k % 128 == 0 else TOL
    x = _x(m, k, m + k).half()
    rows, xc = (rq, rkv, rkv), x.cuda()
    bias = [torch.randn(r, generator=torch.Generator().manual_seed(r)) for r in rows]
    y = [torch.full((m, r), float("nan"), device="cuda") for r in rows]
    q = [_q4(r, k, 17 + i, sdt) for i, r in enumerate(rows)]
    ops.encode_qkv_q4_affine(*q[0][:3], *q[1][:3], *q[2][:3], xc, *y, biasq=bias[0].cuda(), biasv=bias[2].cuda())
    torch.cuda.synchronize()
    for i in range(3):
        assert _rel(y[i].cpu(), x.double() @ q[i][3].t() + (bias[i].double() if i != 1 else 0)) <= tol, i
    x = (x * 0.3).half()
    g, u = _q4(rq, k, 5, sdt), _q4(rq, k, 6, sdt)
    h = torch.full((m, rq), float("nan"), device="cuda")
    for act, fn in (("silu", ops.encode_gate_up_silu_q4_affine), ("gelu", ops.encode_gate_up_gelu_q4_affine)):
        h.fill_(float("nan"))
        fn(*g[:3], *u[:3], x.cuda(), h)
        torch.cuda.synchronize()
        assert _rel(h.cpu(), _act(x.double() @ g[3].t(), x.double() @ u[3].t(), act)) <= 2 * tol, act


# The bar is the error of kernels whose lanes sum a row's products in a tree, on the same x: int8 in calls of four f32
# rows (1.0e-7 to 1.1e-7 here; sums of four 64-k steps 8.2e-8 to 1.1e-7, one chain over K 1.6e-7 to 4.2e-7), q4 the
# single call, which runs one wave per row at k % 64 == 32 (1.3e-7 / 1.6e-7; steps in pairs 9.2e-8 / 1.2e-7, each onto
# the total 1.5e-7 / 2.1e-7)
@pytest.mark.parametrize("m,n,k", [(1100, 2048, 976), (300, 2560, 2032), (1100, 2048, 4080)])
def test_i8_f16_rows_ragged_k_sum_as_well_as_single_rows(ops, m, n, k):
    x = _x(m, k, k).half().cuda()
    w, s = (t.cuda() for t in _i8(n, k, 3))
    ref = torch.matmul(x.double(), w.double().t().contiguous()) * s.double()
    y, rows = (torch.full((m, n), float("nan"), device="cuda") for _ in range(2))
    ops.encode_qgemv_i8(w, s, x, y)
    for r in range(0, m, 4):
        ops.encode_qgemv_i8(w, s, x[r:r + 4].float(), rows[r:r + 4])
    torch.cuda.synchronize()
    assert _rel(y, ref) <= 1.05 * _rel(rows, ref)


@pytest.mark.parametrize("m,n,k", [(300, 2560, 2016), (1100, 2048, 4064)])
def test_q4_f16_rows_ragged_k_sum_as_well_as_single_rows(ops, m, n, k):
    x = _x(m, k, k).half().cuda()
    w, s, b, dense = _q4(n, k, 3)
    ref = torch.matmul(x.double(), dense.cuda().t().contiguous())
    y, rows, *kv = (torch.full((m, n), float("nan"), device="cuda") for _ in range(4))
    ops.encode_qkv_q4_affine(w, s, b, w, s, b, w, s, b, x, y, *kv)
    ops.encode_qgemv_q4_affine(w, s, b, x, rows)
    torch.cuda.synchronize()
    assert _rel(y, ref) <= 1.05 * _rel(rows, ref)
    assert torch.equal(kv[0], y) and torch.equal(kv[1], y)


@pytest.mark.parametrize("m,k", [(9, 832), (70, 2560)])
def test_i4_and_grouped_i4_non_finite(ops, m, k):
    """inf and NaN in x, and in a group's scale, reach exactly the outputs they reach in a plain f32 sum."""
    n = 70
    x = _x(m, k, 8)
    x[1, 5], x[2, 7], x[3, 0], x[3, 1] = float("inf"), float("nan"), float("inf"), float("-inf")
    for gs in (k, 64):
        w, s, _ = _i4(n, k, gs, 9)
        if gs != k:
            s[4, 2], s[5, 3] = float("inf"), float("nan")
        w[::3, 2] |= 0x80  # k = 5 of these rows: q - 8 = 0
        w[::3, 2] &= 0x8F
        q = torch.stack([w.cpu() & 15, w.cpu() >> 4], 2).reshape(n, k).float() - 8
        dense = q * s.cpu().float().repeat_interleave(gs, 1)[:, :k]
        y = torch.empty(m, n, device="cuda")
        ops.encode_qgemv_i4_sym(w, s, gs, x.cuda(), y, k)
        torch.cuda.synchronize()
        got, ref = y.cpu(), (x[:, None] * dense[None]).sum(2)
        for f in (torch.isnan, torch.isposinf, torch.isneginf):
            assert torch.equal(f(got), f(ref)), (gs, f)
        fine = torch.isfinite(ref)
        assert _rel(got[fine], ref[fine]) <= 1e-5  # against f32 sums


@pytest.mark.parametrize("m,k", [(70, 832), (70, 840), (300, 2560)])  # in place and padded
def test_i8_f16_rows_non_finite(ops, m, k):
    n = 70
    x = _x(m, k, 8).half()
    x[1, 5], x[2, 7], x[3, 0], x[3, 1] = float("inf"), float("nan"), float("inf"), float("-inf")
    w, s = _i8(n, k, 9)
    w[::3, 5] = 0
    y = torch.empty(m, n, device="cuda")
    ops.encode_qgemv_i8(w.cuda(), s.cuda(), x.cuda(), y)
    torch.cuda.synchronize()
    got, ref = y.cpu(), (x.float()[:, None] * w.float()[None]).sum(2) * s
    for f in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(f(got), f(ref)), f
    fine = torch.isfinite(ref)
    assert _rel(got[fine], ref[fine]) <= 1e-5


# the time of a call in times of the finite call.  One infinite weight (a column of outputs again): 9 (f16) and 20 (q4)
# where the sums took an element at a time; an infinity in every row of x (every output again): 230 and 580, int8, which
# needs no second sum, 170
@pytest.mark.parametrize("fmt,one,all_", [("f16", 6, 60), ("q4", 10, 100), ("i8", 2, 2)])
def test_non_finite_inputs_in_bounded_time(ops, fmt, one, all_):
    m, n, k = 512, 2048, 2048
    g = torch.Generator(device="cuda").manual_seed(1)
    x, y = torch.randn(m, k, generator=g, device="cuda"), torch.empty(m, n, device="cuda")
    if fmt == "f16":
        w = (torch.randn(n, k, generator=g, device="cuda") * 0.02).half()
        call, poison = lambda v: ops.encode_qgemv_f16(w, v, y), lambda: w[3, 7].fill_(float("inf"))
    elif fmt == "q4":
        w, s, b, _ = _q4(n, k, 3)
        call, poison = lambda v: ops.encode_qgemv_q4_affine(w, s, b, v, y), lambda: s[3, 0].fill_(float("inf"))
    else:
        w, s = (t.cuda() for t in _i8(n, k, 3))
        call, poison = lambda v: ops.encode_qgemv_i8(w, s, v, y), lambda: s[3].fill_(float("inf"))

    def time(v):
        call(v)
        best = float("inf")
        for _ in range(3):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(5):
                call(v)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    fine = time(x)
    bad = x.clone()
    bad[:, 7] = float("inf")
    every = time(bad)
    assert not bool(torch.isfinite(y).any()) and every <= all_ * fine, (every, fine)
    poison()
    column = time(x)
    assert not bool(torch.isfinite(y[:, 3]).any()) and column <= one * fine, (column, fine)


def _wide(fmt, n, k):
    """One matrix: its call over x and y, and its dense 64-bit weights."""
    if fmt in ("i8", "i8 f16 x"):
        w, s = (t.cuda() for t in _i8(n, k, 3))
        return (lambda ops, x, y: ops.encode_qgemv_i8(w, s, x, y)), lambda: w.double() * s.double()[:, None]
    if fmt == "f16":
        w = (torch.randn(n, k, generator=torch.Generator().manual_seed(3)) * 0.02).half().cuda()
        return (lambda ops, x, y: ops.encode_qgemv_f16(w, x, y)), lambda: w.double()
    if fmt == "i4":
        w, s, dense = _i4(n, k, k, 3)
        return (lambda ops, x, y: ops.encode_qgemv_i4_sym(w, s, k, x, y, k)), lambda: dense.cuda()
    w, s, b, dense = _q4(n, k, 3)
    return (lambda ops, x, y: ops.encode_qgemv_q4_affine(w, s, b, x, y)), lambda: dense.cuda()


# the tile heights of few rows over outputs wide enough for the tallest (int8 over f16 x: k not a multiple of 64)
@pytest.mark.parametrize("fmt,k", [("i8", 96), ("i8 f16 x", 112), ("f16", 96), ("i4", 96), ("q4", 160)])
@pytest.mark.parametrize("m", [32, 33, 64, 65])
def test_few_rows_of_wide_outputs(ops, fmt, k, m):
    n = 50100
    call, dense = _wide(fmt, n, k)
    x = _x(m, k, m).cuda()
    x = x.half() if fmt == "i8 f16 x" else x
    y = torch.full((m, n), float("nan"), device="cuda")
    call(ops, x, y)
    torch.cuda.synchronize()
    assert _rel(y, torch.matmul(x.double(), dense().t().contiguous())) <= TOL


@pytest.mark.parametrize("fmt", ["i8", "f16", "i4", "q4"])
def test_five_rows_of_a_wide_output_take_less_than_128(ops, fmt):
    n, k = 131072, 1152
    call, _ = _wide(fmt, n, k)
    x, y = _x(128, k, 1).cuda(), torch.empty(128, n, device="cuda")

    def time(rows):
        call(ops, x[:rows], y[:rows])
        best = float("inf")
        for _ in range(3):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(5):
                call(ops, x[:rows], y[:rows])
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    few, many = time(5), time(128)
    assert few <= 0.7 * many, (few, many)  # 0.3 to 0.6; 0.8 to 0.9 in tiles of 128 rows


# the tallest tiles (192 of them and more): several matrices, the activation in the epilogue, a padded last step
@pytest.mark.parametrize("m,n,k,x_f16", [(1100, 2900, 320, False), (2049, 3300, 192, True), (1100, 2900, 336, True)])
def test_gate_up_i8_tall_tiles(ops, m, n, k, x_f16):
    x = _x(m, k, 8).cuda() * 0.3
    x = x.half() if x_f16 else x
    (wg, sg), (wu, su) = ((w.cuda(), s.cuda() * 0.02) for w, s in (_i8(n, k, 1), _i8(n, k, 2)))
    h = torch.full((m, n), float("nan"), device="cuda")
    ops.encode_gate_up_silu_i8(wg, sg, wu, su, x, h)
    torch.cuda.synchronize()
    g, u = (torch.matmul(x.double(), w.double().t().contiguous()) * s.double() for w, s in ((wg, sg), (wu, su)))
    assert _rel(h, _act(g, u, "silu")) <= 2 * TOL


@pytest.mark.parametrize("m,n,k", [(1100, 2900, 320), (1100, 2900, 352)])
def test_q4_and_i4_tall_tiles(ops, m, n, k):
    x = _x(m, k, 8).cuda() * 0.3
    h = torch.full((m, n), float("nan"), device="cuda")
    one = lambda w, x: torch.matmul(x.double(), w.cuda().t().contiguous())
    for v in (x, x.half()):
        if v.dtype == torch.float16 and k % 128 == 0:
            continue
        g, u = _q4(n, k, 5), _q4(n, k, 6)
        h.fill_(float("nan"))
        ops.encode_gate_up_silu_q4_affine(*g[:3], *u[:3], v, h)
        torch.cuda.synchronize()
        assert _rel(h, _act(one(g[3], v), one(u[3], v), "silu")) <= 2 * TOL, v.dtype
    g, u = _i4(n, k, k, 8), _i4(n, k, k, 9)
    h.fill_(float("nan"))
    ops.encode_gate_up_gelu_i4_sym(*g[:2], *u[:2], k, x, h, k)
    torch.cuda.synchronize()
    assert _rel(h, _act(one(g[2], x), one(u[2], x), "gelu")) <= 2 * TOL


@pytest.mark.parametrize("m,rq,rkv,k,x_f16", [(1030, 4000, 700, 320, False), (2049, 4000, 700, 128, True),
                                              (1100, 4000, 700, 976, True)])
def test_qkv_i8_tall_tiles(ops, m, rq, rkv, k, x_f16):
    x = _x(m, k, k).cuda()
    x = x.half() if x_f16 else x
    rows = (rq, rkv, rkv)
    w = [tuple(t.cuda() for t in _i8(r, k, 7 + i)) for i, r in enumerate(rows)]
    y = [torch.full((m, r), float("nan"), device="cuda") for r in rows]
    ops.encode_qkv_i8(*[t for ws in w for t in ws], x, *y)
    torch.cuda.synchronize()
    for i in range(3):
        assert _rel(y[i], torch.matmul(x.double(), w[i][0].double().t().contiguous()) * w[i][1].double()) <= TOL, i
