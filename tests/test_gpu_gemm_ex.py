"""f32 activations on the f16 matrix cores (k_gemm_ex.hip): every format,
plain and gate/up, against the f64 product with the library's f32
dequantization (pinned bit-exact elsewhere).

Bound: relative error of the whole result (2-norm) <= 2e-7.  The scalar f32
kernel it replaces measures 1.18e-7 .. 1.37e-7 over N(0, 1) rows, K = 1024 ..
17408, this one 0.67e-7 .. 1.0e-7; the reference's own f32-rounded weights add
about 4e-8.  Covered: the edges of the stacked forms (8 / 9, 16 / 17 rows),
whole and partial row groups, ragged outputs, one chunk and several K splits,
bf16 output, rows of very large, very small and non-finite values, every bit
of x, values beside outliers, captured calls (the eager call's bits, warmed up
or not), graphs beside each other and beside eager calls, and calls on two
streams.
"""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import activations, q6k_bytes, rand_qlin_fast, weight_bytes

pytestmark = pytest.mark.gpu

thq = pytest.importorskip("thq")
FORMATS = ["q8_0", "q4_k", "q6_k", "affine"]


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.init()
    yield
    torch.cuda.synchronize()


@pytest.fixture(autouse=True)
def _route(monkeypatch):
    monkeypatch.setenv("THQ_GEMM_EX", "1")  # small calls too


def weight(fmt, n, k, ctx=None):
    if fmt == "affine":
        wq, sb = rand_qlin_fast(n, k, seed=n + k)
        return thq.QTensor.from_affine(wq, sb, n, k, ctx=ctx)
    if fmt == "q6_k":
        return thq.QTensor.from_gguf_bytes(thq.Q6_K, q6k_bytes(n, k, seed=3), n, k, ctx=ctx)
    qt = O.Q8_0 if fmt == "q8_0" else O.Q4_K
    return thq.QTensor.from_gguf_bytes(qt, weight_bytes(qt, n, k, seed=3), n, k, ctx=ctx)


def rows(m, k, seed=0):
    return torch.from_numpy(activations(m, k, seed=seed)).cuda()


def rel(y, ref):
    return float((y.double() - ref).norm() / ref.norm())


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("m,n,k", [(2, 40, 256), (8, 96, 512), (9, 130, 768), (16, 300, 1792), (17, 512, 1024), (33, 257, 2048), (70, 1000, 4096),
                                   (3, 96, 17408)])
def test_rows_match_f64(fmt, m, n, k):
    w, x = weight(fmt, n, k), rows(m, k)
    ref = x.double() @ w.dequantize().double().T
    assert rel(thq.matmul(w, x, torch.float32), ref) <= 2e-7
    assert rel(thq.matmul(w, x, torch.bfloat16), ref) <= 2e-3  # bf16 rounding of the result: 2^-9 / sqrt(3)


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("m,h,k", [(5, 96, 512), (40, 200, 1792)])
def test_gate_up(fmt, m, h, k, monkeypatch):
    w, x = weight(fmt, 2 * h, k), rows(m, k, seed=4)
    y = thq.gate_up_silu(w, x, torch.float32)
    monkeypatch.setenv("THQ_GEMM_EX", "0")
    ref = thq.gate_up_silu(w, x, torch.float32)
    # both round their gate and up sums to bf16: equal but where a sum lies between two neighbours
    assert rel(y, ref.double()) <= 1e-3
    assert float((y != ref).float().mean()) <= 0.02


def test_q6k_single_row():
    w, x = weight("q6_k", 130, 512), rows(1, 512)
    assert rel(thq.matmul(w, x, torch.float32), x.double() @ w.dequantize().double().T) <= 2e-7


@pytest.mark.parametrize("m", [6, 40])
@pytest.mark.parametrize("fmt", FORMATS)
def test_extreme_rows(fmt, m):
    n, k = 64, 512
    w, x = weight(fmt, n, k), rows(m, k, seed=7)
    x[0] *= 1e30
    x[1] *= 1e-33
    x[2] = 0.0
    x[3, 5] = 3e4 * x[3].abs().max()
    ref = x.double() @ w.dequantize().double().T
    y = thq.matmul(w, x, torch.float32)
    for i in (0, 1, 3, 4):
        assert rel(y[i], ref[i]) <= 3e-7, i
    assert not y[2].any()
    x[1, 9] = float("inf")
    x[4, 300] = float("nan")
    z = thq.matmul(w, x, torch.float32)
    wd = w.dequantize()
    assert z[4].isnan().all()
    assert torch.equal(z[1][wd[:, 9] != 0], torch.sign(wd[:, 9][wd[:, 9] != 0]) * float("inf"))
    keep = [i for i in range(m) if i not in (1, 4)]
    assert torch.equal(z[keep], y[keep])


def wide_rows(m, k, seed):
    """Rows of every spread: N(0, 1), up to 1e+-5 and 1e+-35 in one row, and a few values of 1e-12 and 1e9 beside N(0, 1)."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn((m, k), generator=g)
    ten = torch.rand((m, k), generator=g) * 2 - 1
    x[1::4] *= 10 ** (5 * ten[1::4])
    x[2::4] *= 10 ** (35 * ten[2::4])
    few = torch.rand((m, k), generator=g)
    x[3::4][few[3::4] < 4 / k] *= 1e9
    x[3::4][few[3::4] > 1 - 8 / k] *= 1e-12
    x[0, :7] = torch.tensor([0.0, -0.0, 1e-45, -1e-38, 3e38, 1.0, 2.0**-149])
    return x.cuda()


@pytest.mark.parametrize("m", [2, 5, 8, 12, 16, 40])
def test_every_bit_of_x(m):
    """An identity weight (Q8_0: d = 1, one code of 1 per row) returns x itself."""
    n = k = 768
    blk = np.zeros((n, k // 32, 34), np.uint8)
    blk[:, :, :2] = np.array([1.0], np.float16).view(np.uint8)
    blk[np.arange(n), np.arange(n) // 32, 2 + np.arange(n) % 32] = 1
    w = thq.QTensor.from_gguf_bytes(O.Q8_0, blk.reshape(n, -1), n, k)
    for seed in range(3):
        x = wide_rows(m, k, seed)
        assert torch.equal(thq.matmul(w, x, torch.float32), x)


@pytest.mark.parametrize("m", [5, 12, 40])
@pytest.mark.parametrize("fmt", FORMATS)
def test_values_beside_outliers(fmt, m, monkeypatch):
    """Each output against the size of its own products, not the row's: what an outlier adds where its weight is
    small is no more than a f32 dot's rounding of the products that are there.  The bound is four times the scalar
    kernel's largest error (4.0e-7 .. 5.5e-7; this one measures 5.2e-7 .. 1.02e-6)."""
    n, k = 768, 1024
    w, x = weight(fmt, n, k), wide_rows(m, k, seed=50)
    x[0, 4] = 1.0  # 3e38 would overflow the products
    x[2::4] *= 1e-2
    wd = w.dequantize().double()
    ref = x.double() @ wd.T
    size = (x.double().square() @ wd.square().T).sqrt()
    err = {}
    for v in ("0", "1"):
        monkeypatch.setenv("THQ_GEMM_EX", v)
        err[v] = float(((thq.matmul(w, x, torch.float32).double() - ref).abs() / size).max())
    print(f"[outliers] {fmt} m={m}: scalar {err['0']:.3g} planes {err['1']:.3g}", flush=True)
    assert err["1"] <= 4 * err["0"]


def captured(w, x, out, s):
    g = torch.cuda.CUDAGraph()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s), torch.cuda.graph(g, stream=s):
        thq.matmul(w, x, out=out)
    return g


def test_capture_takes_the_eager_kernel():
    """A captured call runs the eager call's kernels (its bits), warmed up on its stream, on another, or not at all."""
    ctx = thq.Context(0)
    w, x = weight("q4_k", 256, 1024, ctx), rows(5, 1024)
    out = torch.empty((5, 256), device="cuda")
    s = torch.cuda.Stream()
    gs = [captured(w, x, out, s)]  # the context's first call
    ref = thq.matmul(w, x, torch.float32)  # warm on the default stream
    gs.append(captured(w, x, out, s))
    with torch.cuda.stream(s):
        s.wait_stream(torch.cuda.default_stream())
        thq.matmul(w, x[:2], torch.float32)  # the stream's own scratch is then too small for x
    gs.append(captured(w, x, out, s))
    for g in gs:
        for _ in range(3):
            out.fill_(float("nan"))
            torch.randn(64, 64, device="cuda") @ torch.randn(64, 64, device="cuda")
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, ref)


def test_capture_without_scratch(monkeypatch):
    """Past the bound on graph scratch a captured call runs the scalar kernel, which needs none."""
    ctx = thq.Context(0)
    w, x = weight("q4_k", 256, 1024, ctx), rows(5, 1024)
    with monkeypatch.context() as mp:
        mp.setenv("THQ_GEMM_EX", "0")
        ref = thq.matmul(w, x, torch.float32)
    monkeypatch.setenv("THQ_GRAPH_SCRATCH_MB", "0")
    out = torch.empty_like(ref)
    g = captured(w, x, out, torch.cuda.Stream())
    for _ in range(3):
        out.fill_(float("nan"))
        torch.randn(64, 64, device="cuda") @ torch.randn(64, 64, device="cuda")
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)


def test_graphs_beside_each_other_and_eager_calls():
    """Graphs captured on one stream, replayed on others beside eager calls on that stream: every call's own bits."""
    w = weight("q4_k", 2048, 1024)
    xs = [rows(40, 1024, seed=40 + i) for i in range(3)]
    ref = [thq.matmul(w, x, torch.float32) for x in xs]
    torch.cuda.synchronize()
    cap, others = torch.cuda.Stream(), [torch.cuda.Stream() for _ in range(2)]
    out = [torch.empty_like(ref[0]) for _ in range(2)]
    graphs = [captured(w, x, y, cap) for x, y in zip(xs, out)]
    torch.cuda.synchronize()
    kept, eager = [[], []], []
    for _ in range(30):
        for i, s in enumerate(others):
            with torch.cuda.stream(s):
                graphs[i].replay()
                kept[i].append(out[i].clone())
        with torch.cuda.stream(cap):
            eager.append(thq.matmul(w, xs[2], torch.float32))
    torch.cuda.synchronize()
    for i in range(2):
        assert all(torch.equal(y, ref[i]) for y in kept[i])
    assert all(torch.equal(y, ref[2]) for y in eager)


def test_rule(monkeypatch):
    monkeypatch.delenv("THQ_GEMM_EX")
    w = weight("q4_k", 4096, 4096)
    assert thq.call_scratch_bytes(w, 2, x_dtype=torch.float32) == 0  # the scalar kernel
    assert thq.call_scratch_bytes(w, 3, x_dtype=torch.float32) > 0


def test_two_streams():
    """f32 calls of one context on two streams do not share scratch."""
    w = weight("q4_k", 2048, 1024)
    xs = [rows(40, 1024, seed=20 + i) for i in range(2)]
    ref = [thq.matmul(w, x, torch.float32) for x in xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in xs]
    out = [[], []]
    for _ in range(8):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                out[i].append(thq.matmul(w, xs[i], torch.float32))
    torch.cuda.synchronize()
    for i in range(2):
        assert all(torch.equal(y, ref[i]) for y in out[i])


def test_many_rows_in_chunks():
    """Scratch past the cap: row chunks, each row's bits as in a call of its own chunk."""
    n, k, m = 65536, 2048, 1100
    w, x = weight("affine", n, k), rows(m, k, seed=9)
    assert thq.call_scratch_bytes(w, m, x_dtype=torch.float32) <= 512 << 20
    y = thq.matmul(w, x, torch.float32)
    parts = [thq.matmul(w, x[a:b], torch.float32) for a, b in ((0, 512), (512, 1024), (1024, m))]
    assert torch.equal(y, torch.cat(parts))
    pick = np.r_[0, 511, 512, 1023, 1024, 1099]
    ref = x[pick].double() @ w.dequantize().double().T
    assert rel(y[pick], ref) <= 2e-7
