"""THQ_MODE_Q8ACT over many rows on the int8 matrix cores (k_q8act_gemm.hip)
against the row-tile kernels (THQ_Q8ACT_GEMM=0, themselves pinned to the
oracle): the same exact block integers, so only the f32 order differs: relative
2-norm <= 4e-7 (the row-tile kernels are up to 2.1e-7 from 64-bit sums, this
one up to 0.8e-7).  Covered: row-group edges, ragged outputs, one chunk and K
splits, extreme quants (every product at its largest: the two int8 planes, the
minimum's sums), gate/up, prepared buffers, the emitted operand, and the rule.
"""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import activations, weight_bytes

pytestmark = pytest.mark.gpu

thq = pytest.importorskip("thq")


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.init()
    yield
    torch.cuda.synchronize()


def rel(y, ref):
    return float((y.double() - ref.double()).norm() / ref.double().norm())


def both(monkeypatch, f):
    out = []
    for v in ("0", "1"):
        monkeypatch.setenv("THQ_Q8ACT_GEMM", v)
        out.append(f())
    return out


@pytest.mark.parametrize("qt", [O.Q4_K, O.Q8_0])
@pytest.mark.parametrize("m,n,k", [(1, 40, 256), (31, 300, 1792), (33, 512, 1024), (64, 257, 2048), (70, 1000, 4096),
                                   (9, 96, 17408)])
def test_matches_row_tiles(qt, m, n, k, monkeypatch):
    w = thq.QTensor.from_gguf_bytes(qt, weight_bytes(qt, n, k, seed=5), n, k)
    x = torch.from_numpy(activations(m, k, seed=6)).cuda()
    ref, y = both(monkeypatch, lambda: thq.matmul(w, x, torch.float32, thq.MODE_Q8ACT))
    assert rel(y, ref) <= 4e-7
    q = thq.Q8Act(x, thq.Q8_K if qt == O.Q4_K else thq.Q8_0)
    assert torch.equal(q.matmul(w, torch.float32), y)


@pytest.mark.parametrize("rest,quant", [(1.0, -128), (0.999, -128), (-0.999, 127)])
def test_largest_integers(rest, quant, monkeypatch):
    """All nibbles 15, all scales and minima 63, and rows whose quants are all -128 (a block's largest value always is;
    the rest of its sign too) or, past the largest, 127: the largest sums of either sign that the planes can reach."""
    n, k, m = 64, 512, 40
    blk = np.zeros((n, k // 256, 144), np.uint8)
    blk[:, :, 0:4] = np.array([1.0, 0.5], np.float16).view(np.uint8)
    blk[:, :, 4:] = 0xFF
    w = thq.QTensor.from_gguf_bytes(O.Q4_K, blk.reshape(n, -1), n, k)
    x = torch.full((m, k), rest, device="cuda")
    x[:, ::256] = 1.0
    codes = thq.quantize_act(x, thq.Q8_K).view(m, k // 256, 292)[:, :, 4:260].contiguous().view(torch.int8)
    assert (codes[:, :, 0] == -128).all() and (codes[:, :, 1:] == quant).all()
    ref, y = both(monkeypatch, lambda: thq.matmul(w, x, torch.float32, thq.MODE_Q8ACT))
    assert rel(y, ref) <= 4e-7
    s = codes.double().sum(-1).sum(-1) * codes.new_tensor(-1.0 / 128, dtype=torch.float64)  # d = 1 / iscale = -1 / 128
    exact = (63.0 * 15 - 0.5 * 63) * s  # d sc q - dmin m of every weight
    assert rel(y, exact[:, None].expand(m, n)) <= 4e-7


@pytest.mark.parametrize("qt", [O.Q4_K, O.Q8_0])
def test_gate_up_and_emit(qt, monkeypatch):
    h, k, m = 256, 1024, 64  # whole 256-B planes: the buffers hold no padding
    w = thq.QTensor.from_gguf_bytes(qt, weight_bytes(qt, 2 * h, k, seed=8), 2 * h, k)
    x = torch.from_numpy(activations(m, k, seed=9)).cuda()
    ref, y = both(monkeypatch, lambda: thq.gate_up_silu(w, x, torch.float32, thq.MODE_Q8ACT))
    assert rel(y, ref) <= 1e-3 and float((y != ref).float().mean()) <= 0.02  # sums round to bf16 first
    if qt == O.Q4_K:
        z, nxt = thq.Q8Act(x, thq.Q8_K).gate_up_silu_emit(w, torch.float32)
        assert torch.equal(z, y)
        assert torch.equal(nxt.buf, thq.Q8Act(y, thq.Q8_K).buf)


def test_rule_and_capture():
    """Captured prepared dots run the eager call's kernels (its bits), warmed up or not."""
    ctx = thq.Context(0)
    n, k, m = 4096, 1024, 96  # large enough for the int8 GEMM, K splits among them
    w = thq.QTensor.from_gguf_bytes(O.Q4_K, weight_bytes(O.Q4_K, n, k, seed=5), n, k, ctx=ctx)
    x = torch.from_numpy(activations(m, k, seed=6)).cuda()
    q = thq.Q8Act(x, thq.Q8_K, ctx=ctx)
    s = torch.cuda.Stream()
    out = []
    with torch.cuda.stream(s):
        s.wait_stream(torch.cuda.default_stream())
        for warm in (False, True):
            if warm:
                ref = q.matmul(w, torch.float32)
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=s):
                y = q.matmul(w, torch.float32)
            out.append((g, y))
    assert torch.equal(thq.matmul(w, x, torch.float32, thq.MODE_Q8ACT), ref)
    for g, y in out:
        for _ in range(3):
            y.fill_(float("nan"))
            torch.randn(64, 64, device="cuda") @ torch.randn(64, 64, device="cuda")
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, ref)


def capture(f):
    g, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s), torch.cuda.graph(g, stream=s):
        return g, f()


def test_captured_without_scratch(monkeypatch):
    """Captures that get no graph scratch run the row-tile kernels, the emitting gate/up too, though no eager call of
    this size has made its counters."""
    ctx, ctx_ref = thq.Context(0), thq.Context(0)
    h, k, m = 4096, 4096, 16
    w = thq.QTensor.from_gguf_bytes(O.Q4_K, weight_bytes(O.Q4_K, 2 * h, k, seed=12), 2 * h, k, ctx=ctx)
    x = torch.from_numpy(activations(m, k, seed=13)).cuda()
    planes = thq.Q8Act(x, thq.Q8_K, ctx=ctx)
    assert thq.call_scratch_bytes(w, m, torch.float32, thq.MODE_Q8ACT, True) > 8 * m * h  # split sums
    planes.gate_up_silu_emit(w, torch.float32)  # warm
    with monkeypatch.context() as mp:
        mp.setenv("THQ_Q8ACT_GEMM", "0")
        ref, nref = thq.Q8Act(x, thq.Q8_K, ctx=ctx_ref).gate_up_silu_emit(w, torch.float32)
        pref = planes.matmul(w, torch.float32)
    monkeypatch.setenv("THQ_GRAPH_SCRATCH_MB", "0")
    g, (y, nxt, p) = capture(lambda: (*planes.gate_up_silu_emit(w, torch.float32), planes.matmul(w, torch.float32)))
    for _ in range(3):
        y.fill_(float("nan"))
        p.fill_(float("nan"))
        nxt.buf.zero_()
        torch.randn(64, 64, device="cuda") @ torch.randn(64, 64, device="cuda")
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ref) and torch.equal(p, pref)
        assert torch.equal(nxt.buf, nref.buf)


def test_many_rows_in_chunks():
    """Split sums past 512 MiB: row chunks, each row's bits as in a call of its own chunk, prepared or not."""
    n, k, m = 65536, 4352, 1100
    w = thq.QTensor.from_gguf_bytes(O.Q4_K, np.tile(weight_bytes(O.Q4_K, 1024, k, seed=15).reshape(1024, -1), (64, 1)),
                                    n, k)
    x = torch.from_numpy(activations(m, k, seed=16)).cuda()
    size = thq.call_scratch_bytes(w, m, torch.float32, thq.MODE_Q8ACT)
    assert (256 << 20) < size <= (512 << 20) + 2 * m * k
    y = thq.matmul(w, x, torch.float32, thq.MODE_Q8ACT)
    parts = [thq.matmul(w, x[a:b], torch.float32, thq.MODE_Q8ACT) for a, b in ((0, 512), (512, 1024), (1024, m))]
    assert torch.equal(y, torch.cat(parts))
    assert torch.equal(thq.Q8Act(x, thq.Q8_K).matmul(w, torch.float32), y)
