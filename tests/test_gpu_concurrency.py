"""Re-entrancy as include/thq.h states it: calls on distinct streams, from
distinct host threads, give the bits the same calls give one after another
on one stream.  The paths used hold no context workspace (M = 1 GEMV, the
M = 2 row GEMV, the unsplit GEMM, the MFMA decode GEMV at one split); calls
that share the workspace must be ordered on one stream and are not mixed
here.  Calls from several threads on one stream are ordered there whatever
scratch they use.  Streams keep the default priority.
"""
import ctypes as C
import threading

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


def test_two_threads_two_streams_bit_identical():
    w_big = thq.QTensor.from_gguf_bytes(thq.Q4_K, weight_bytes(O.Q4_K, 12288, 4096, seed=71), 12288, 4096)
    w_q8 = thq.QTensor.from_gguf_bytes(thq.Q8_0, weight_bytes(O.Q8_0, 3072, 1024, seed=72), 3072, 1024)
    xs = {m: torch.from_numpy(O.bf16_round(activations(m, 4096, seed=m))).cuda().to(torch.bfloat16)
          for m in (1, 2, 5, 2048)}
    x8 = torch.from_numpy(O.bf16_round(activations(1, 1024, seed=6))).cuda().to(torch.bfloat16)
    # 12288 x 4096 at M = 5: 384 row tiles, one K split (no workspace)
    jobs = [(w_big, xs[1]), (w_big, xs[2]), (w_big, xs[5]), (w_big, xs[2048]), (w_q8, x8)]
    print("[concurrency] reference on one stream", flush=True)
    ref = [thq.matmul(w, x, torch.float32) for w, x in jobs]
    torch.cuda.synchronize()

    results = {}
    errors = []

    def worker(tid):
        try:
            s = torch.cuda.Stream()
            out = []
            with torch.cuda.stream(s):
                for rep in range(4):
                    order = jobs if (tid + rep) % 2 == 0 else jobs[::-1]
                    ys = [thq.matmul(w, x, torch.float32) for w, x in order]
                    out.append(ys if (tid + rep) % 2 == 0 else ys[::-1])
            s.synchronize()
            results[tid] = out
        except Exception as e:  # reported below, in the main thread
            errors.append(e)

    print("[concurrency] two threads, two streams", flush=True)
    threads = [threading.Thread(target=worker, args=(t,)) for t in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=120)
    assert not any(t.is_alive() for t in threads)
    assert not errors, errors
    for tid in range(2):
        for ys in results[tid]:
            for y, r in zip(ys, ref):
                assert torch.equal(y.view(torch.int32), r.view(torch.int32))


def run_threads(fns):
    """Each function in a thread of its own, started together; re-raises the first error."""
    errors = []
    gate = threading.Barrier(len(fns))

    def body(f):
        try:
            gate.wait(60)
            f()
        except Exception as e:
            errors.append(e)

    threads = [threading.Thread(target=body, args=(f,)) for f in fns]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=120)
    assert not any(t.is_alive() for t in threads)
    assert not errors, errors


def test_two_threads_one_stream_prepared_q8act():
    """A prepared dot of 9 rows and more is a GEMM into split sums and a reduce: two threads' calls on one stream
    share the buffer, so neither may come between the other's two launches."""
    n, k = 4096, 4096
    ctx = thq.Context(0)
    w = thq.QTensor.from_gguf_bytes(thq.Q4_K, weight_bytes(O.Q4_K, n, k, seed=75), n, k, ctx=ctx)
    acts = [thq.Q8Act(torch.from_numpy(activations(m, k, seed=m)).cuda(), thq.Q8_K, ctx=ctx) for m in (64, 48)]
    for m in (64, 48):  # two or more splits: partials beside the quantized rows (about m * k bytes)
        assert thq.call_scratch_bytes(w, m, x_dtype=torch.float32, flags=thq.MODE_Q8ACT) > 8 * m * n
    ref = [a.matmul(w, torch.float32) for a in acts]
    torch.cuda.synchronize()
    out = [[], []]

    def worker(i):
        for _ in range(200):  # both on the default stream
            out[i].append(acts[i].matmul(w, torch.float32))

    run_threads([lambda: worker(0), lambda: worker(1)])
    torch.cuda.synchronize()
    for ys, r in zip(out, ref):
        assert all(torch.equal(y, r) for y in ys)


def f32_case(n=2048, k=1024, m=40):
    """A weight, and x / its product by the f16 matrix-core kernel (whose scratch the tests below are about)."""
    ctx = thq.Context(0)
    w = thq.QTensor.from_gguf_bytes(thq.Q4_K, weight_bytes(O.Q4_K, n, k, seed=76), n, k, ctx=ctx)
    xs = [torch.from_numpy(activations(m, k, seed=80 + i)).cuda() for i in range(2)]
    ref = [thq.matmul(w, x, torch.float32) for x in xs]
    torch.cuda.synchronize()
    return w, xs, ref


def test_more_streams_than_scratch_buffers():
    """f32 calls on 20 streams: the context keeps 16 buffers, the others wait for one; every call's own bits."""
    w, xs, ref = f32_case()
    streams = [torch.cuda.ExternalStream(s.cuda_stream) for s in (torch.cuda.Stream() for _ in range(20))]
    assert len({s.cuda_stream for s in streams}) == 20
    out = []
    for rep in range(4):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                out.append((i & 1, thq.matmul(w, xs[i & 1], torch.float32)))
    torch.cuda.synchronize()
    assert all(torch.equal(y, ref[i]) for i, y in out)


def test_per_thread_stream(monkeypatch):
    """hipStreamPerThread is one handle for a stream of each thread's own: its f32 calls take the kernel without
    scratch."""
    w, xs, _ = f32_case()
    monkeypatch.setenv("THQ_GEMM_EX", "0")
    ref = [thq.matmul(w, x, torch.float32) for x in xs]
    monkeypatch.delenv("THQ_GEMM_EX")
    out = [[torch.empty_like(ref[0]) for _ in range(100)] for _ in range(2)]
    torch.cuda.synchronize()
    per_thread, hip = C.c_void_p(2), C.CDLL("libamdhip64.so.7")  # the runtime that is loaded already

    def worker(i):
        for y in out[i]:
            rc = thq.lib.thq_matmul(w.ctx.h, w.h, C.c_void_p(xs[i].data_ptr()), thq.ACT_F32, xs[i].shape[0],
                                    C.c_void_p(y.data_ptr()), thq.ACT_F32, 0, per_thread)
            assert rc == thq.OK, thq.last_error()
        assert hip.hipStreamSynchronize(per_thread) == 0

    run_threads([lambda: worker(0), lambda: worker(1)])
    for ys, r in zip(out, ref):
        assert all(torch.equal(y, r) for y in ys)
