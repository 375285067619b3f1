"""Runtime behaviour on the GPU that the op tests do not see on their own:
sharing a process, device and stream with PyTorch."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def test_kernel_lookups_leave_no_hip_error_for_torch(rt):
    """Every code object's kernels are looked up (GEMV, misc, attention, GEMM),
    then torch allocates and launches: no HIP error may be left pending for it."""
    import torch
    import rxla_amd as rx

    torch.cuda.synchronize()
    rng = np.random.default_rng(1)
    x = rng.standard_normal((130, 256)).astype(np.float32)
    u8, s = oracle.quantize_w8((rng.standard_normal((128, 256)) * 0.02).astype(np.float32), 256)
    rx.quantized_linear(rt, rt.buffer(x[:4]), rt.buffer(u8), rt.buffer(s))   # GEMV
    rx.quantized_linear(rt, rt.buffer(x), rt.buffer(u8), rt.buffer(s))       # GEMM
    rx.dequantize(rt, rt.buffer(u8), rt.buffer(s))                           # misc module
    q = rng.standard_normal((1, 4, 128)).astype(np.float32)
    kc = oracle.bf16_bits(rng.standard_normal((1, 2, 16, 128)).astype(np.float32))
    rx.grouped_query_attention(rt, rt.buffer(q), rt.buffer(kc, rx.DType.BF16),
                               rt.buffer(kc, rx.DType.BF16), rt.buffer(np.array([5], np.int32)))
    rt.synchronize()
    t = torch.ones(1024, device="cuda") * 3  # raises if a HIP error is pending
    torch.cuda.synchronize()
    assert float(t.sum()) == 3072.0


def test_wrapped_torch_tensors_on_torch_stream(rt):
    """rxw8 writes into torch-owned memory on torch's stream; ordering follows
    that stream."""
    import torch
    import rxla_amd as rx

    stream = torch.cuda.Stream()
    rt.set_stream(stream.cuda_stream)
    try:
        rng = np.random.default_rng(2)
        x = rng.standard_normal((200, 512)).astype(np.float32)
        u8, s = oracle.quantize_w8((rng.standard_normal((256, 512)) * 0.02).astype(np.float32), 128)
        with torch.cuda.stream(stream):
            xt = torch.from_numpy(x).cuda()
            ut = torch.from_numpy(u8).cuda()
            st = torch.from_numpy(s).cuda()
            yt = torch.full((200, 256), float("nan"), device="cuda")
        rx.quantized_linear(rt, rt.wrap_tensor(xt), rt.wrap_tensor(ut), rt.wrap_tensor(st),
                            out=rt.wrap_tensor(yt))
        with torch.cuda.stream(stream):
            y = yt.cpu()
        ref = oracle.quantized_linear(x, u8, s)
        assert float(np.abs(y.numpy() - ref).max() / np.abs(ref).max()) <= 1e-2
    finally:
        rt.set_stream(0)


LINEARS = {  # kind: (rows, n, k, x, compute), a larger call of the same runtime, the splits of the mid-size GEMM
    "mid-size splits": ((100, 2048, 6144, "bf16", "bf16"), (330, 4096, 6144, "bf16", "bf16"), "3"),
    "bf16 copy of f32 rows": ((100, 1040, 512, "f32", "bf16"), (330, 1040, 4096, "f32", "bf16"), "1"),
    "hi and lo parts": ((40, 1024, 2048, "f32", "f32"), (300, 1024, 2048, "f32", "f32"), "1"),
    "gemv splits": ((8, 1024, 8192, "bf16", "bf16"), (16, 4096, 8192, "bf16", "bf16"), "1"),
    "decode splits": (None, None, "1"),
}


@pytest.mark.parametrize("given", [True, False])
@pytest.mark.parametrize("kind", list(LINEARS))
def test_a_captured_call_outlives_its_workspaces(monkeypatch, kind, given):
    """A caller's graph (of a stream that it gave the runtime, or of the
    runtime's own) holds the addresses of the workspaces that its calls used. A
    larger eager call replaces them; the replays still give the eager result
    and touch nothing that was allocated since."""
    import torch
    import rxla_amd as rx

    small, large, ks = LINEARS[kind]
    monkeypatch.setenv("RXW8_MID_KS", ks)
    own = rx.Runtime(0)
    stream = torch.cuda.Stream() if given else torch.cuda.ExternalStream(own.stream())
    g = torch.Generator(device="cuda").manual_seed(5)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    keep = []

    def linear(m, n, k, x, compute):
        t = [rand(m, k).to(torch.bfloat16 if x == "bf16" else torch.float32),
             torch.randint(1, 256, (n, k), generator=g, device="cuda", dtype=torch.uint8),
             rand(n, k // 128).abs() * 1e-3, torch.empty(m, n, device="cuda")]
        keep.append(t)
        b = [own.wrap_tensor(v) for v in t]
        dt = rx.DType.F32 if compute == "f32" else rx.DType.BF16
        return lambda: rx.quantized_linear(own, *b[:3], dt, rx.DType.F32, out=b[3]), t[3]

    def decode(batch, length):
        t = [rand(batch, 64, 128), rand(batch, 8, length, 128).bfloat16(), rand(batch, 8, length, 128).bfloat16(),
             torch.full((batch,), length, device="cuda", dtype=torch.int32), torch.empty(batch, 64, 128, device="cuda")]
        keep.append(t)
        b = [own.wrap_tensor(v) for v in t]
        return lambda: rx.grouped_query_attention(own, *b[:4], out=b[4]), t[4]

    (call, y), (bigger, _) = ((linear(*small), linear(*large)) if small else (decode(1, 600), decode(8, 4000)))
    torch.cuda.synchronize()
    own.set_stream(stream.cuda_stream)
    call()
    own.synchronize()
    eager = y.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
        call()
    torch.cuda.synchronize()
    bigger()
    own.synchronize()
    # whatever the runtime gave back is handed out again here
    since = [own.zeros((1 << 18,), rx.DType.F32) for _ in range(8)]
    guard = [torch.full((1 << s,), 3.0, device="cuda") for s in range(16, 25)]
    for _ in range(3):
        y.fill_(7.0)
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, eager)
        bigger()
        own.synchronize()
    assert all(bool((t == 3.0).all()) for t in guard)
    assert all(not b.to_numpy().any() for b in since)
    own.set_stream(None)


@pytest.mark.parametrize("mode", ["thread_local", "global"])
@pytest.mark.parametrize("same_thread", [True, False])
def test_a_runtime_is_created_beside_a_capture(mode, same_thread):
    """While a stream is being captured, by this thread or another one, a
    runtime can be created (loading its kernels may end that capture: HIP's
    own rule), and its split attention works once the capture is over."""
    import threading

    import torch
    import rxla_amd as rx

    made, stream = [], torch.cuda.Stream()
    x = torch.zeros(4, device="cuda")

    def make():
        try:
            made.append(rx.Runtime(0))
        except rx.Error as e:
            made.append(e)

    torch.cuda.synchronize()
    try:
        with torch.cuda.graph(torch.cuda.CUDAGraph(), stream=stream, capture_error_mode=mode):
            x += 1
            if same_thread:
                make()
            else:
                t = threading.Thread(target=make)
                t.start()
                t.join()
    except RuntimeError:
        pass
    torch.cuda.synchronize()
    assert isinstance(made[0], rx.Runtime), made[0]
    own, rng = made[0], np.random.default_rng(4)
    q, k, v = (rng.standard_normal(s).astype(np.float32) for s in ((1, 4, 256), (1, 2, 600, 256), (1, 2, 600, 256)))
    out = [rx.grouped_query_attention(own, own.buffer(q), own.buffer(k), own.buffer(v),
                                      own.buffer(np.array([600], np.int32))).to_numpy() for _ in range(3)]
    s = np.einsum("hgd,hkd->hgk", q[0].reshape(2, 2, 256).astype(np.float64), k[0]) / 16
    p = np.exp(s - s.max(-1, keepdims=True))
    want = np.einsum("hgk,hkd->hgd", p / p.sum(-1, keepdims=True), v[0].astype(np.float64)).reshape(4, 256)
    for o in out:
        assert np.abs(o[0] - want).max() <= 1e-5
