"""The mid-size W8A16 GEMM (a few dozen to a few hundred rows) at the edges of
its tiles, against the CPU oracle on every plan: 16-row fragments, 64-row
tiles, 64- and 128-channel tiles, K splits (also uneven ones and more wave
groups than chunks), grouped scales that straddle the 256-wide chunks, f32 and
bf16 rows, both weight layouts. Tolerance: the operands are the oracle's bf16
values and the sums f32, so results agree to one bf16 rounding (2^-8 of the
element) with most bits equal; normwise 1e-2 / 2."""
import numpy as np
import pytest

import oracle
from conftest import rel_err

pytestmark = pytest.mark.gpu


def rx():
    import rxla_amd
    return rxla_amd


def run(rt, x, u8, s, xd, packed, yd):
    r = rx()
    xb = rt.buffer(oracle.bf16_bits(x), r.DType.BF16) if xd == "bf16" else rt.buffer(x)
    wb = rt.buffer(u8)
    if packed:
        wb = r.pack_weight(rt, wb)
    y = r.quantized_linear(rt, xb, wb, rt.buffer(s), r.DType.BF16,
                           r.DType.F32 if yd == "f32" else r.DType.BF16).to_numpy()
    return r.bf16_to_f32(y) if yd == "bf16" else y


@pytest.mark.parametrize("m,n,k,g", [(17, 64, 256, 256), (32, 48, 512, 64), (48, 208, 1024, 128),
                                     (64, 128, 768, 192), (65, 256, 512, 512), (100, 80, 1280, 320),
                                     (130, 384, 2304, 128), (5, 144, 512, 512)])
@pytest.mark.parametrize("rg,ks", [(1, 1), (2, 1), (1, 2), (2, 3)])
def test_tiles_against_the_oracle(rt, monkeypatch, m, n, k, g, rg, ks):
    monkeypatch.setenv("RXW8_GEMM_MID", "2")
    monkeypatch.setenv("RXW8_MID_RG", str(rg))
    monkeypatch.setenv("RXW8_MID_KS", str(ks))
    rng = np.random.default_rng(m + n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    u8, s = oracle.quantize_w8((rng.standard_normal((n, k)) * 0.02).astype(np.float32), g)
    want = oracle.quantized_linear(x, u8, s, oracle.COMPUTE_BF16)
    for xd in ("f32", "bf16") if m > 16 else ("f32",):
        for packed in (False, True) if m <= 64 or n % 128 == 0 else (False,):
            for yd in ("f32", "bf16"):
                got = run(rt, x, u8, s, xd, packed, yd)
                assert rel_err(got, want) <= 5e-3
                # one bf16 step, at most, per element
                assert np.max(np.abs(got - want) / np.maximum(np.abs(want), 0.05)) <= 2.0 ** -7


@pytest.mark.parametrize("m,n,k", [(48, 6144, 4096), (33, 4096, 1024), (100, 2048, 6144), (200, 1040, 512)])
def test_default_plans(rt, monkeypatch, m, n, k):
    """The default rule's choice against the paths it replaces (one bf16 step)."""
    rng = np.random.default_rng(n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    u8, s = oracle.quantize_w8((rng.standard_normal((n, k)) * 0.02).astype(np.float32), 128)
    got = run(rt, x, u8, s, "f32", False, "f32")
    again = run(rt, x, u8, s, "f32", False, "f32")
    np.testing.assert_array_equal(got, again)
    monkeypatch.setenv("RXW8_GEMM_MID", "0")
    want = run(rt, x, u8, s, "f32", False, "f32")
    rms = np.sqrt(np.mean(want * want))
    assert np.max(np.abs(got - want) / np.maximum(np.abs(want), rms)) <= 2.0 ** -7
    assert np.mean(got != want) < 0.05


def test_rows_and_scales_that_are_not_numbers_stay_in_their_row(rt):
    """NaN and infinite activations reach their own row's outputs alone."""
    rng = np.random.default_rng(2)
    x = rng.standard_normal((40, 2048)).astype(np.float32)
    u8, s = oracle.quantize_w8((rng.standard_normal((4096, 2048)) * 0.02).astype(np.float32), 2048)
    clean = run(rt, x, u8, s, "bf16", False, "f32")
    x[7, 100], x[39, 2047] = np.nan, np.inf
    got = run(rt, x, u8, s, "bf16", False, "f32")
    keep = np.array([i for i in range(40) if i not in (7, 39)])
    np.testing.assert_array_equal(got[keep], clean[keep])
    assert np.isnan(got[7]).all() and not np.isfinite(got[39]).any()


@pytest.mark.parametrize("m,n,k,g", [(17, 256, 128, 64), (33, 272, 384, 128), (64, 512, 768, 192),
                                     (65, 48, 640, 640), (130, 304, 1024, 128), (200, 256, 1280, 64)])
@pytest.mark.parametrize("ks", [1, 2, 3])
@pytest.mark.parametrize("packed", [False, True])
def test_f32_compute_tiles(rt, monkeypatch, m, n, k, g, ks, packed):
    """The F32-compute tiles of the same file, 32- and 64-row tiles, splits
    that cut scale groups, against the oracle's float64 result: x enters as
    bf16 hi + lo parts (2^-17 of the value), the sums are f32."""
    monkeypatch.setenv("RXW8_F32_MID_KS", str(min(ks, k // 128)))
    r = rx()
    rng = np.random.default_rng(m + k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    u8, s = oracle.quantize_w8((rng.standard_normal((n, k)) * 0.02).astype(np.float32), g)
    wb = rt.buffer(u8)
    if packed:
        wb = r.pack_weight(rt, wb)
    got = r.quantized_linear(rt, rt.buffer(x), wb, rt.buffer(s), r.DType.F32, r.DType.F32).to_numpy()
    want = x.astype(np.float64) @ (((u8.astype(np.float64) - 128).reshape(n, k // g, g)
                                    * s.astype(np.float64)[:, :, None]).reshape(n, k)).T
    assert rel_err(got, want) <= 1e-5
    # whole-number inputs that need the lo part: exact
    xi = rng.integers(-2000, 2001, (m, k)).astype(np.float32)
    si = np.ones_like(s)
    ui = rng.integers(126, 131, (n, k)).astype(np.uint8)
    wi = rt.buffer(ui)
    if packed:
        wi = r.pack_weight(rt, wi)
    yi = r.quantized_linear(rt, rt.buffer(xi), wi, rt.buffer(si), r.DType.F32, r.DType.F32).to_numpy()
    np.testing.assert_array_equal(yi, xi.astype(np.float64) @ (ui.astype(np.float64) - 128).T)


@pytest.mark.parametrize("m,n,k,x,compute,split", [
    (100, 1040, 512, "f32", "bf16", False), (300, 1040, 512, "f32", "bf16", False),
    (300, 2048, 4096, "bf16", "bf16", True), (17, 32768, 1024, "f32", "f32", True)])
def test_a_first_call_in_a_capture(m, n, k, x, compute, split):
    """A capture can't size a workspace. A call that comes first there, with no
    room for the bf16 copy of its f32 rows, gives the eager bits; one with no
    room for its K splits runs without them (the sums in another order: one
    bf16 step, or 1e-5 in F32)."""
    import torch
    r = rx()
    g = torch.Generator(device="cuda").manual_seed(m)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    t = [rand(m, k).to(torch.float32 if x == "f32" else torch.bfloat16),
         torch.randint(1, 256, (n, k), generator=g, device="cuda", dtype=torch.uint8),
         rand(n, k // 128).abs() * 1e-3, torch.zeros(m, n, device="cuda")]
    torch.cuda.synchronize()
    dt = r.DType.F32 if compute == "f32" else r.DType.BF16

    def call(own, rows=m, chans=n):
        b = [own.wrap_tensor(v) for v in (t[0][:rows], t[1][:chans], t[2][:chans])]
        out = t[3][:rows, :chans] if chans == n else torch.empty(rows, chans, device="cuda")
        return r.quantized_linear(own, *b, dt, r.DType.F32, out=own.wrap_tensor(out)), out

    eager = r.Runtime(0)
    call(eager)
    eager.synchronize()
    want = t[3].clone()
    own, stream = r.Runtime(0), torch.cuda.Stream()
    own.set_stream(stream.cuda_stream)
    if compute == "f32":  # (its hi and lo parts need their buffer in any plan)
        _, small = call(own, chans=64)
        own.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
        call(own)
    for _ in range(3):
        t[3].fill_(7.0)
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            graph.replay()
        torch.cuda.synchronize()
        if not split:
            assert torch.equal(t[3], want)
        else:
            step = 1e-5 if compute == "f32" else 2.0 ** -7
            assert float(((t[3] - want).abs() / want.abs().clamp_min(want.std())).max()) <= step
    own.set_stream(None)


@pytest.mark.parametrize("m,n,k,compute,mid", [
    (8, 4096, 1024, "bf16", False), (16, 2048, 2048, "bf16", False), (6, 24576, 1536, "bf16", False),
    (12, 12288, 2048, "bf16", True), (48, 2048, 2048, "bf16", True),
    (4096, 2048, 2048, "f32", False), (512, 16384, 2048, "f32", False), (2048, 3072, 3584, "f32", False),
    (500, 7168, 1024, "f32", True), (300, 1024, 3584, "f32", True), (5000, 5120, 1024, "f32", True)])
def test_default_route(rt, monkeypatch, m, n, k, compute, mid):
    """Where the mid-size tiles measured slower than the kernels that they
    stand beside, the default rule leaves the call to those: its bits are those
    of the one path, and not those of the other (other orders of summation)."""
    import torch
    r = rx()
    g = torch.Generator(device="cuda").manual_seed(m + n)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    t = [rand(m, k), torch.randint(1, 256, (n, k), generator=g, device="cuda", dtype=torch.uint8),
         rand(n, k // 128).abs() * 1e-3]
    torch.cuda.synchronize()
    dt = r.DType.F32 if compute == "f32" else r.DType.BF16
    env = "RXW8_F32_MID" if compute == "f32" else "RXW8_GEMM_MID"
    wb = r.pack_weight(rt, rt.wrap_tensor(t[1]))

    def call(mode):
        if mode:
            monkeypatch.setenv(env, mode)
        y = torch.empty(m, n, device="cuda")
        torch.cuda.synchronize()
        r.quantized_linear(rt, rt.wrap_tensor(t[0]), wb, rt.wrap_tensor(t[2]), dt, r.DType.F32, out=rt.wrap_tensor(y))
        rt.synchronize()
        return y

    default, without, forced = call(None), call("0"), call("2")
    assert not torch.equal(without, forced)
    assert torch.equal(default, forced if mid else without)
