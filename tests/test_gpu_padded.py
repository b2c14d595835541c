"""GPU parity of widths that are no multiples of 64, which the 16-bit linears run on zero-padded
copies of their operands (the few smallest layers excepted), against the f64 oracle with the bf16
tolerance of tests/_util.assert_parity: forward, h, dx, dA, dB and the bias gradient in both
16-bit types, on both sides of the rule that picks the copies, for ranks that are no multiples of
16, operands off their 16-byte alignment, and the allocation-free forward."""
import ctypes

import numpy as np
import pytest

import oracle
from tests._util import assert_parity, bf16_f32, to_dev

pytestmark = pytest.mark.gpu


def _case(M, K, N, r, seed, f16):
    x = oracle.normal_bf16(seed + 1, (M, K), 1.0)
    q, s, st = oracle.pack(oracle.normal_bf16(seed + 2, (N, K), 0.02), "bf16")
    assert st == 0
    A = oracle.normal_bf16(seed + 3, (K, r), 0.05) if r else None
    B = oracle.normal_bf16(seed + 4, (r, N), 0.05) if r else None
    dy = oracle.normal_bf16(seed + 5, (M, N), 1.0)
    bias = oracle.normal_bf16(seed + 6, (N,), 0.1)
    if f16:
        x, A, B, dy, bias = (None if a is None else oracle.f32_to_f16(oracle.bf16_to_f32(a))
                             for a in (x, A, B, dy, bias))
    return dict(x=x, q=q, s=s, A=A, B=B, dy=dy, bias=bias)


def _dev(a, dev, f16, offset=0):
    """The operand on the device, its first element ``offset`` elements past a 16-byte boundary."""
    import torch
    if a is None:
        return None
    t = (torch.from_numpy(np.ascontiguousarray(a).view(np.float16)).to(dev) if f16
         else to_dev(a, dev))
    if not offset:
        return t
    flat = torch.zeros((t.numel() + offset,), dtype=t.dtype, device=dev)
    flat[offset:] = t.reshape(-1)
    return flat[offset:].view(t.shape)


def _np(t):
    import torch
    return bf16_f32(t) if t.dtype == torch.bfloat16 else t.float().cpu().numpy()


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("M,K,N,r", [
    (65, 100, 101, 3),      # just past the tiny layers
    (64, 129, 127, 4),      # past them by one width
    (64, 128, 127, 4),      # the last tiny layer: direct kernels
    (1, 1000, 65, 8),       # one token
    (300, 63, 1025, 24),    # a width under one step, one past a tile
    (1500, 2111, 190, 16),  # the split-reduction GEMMs, odd width
    (530, 144, 2560, 40),   # only the input padded
    (777, 1024, 1000, 0),   # only the output padded, no adapter
    (2600, 520, 777, 160),  # rank above one chunk
])
def test_padded_widths(dev, M, K, N, r, f16):
    import torch
    from reels_amd import QuantizedMatrix, i8lora_backward, i8lora_forward
    print(f"[padded] M={M} K={K} N={N} r={r} f16={f16}", flush=True)
    cs = _case(M, K, N, r, 300 + M + K + N + r, f16)
    elt = "f16" if f16 else "bf16"
    W = QuantizedMatrix(to_dev(cs["q"], dev, "raw"), to_dev(cs["s"], dev, "raw"))
    res = []
    for off in (0, 1):  # aligned, and every 16-bit operand two bytes past alignment
        x, A, B, bias, dy = (_dev(cs[k], dev, f16, off) for k in ("x", "A", "B", "bias", "dy"))
        y, h = i8lora_forward(x, W, A, B, bias, 0.5, save_h=r > 0)
        g = i8lora_backward(dy, x, W, A, B, 0.5, h=h, want_dbias=True)
        g2 = i8lora_backward(dy, x, W, A, B, 0.5, h=None)  # h recomputed
        torch.cuda.synchronize(dev)
        res.append((y, h, g))
        if r:
            assert torch.equal(g[2], g2[2]), "dB from a recomputed h differs"
    yo, ho = oracle.lora_forward(cs["x"], cs["q"], cs["s"], cs["A"], cs["B"], 0.5, cs["bias"], elt=elt)
    Ao = cs["A"] if r else np.zeros((K, 0), np.uint16)
    Bo = cs["B"] if r else np.zeros((0, N), np.uint16)
    ref = oracle.lora_backward(cs["dy"], cs["x"], cs["q"], cs["s"], Ao, Bo, 0.5,
                               want=("dx", "dA", "dB") if r else ("dx",), elt=elt)
    for y, h, (dx, dA, dB, db) in res:
        assert_parity(_np(y), yo, "y")
        assert_parity(_np(dx), ref["dx"], "dx")
        assert_parity(db.cpu().numpy(), oracle.bias_gradient(cs["dy"], elt=elt), "dbias", tol=1e-5)
        if r:
            assert_parity(_np(h), ho, "h")
            assert_parity(dA.cpu().numpy(), ref["dA"], "dA")
            assert_parity(dB.cpu().numpy(), ref["dB"], "dB")


@pytest.mark.parametrize("M,K,N,r", [(300, 500, 513, 8), (5000, 1000, 2500, 16)])
def test_padded_noalloc_forward(dev, M, K, N, r):
    """The allocation-free forward: the workspace forward's bits where the padded copies fit its
    scratch (the first case), the direct kernels beyond it (the second), the oracle in both."""
    import torch
    from reels_amd import QuantizedMatrix, _lib, i8lora_forward
    L = _lib.lib()
    cs = _case(M, K, N, r, 900 + M, False)
    print(f"[padded] noalloc M={M} K={K} N={N} r={r}", flush=True)
    x, A, B, bias = (to_dev(cs[k], dev) for k in ("x", "A", "B", "bias"))
    W = QuantizedMatrix(to_dev(cs["q"], dev, "raw"), to_dev(cs["s"], dev, "raw"))
    y0, h0 = i8lora_forward(x, W, A, B, bias, 1.0, save_h=True)
    y = torch.empty_like(y0)
    h = torch.empty_like(h0)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    st = ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)
    fits = L.reels_hip_i8lora_workspace_bytes(M, K, N, r, _lib.WS_FWD) <= 32 << 20
    assert fits == (M == 300)
    assert L.reels_hip_i8lora_workspace_bytes(M, K, N, r, _lib.WS_FWD_NOALLOC) <= 32 << 20
    _lib.check("reels_hip_i8lora_fwd_noalloc", L.reels_hip_i8lora_fwd_noalloc(
        p(x), p(W.values), p(W.scales), p(A), p(B), p(bias), M, K, N, r, 1.0, p(y), p(h), st))
    torch.cuda.synchronize(dev)
    if fits:
        assert torch.equal(y.view(torch.int16), y0.view(torch.int16))
        assert torch.equal(h.view(torch.int16), h0.view(torch.int16))
    rows = np.unique(np.linspace(0, M - 1, 40).astype(int))
    yo, _ = oracle.lora_forward(cs["x"][rows], cs["q"], cs["s"], cs["A"], cs["B"], 1.0, cs["bias"])
    assert_parity(bf16_f32(y)[rows], yo, "noalloc y")


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("M,K,N,r", [
    (777, 1000, 3000, 8),   # row-wave launches
    (65, 300, 127, 0),      # the few-token path
    (9000, 1000, 500, 16),  # the GEMM
    (1500, 130, 1111, 4),   # its split reduction
])
def test_padded_dx_rounding_points(dev, M, K, N, r, f16):
    """dX of widths that are no multiples of 64 multiplies bf16(dy s) and the exact codes (f16: dy and
    f16(q f16(s))). With one nonzero per row of dy a sum has one term, so dx is that product rounded
    once, bit for bit; dA takes u from dy itself."""
    import torch
    from reels_amd import QuantizedMatrix, i8lora_backward
    print(f"[padded] rounding points M={M} K={K} N={N} r={r} f16={f16}", flush=True)
    cs = _case(M, K, N, r, 1200 + M + K + N + r, f16)
    x, A, B, dy = (_dev(cs[k], dev, f16) for k in ("x", "A", "B", "dy"))
    hot = torch.arange(M, device=dev) * 7 % N
    keep = torch.zeros((M, N), dtype=torch.bool, device=dev)
    keep[torch.arange(M, device=dev), hot] = True
    dy = torch.where(keep, dy, torch.zeros_like(dy))
    q, s = to_dev(cs["q"], dev, "raw"), to_dev(cs["s"], dev, "raw")
    A0 = torch.zeros_like(A) if r else None
    dx = i8lora_backward(dy, x, QuantizedMatrix(q, s), A0, B, 1.0)[0]
    d = dy[torch.arange(M, device=dev), hot].float()
    if f16:
        w = (q.half() * s.half()[:, None])[hot].double()
        want = (d.double()[:, None] * w).to(torch.float32).half()
    else:
        ds = (d * s[hot]).bfloat16().float()
        want = (ds[:, None] * q[hot].float()).bfloat16()
    assert torch.equal(dx, want)
    if r:
        _, dA, _ = i8lora_backward(dy, x, QuantizedMatrix(q, s), A, B, 1.0)
        u = (dy.double() @ B.double().t()).to(dy.dtype).double()
        assert_parity(dA.cpu().numpy(), (x.double().t() @ u).cpu().numpy(), "dA")


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("M,K,N,r", [
    (777, 1000, 3000, 3),   # row-wave launches
    (20, 300, 127, 1),      # the few-token path
    (9000, 1000, 500, 5),   # the GEMM
])
def test_padded_infinite_rows(dev, M, K, N, r, f16):
    """An infinite x (dy) with positive codes, scales and adapters gives infinite y and h (dx) in its
    own row and changes no other row: the padding of the rank adds nothing, also to infinities."""
    import torch
    from reels_amd import QuantizedMatrix, i8lora_backward, i8lora_forward
    print(f"[padded] infinite rows M={M} K={K} N={N} r={r} f16={f16}", flush=True)
    cs = _case(M, K, N, r, 1500 + M, f16)
    x, A, B, dy = (_dev(cs[k], dev, f16) for k in ("x", "A", "B", "dy"))
    W = QuantizedMatrix(to_dev(cs["q"], dev, "raw").abs().clamp(min=1), to_dev(cs["s"], dev, "raw"))
    A, B = A.abs() + 0.01, B.abs() + 0.01

    def run(x, dy):
        y, h = i8lora_forward(x, W, A, B, None, 1.0, save_h=True)
        return y, h, i8lora_backward(dy, x, W, A, B, 1.0, h=h)[0]
    ref = run(x, dy)
    bad = M // 2
    x[bad, K - 1] = float("inf")
    dy[bad, N - 1] = float("inf")
    got = run(x, dy)
    rest = torch.arange(M, device=dev) != bad
    for name, a, b in zip(("y", "h", "dx"), ref, got):
        assert bool(torch.isposinf(b[bad]).all()), name
        assert torch.equal(a[rest], b[rest]), name
