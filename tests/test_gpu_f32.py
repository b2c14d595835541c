"""GPU parity of the fp32 entry points (reels_hip_i8lora_fwd_f32 / _bwd_f32 / gelu_tanh_f32): the
reference's Float32 compute with int8 frozen weights (_dequantize_for_compute with T = Float32,
src/layers/quantization.jl:61-64; lora_forward / lora_backward in Float32, lora.jl:56-118),
checked against the f64 oracle (elt="f32") on the same seeded float32 inputs.

Tolerance: fp32 compute with f32 sums over at most 5120 terms keeps the error near 2^-24 times a
small multiple of sqrt(K); the bar here is normwise and elementwise 1e-5 (tests/_util.assert_parity
with tol=1e-5), a thousand times tighter than the bf16 bar. Covered: the GEMM on bf16 planes (any
widths, any 4-byte aligned operands, chunks of tokens), the fp32 projection and split-M gradient
kernels, the generic kernels (a workspace off its alignment), and the mirror API with autograd."""
import numpy as np
import pytest

import oracle
from tests._util import assert_parity

pytestmark = pytest.mark.gpu
TOL = 1e-5


def f32v(seed, shape, sigma):
    """Seeded N(0, sigma^2) float32 values with all 24 significant bits in use."""
    return (np.random.default_rng(seed).standard_normal(shape) * sigma).astype(np.float32)


def make_case(M, K, N, r, alpha, seed=0, bias=False, w_sigma=0.02, ab_sigma=0.01):
    x = f32v(seed + 1, (M, K), 1.0)
    w = f32v(seed + 2, (N, K), w_sigma)
    q, s, st = oracle.pack(w, "f32")
    assert st == 0
    A = f32v(seed + 3, (K, r), ab_sigma) if r else None
    B = f32v(seed + 4, (r, N), ab_sigma) if r else None
    dy = f32v(seed + 5, (M, N), 1.0)
    b = f32v(seed + 6, (N,), 0.1) if bias else None
    c = float(np.float32(alpha) / np.float32(r)) if r else 0.0
    return dict(x=x, q=q, s=s, A=A, B=B, dy=dy, bias=b, c=c, M=M, K=K, N=N, r=r)


def todev(a, d):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(d)


def run_gpu(d, cs):
    import torch
    from reels_amd import QuantizedMatrix, i8lora_backward, i8lora_forward
    W = QuantizedMatrix(todev(cs["q"], d), todev(cs["s"], d), torch.float32)
    x = todev(cs["x"], d)
    A = todev(cs["A"], d) if cs["r"] else None
    B = todev(cs["B"], d) if cs["r"] else None
    bias = todev(cs["bias"], d) if cs["bias"] is not None else None
    y, h = i8lora_forward(x, W, A, B, bias, cs["c"], save_h=cs["r"] > 0)
    assert y.dtype == torch.float32
    dx, dA, dB = i8lora_backward(todev(cs["dy"], d), x, W, A, B, cs["c"], h=h)
    assert dx.dtype == torch.float32
    torch.cuda.synchronize(d)
    out = dict(y=y.cpu().numpy(), dx=dx.cpu().numpy())
    if h is not None:
        out["h"] = h.cpu().numpy()
        out["dA"], out["dB"] = dA.cpu().numpy(), dB.cpu().numpy()
    return out


def check(d, cs, label):
    print(f"[f32] {label}: M={cs['M']} K={cs['K']} N={cs['N']} r={cs['r']}", flush=True)
    g = run_gpu(d, cs)
    y, h = oracle.lora_forward(cs["x"], cs["q"], cs["s"], cs["A"], cs["B"], cs["c"], cs["bias"],
                               elt="f32")
    assert_parity(g["y"], y, f"{label} y", tol=TOL)
    if cs["r"]:
        assert_parity(g["h"], h, f"{label} h", tol=TOL)
        ref = oracle.lora_backward(cs["dy"], cs["x"], cs["q"], cs["s"], cs["A"], cs["B"], cs["c"],
                                   elt="f32")
        assert_parity(g["dA"], ref["dA"], f"{label} dA", tol=TOL)
        assert_parity(g["dB"], ref["dB"], f"{label} dB", tol=TOL)
    else:
        z = np.zeros((cs["K"], 0), np.float32), np.zeros((0, cs["N"]), np.float32)
        ref = oracle.lora_backward(cs["dy"], cs["x"], cs["q"], cs["s"], z[0], z[1], 0.0,
                                   want=("dx",), elt="f32")
    assert_parity(g["dx"], ref["dx"], f"{label} dx", tol=TOL)
    return g


@pytest.mark.parametrize("M,K,N,r,bias", [
    (1024, 1536, 1536, 16, False),  # the CPU-runnable workload's shape
    (333, 512, 768, 16, True),      # bias, partial tiles in every dimension
    (300, 384, 320, 128, True),     # rank 128
    (130, 1536, 8960, 32, False),   # FFN-in shape
    (77, 100, 36, 3, True),         # rank 3, K not a multiple of the 32-wide k-step
    (65, 48, 80, 16, False),        # a single partial k-step
    (50, 256, 256, 0, True),        # base-only linear with bias
    (40, 22, 20, 5, True),          # K not a multiple of 4: generic kernels
    (33, 64, 30, 2, False),         # N not a multiple of 4: generic kernels
])
def test_f32_shapes(dev, M, K, N, r, bias):
    check(dev, make_case(M, K, N, r, float(r) if r else 1.0, seed=700 + M + K + N + r, bias=bias),
          f"f32 {M}x{K}x{N}r{r}")


def test_f32_wan14b_q_sampled(dev):
    # 2048 tokens of the 14B q projection; rows and columns sampled against the oracle
    import torch
    from reels_amd import QuantizedMatrix, i8lora_backward, i8lora_forward
    cs = make_case(2048, 5120, 5120, 32, 32.0, seed=750)
    print("[f32] 2048x5120x5120 r32 (sampled)", flush=True)
    W = QuantizedMatrix(todev(cs["q"], dev), todev(cs["s"], dev), torch.float32)
    x, A, B = todev(cs["x"], dev), todev(cs["A"], dev), todev(cs["B"], dev)
    y, h = i8lora_forward(x, W, A, B, None, cs["c"], save_h=True)
    dx, dA, dB = i8lora_backward(todev(cs["dy"], dev), x, W, A, B, cs["c"], h=h)
    torch.cuda.synchronize(dev)
    rows = np.array([0, 1, 127, 128, 1023, 2000, 2047])
    yr, hr = oracle.lora_forward(cs["x"], cs["q"], cs["s"], cs["A"], cs["B"], cs["c"], rows=rows,
                                 elt="f32")
    ref = oracle.lora_backward(cs["dy"], cs["x"], cs["q"], cs["s"], cs["A"], cs["B"], cs["c"],
                               rows=rows, kcols=[0, 77, 5119], ncols=[1, 4096, 5119], elt="f32")
    assert_parity(y.cpu().numpy()[rows], yr, "f32 14b-q y (sampled rows)", tol=TOL)
    assert_parity(h.cpu().numpy()[rows], hr, "f32 14b-q h (sampled rows)", tol=TOL)
    assert_parity(dx.cpu().numpy()[rows], ref["dx"], "f32 14b-q dx (sampled rows)", tol=TOL)
    assert_parity(dA.cpu().numpy()[[0, 77, 5119]], ref["dA"], "f32 14b-q dA (sampled)", tol=TOL)
    assert_parity(dB.cpu().numpy()[:, [1, 4096, 5119]], ref["dB"], "f32 14b-q dB (sampled)",
                  tol=TOL)
    # size-independent: scaling x by 2 scales y, h, dA exactly (powers of two are exact in f32)
    y2, h2 = i8lora_forward(x * 2, W, A, B, None, cs["c"], save_h=True)
    torch.cuda.synchronize(dev)
    assert torch.equal(y2, y * 2) and torch.equal(h2, h * 2)


def test_f32_backward_bitwise_reproducible(dev):
    cs = make_case(600, 512, 768, 32, 32.0, seed=760)
    a, b = run_gpu(dev, cs), run_gpu(dev, cs)
    for k in ("y", "h", "dx", "dA", "dB"):
        assert np.array_equal(a[k], b[k]), k


def test_f32_mirror_api_autograd_and_transfer(dev):
    import torch
    from reels_amd import (I8LoRALinearFunction, LoRALinear, frozen_weight_transfer,
                           lora_backward, lora_forward, move_weight)
    t = frozen_weight_transfer("hip", "fp32", quantization="int8")
    w = todev(f32v(770, (384, 256), 0.02), dev)
    W = move_weight(w, t)
    assert W.compute_dtype == torch.float32
    q, s, _ = oracle.pack(w.cpu().numpy(), "f32")
    assert np.array_equal(W.values.cpu().numpy(), q)
    layer = LoRALinear(W, rank=16, alpha=32.0)
    assert layer.A.dtype == torch.float32 and layer.B.dtype == torch.float32
    layer.B = todev(f32v(771, (16, 384), 0.05), dev)
    x = todev(f32v(772, (3, 50, 256), 1.0), dev)
    y, h = lora_forward(layer, x, save_h=True)
    assert y.dtype == torch.float32 and y.shape == (3, 50, 384)
    dy = todev(f32v(773, (3, 50, 384), 1.0), dev)
    g = lora_backward(layer, x, dy, h=h)
    A = layer.A.clone().requires_grad_(True)
    B = layer.B.clone().requires_grad_(True)
    xx = x.reshape(-1, 256).clone().requires_grad_(True)
    out = I8LoRALinearFunction.apply(xx, A, B, W.values, W.scales, None, layer.lora_scale)
    out.backward(dy.reshape(-1, 384))
    torch.cuda.synchronize(dev)
    assert torch.equal(out.reshape(3, 50, 384), y)
    assert torch.equal(xx.grad.reshape(3, 50, 256), g["dx"])
    assert torch.equal(A.grad, g["A"]) and torch.equal(B.grad, g["B"])
    # the forward against the oracle through the layer API
    yo, _ = oracle.lora_forward(x.reshape(-1, 256).cpu().numpy(), q, s, layer.A.cpu().numpy(),
                                layer.B.cpu().numpy(), layer.lora_scale, elt="f32")
    assert_parity(y.reshape(-1, 384).cpu().numpy(), yo, "f32 layer y", tol=TOL)


@pytest.mark.parametrize("n", [1, 1000, 65537])
def test_f32_gelu_tanh(dev, n):
    import torch
    from reels_amd import gelu_tanh, gelu_tanh_backward
    xs, dys = f32v(780 + n, (n,), 2.0), f32v(781 + n, (n,), 1.0)
    y = gelu_tanh(todev(xs, dev)).cpu().numpy()
    dx = gelu_tanh_backward(todev(xs, dev), todev(dys, dev)).cpu().numpy()
    assert y.dtype == np.float32 and dx.dtype == np.float32
    yo, dxo = oracle.gelu_tanh(xs, elt="f32"), oracle.gelu_tanh_backward(xs, dys, elt="f32")
    # Device and host f32 tanh may differ in their last bits (t = tanh(...) within a couple of
    # ulps of magnitude <= 1, i.e. 2^-23 absolute). For x < 0, 1 + t cancels, so y = 0.5 x (1 + t)
    # inherits an absolute error up to 0.5 |x| 2^-23 (about 16 ulps of y near x = -2), and the
    # derivative 0.5 (1 + t) + 0.5 x (1 - t^2) k (1 + 3 a x^2) one up to
    # (1 + |x| + 0.14 |x|^3) 2^-23 times |dy|. Allowed: 8 ulps of the result, or those bounds.
    x64 = np.abs(xs.astype(np.float64))
    for got, want, what in ((y, yo, "y"), (dx, dxo, "dx")):
        e = np.abs(got.astype(np.float64) - want.astype(np.float64))
        ok = e <= 8 * np.spacing(np.abs(want)).astype(np.float64) + 2.0 ** -40
        if what == "y":
            ok |= e <= x64 * 2.0 ** -22
        else:
            ok |= e <= (1 + x64 + 0.14 * x64 ** 3) * 2.0 ** -22 * np.abs(dys.astype(np.float64))
        bad = np.flatnonzero(~ok)
        assert bad.size == 0, (what, [(int(i), float(got[i]), float(want[i]), float(xs[i]))
                                      for i in bad[:6]])


@pytest.mark.parametrize("M,K,N,r,bias", [
    (1, 130, 66, 2, True),       # one token; K, N not multiples of 4; split reductions
    (257, 63, 65, 5, True),      # lengths around one GEMM step of 64, rank not a multiple of 4
    (129, 65, 257, 40, False),   # a second output tile of one column, rank above one LDS tile
    (33, 191, 1, 1, True),       # one output column
    (300, 320, 260, 160, True),  # rank above one chunk of 128
    (2100, 72, 1000, 24, True),  # many token splits, ragged output columns
])
def test_f32_plane_gemm_edges(dev, M, K, N, r, bias):
    """The products on bf16 planes at the edges of their tiles and steps: every output against the
    oracle within the file's 1e-5 (the planes are exact, the sums f32), and the result of an unaligned
    (4-byte aligned) x equal to that of an aligned copy bit for bit (every operand:
    test_f32_operands_off_their_alignment)."""
    import torch
    from reels_amd import QuantizedMatrix, i8lora_forward
    cs = make_case(M, K, N, r, float(r), seed=900 + M + K + N + r, bias=bias)
    g = check(dev, cs, f"planes {M}x{K}x{N}r{r}")
    flat = torch.zeros((M * K + 1,), device=dev)
    flat[1:] = todev(cs["x"], dev).reshape(-1)
    x = flat[1:].view(M, K)
    assert x.data_ptr() % 16 != 0
    W = QuantizedMatrix(todev(cs["q"], dev), todev(cs["s"], dev), torch.float32)
    y, _ = i8lora_forward(x, W, todev(cs["A"], dev), todev(cs["B"], dev),
                          todev(cs["bias"], dev) if bias else None, cs["c"])
    torch.cuda.synchronize(dev)
    assert np.array_equal(y.cpu().numpy(), g["y"])


def test_f32_token_chunks(dev):
    # 40200 tokens x 8960: the planes of x would exceed 2 GiB, so the forward runs as chunks; rows on
    # both sides of multiples of 256 tokens against f64 products
    import torch
    from reels_amd import QuantizedMatrix, i8lora_forward
    M, K, N, r = 40200, 8960, 96, 8
    print(f"[f32] token chunks {M}x{K}x{N}r{r}", flush=True)
    g = torch.Generator(device=dev).manual_seed(3)
    x = torch.randn((M, K), generator=g, device=dev)
    q = torch.randint(-127, 128, (N, K), generator=g, device=dev).to(torch.int8)
    s = torch.rand((N,), generator=g, device=dev) * 1e-3
    A = torch.randn((K, r), generator=g, device=dev) * 0.01
    B = torch.randn((r, N), generator=g, device=dev) * 0.01
    y, h = i8lora_forward(x, QuantizedMatrix(q, s, torch.float32), A, B, None, 0.5, save_h=True)
    rows = torch.tensor([0, 255, 20223, 20224, 20479, 20480, 40199], device=dev)
    xd = x[rows].double()
    hd = xd @ A.double()
    yd = xd @ (q.double() * s.double()[:, None]).t() + 0.5 * hd @ B.double()
    assert_parity(y[rows].cpu().numpy(), yd.cpu().numpy(), "chunked y", tol=TOL)
    assert_parity(h[rows].cpu().numpy(), hd.cpu().numpy(), "chunked h", tol=TOL)


def test_f32_special_values(dev):
    """Infinities and NaNs reach exactly the rows they are in, values near the ends of the f32 range
    keep f32's relative precision, scales of zero and of subnormal size multiply as fl32(q s)."""
    import torch
    from reels_amd import QuantizedMatrix, i8lora_backward, i8lora_forward
    M, K, N = 9, 70, 12
    x = f32v(950, (M, K), 1.0)
    q = np.random.default_rng(951).integers(1, 128, (N, K)).astype(np.int8)
    s = np.full(N, 1e-3, np.float32)
    s[3], s[4], s[5] = 0.0, 1e-39, -2e-3
    x[1, 7], x[2, 7], x[3, 7], x[3, 9] = np.inf, np.nan, np.inf, -np.inf
    x[4] *= np.float32(1e34)
    x[5] *= np.float32(1e-30)
    x[6, 0] = np.uint32(0x7f800001).view(np.float32)  # a NaN whose upper half alone is Inf
    W = QuantizedMatrix(todev(q, dev), todev(s, dev), torch.float32)
    y = i8lora_forward(todev(x, dev), W)[0].cpu().numpy()
    with np.errstate(all="ignore"):
        ref = x.astype(np.float64) @ (q.astype(np.float64) * s.astype(np.float64)[:, None]).T
    ok = s != 0  # Inf times a zero weight is NaN
    assert np.isinf(y[1, ok]).all() and (np.sign(y[1, ok]) == np.sign(s[ok])).all()
    assert np.isnan(y[2]).all() and np.isnan(y[3]).all() and np.isnan(y[6]).all()
    for m in (0, 4, 5, 7, 8):
        big = np.abs(ref[m]) > 1e-36  # results above f32's subnormal range
        scale = np.abs(x[m].astype(np.float64)) @ (np.abs(q.astype(np.float64)) * np.abs(s)[:, None]).T
        assert (np.abs(y[m] - ref[m])[big] <= 1e-6 * scale[big]).all(), m
    assert (y[0, 3] == 0) and (y[4, 3] == 0)
    dy = f32v(952, (M, N), 1.0)
    dy[1, 2], dy[2, 3] = np.inf, np.nan
    dx = i8lora_backward(todev(dy, dev), None, W, want_dA=False, want_dB=False)[0].cpu().numpy()
    assert np.isinf(dx[1]).all() and np.isnan(dx[2]).all() and np.isfinite(dx[[0, 3, 4]]).all()


@pytest.mark.parametrize("M,K,N,r", [
    (6000, 8960, 300, 8),    # the forward in chunks, the last a shorter one with a split of its own
    (6000, 300, 8960, 24),   # dX in chunks
])
def test_f32_chunks_of_bounded_planes(dev, M, K, N, r):
    """Calls whose planes would take more than 256 MiB run as chunks of their tokens: every output in
    full against f64 products, h given and recomputed."""
    import torch
    from reels_amd import QuantizedMatrix, i8lora_backward, i8lora_forward
    print(f"[f32] bounded planes {M}x{K}x{N}r{r}", flush=True)
    g = torch.Generator(device=dev).manual_seed(M + K)
    rn = lambda *sh: torch.randn(sh, generator=g, device=dev)
    x, dy, A, B, bias = rn(M, K), rn(M, N), rn(K, r) * 0.01, rn(r, N) * 0.01, rn(N)
    q = torch.randint(-127, 128, (N, K), generator=g, device=dev).to(torch.int8)
    s = torch.rand((N,), generator=g, device=dev) * 1e-3
    W = QuantizedMatrix(q, s, torch.float32)
    y, h = i8lora_forward(x, W, A, B, bias, 0.5, save_h=True)
    first = i8lora_backward(dy, x, W, A, B, 0.5, h=h)
    again = i8lora_backward(dy, x, W, A, B, 0.5, h=None)
    torch.cuda.synchronize(dev)
    assert all(torch.equal(a, b) for a, b in zip(first, again))
    Wd, xd, dyd, Ad, Bd = q.double() * s.double()[:, None], x.double(), dy.double(), A.double(), B.double()
    hd, ud = xd @ Ad, dyd @ Bd.t()
    ref = (xd @ Wd.t() + bias.double() + 0.5 * hd @ Bd, hd, dyd @ Wd + 0.5 * ud @ Ad.t(),
           0.5 * xd.t() @ ud, 0.5 * hd.t() @ dyd)
    for name, a, b in zip(("y", "h", "dx", "dA", "dB"), (y, h) + tuple(first), ref):
        assert_parity(a.cpu().numpy(), b.cpu().numpy(), f"bounded planes {name}", tol=TOL)


@pytest.mark.parametrize("M,K,N,r", [
    (300, 320, 260, 4),    # the adapter tiles in LDS, rows of 16 bytes
    (77, 130, 515, 24),    # split reductions, widths that are no multiples of 4
    (2100, 256, 1000, 32),  # several token splits
    (40, 200, 96, 40),     # ranks above the LDS tile
])
def test_f32_operands_off_their_alignment(dev, M, K, N, r):
    """Every f32 operand and output one element (the codes one byte) past a 16-byte boundary: forward
    with h and bias, backward with h given and recomputed and with the bias gradient, bit for bit as
    with aligned ones."""
    import ctypes
    import torch
    from reels_amd import _lib
    L = _lib.lib()
    print(f"[f32] unaligned {M}x{K}x{N}r{r}", flush=True)
    cs = make_case(M, K, N, r, float(r), seed=1300 + M, bias=True)
    dy = f32v(1301 + M, (M, N), 1.0)
    st = ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)
    nb = max(L.reels_hip_i8lora_workspace_bytes_f32(M, K, N, r, w) for w in (0, 1))
    ws = torch.empty((nb,), dtype=torch.uint8, device=dev)
    assert ws.data_ptr() % 256 == 0

    def shifted(a, off):
        flat = torch.empty((a.numel() + 16,), dtype=a.dtype, device=dev)[off:off + a.numel()]
        return flat.copy_(a.reshape(-1)).view(a.shape)

    def run(off):
        x, A, B, bias, q, s, d = (shifted(todev(a, dev), off) for a in
                                  (cs["x"], cs["A"], cs["B"], cs["bias"], cs["q"], cs["s"], dy))
        y, h, dx, dA, dB, db = (shifted(torch.zeros(sh, device=dev), off) for sh in
                                ((M, N), (M, r), (M, K), (K, r), (r, N), (N,)))
        assert all((t.data_ptr() % 16 != 0) == (off > 0) for t in (x, A, B, bias, q, s, d, y, h, dx, dA, dB, db))
        p = lambda t: ctypes.c_void_p(t.data_ptr())
        _lib.check("fwd", L.reels_hip_i8lora_fwd_f32(
            p(x), p(q), p(s), p(A), p(B), p(bias), M, K, N, r, 0.5, p(y), p(h), p(ws), nb, st))
        out = [y, h]
        for hp in (p(h), None):
            _lib.check("bwd", L.reels_hip_i8lora_bwd_bias_f32(
                p(d), p(x), hp, p(q), p(s), p(A), p(B), M, K, N, r, 0.5, p(dx), p(dA), p(dB), p(db), p(ws), nb, st))
            out += [t.clone() for t in (dx, dA, dB, db)]
        torch.cuda.synchronize(dev)
        return out
    names = ("y", "h") + 2 * ("dx", "dA", "dB", "dbias")
    for name, a, b in zip(names, run(0), run(1)):
        assert torch.equal(a, b), name


def test_f32_generic_kernels(dev):
    """A workspace off its 16-byte alignment: the one-output-per-thread kernels, against the oracle."""
    import ctypes
    import torch
    from reels_amd import _lib
    L = _lib.lib()
    M, K, N, r = 33, 70, 50, 5
    print("[f32] generic kernels", flush=True)
    cs = make_case(M, K, N, r, float(r), seed=1400, bias=True)
    x, A, B, bias, q, s, dy = (todev(cs[k], dev) for k in ("x", "A", "B", "bias", "q", "s", "dy"))
    nb = max(L.reels_hip_i8lora_workspace_bytes_f32(M, K, N, r, w) for w in (0, 1))
    ws = torch.empty((nb + 16,), dtype=torch.uint8, device=dev)[4:4 + nb]
    y, h, dx, dA, dB, db = (torch.zeros(sh, device=dev) for sh in ((M, N), (M, r), (M, K), (K, r), (r, N), (N,)))
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    st = ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)
    c = cs["c"]
    _lib.check("fwd", L.reels_hip_i8lora_fwd_f32(
        p(x), p(q), p(s), p(A), p(B), p(bias), M, K, N, r, c, p(y), p(h), p(ws), nb, st))
    yo, ho = oracle.lora_forward(cs["x"], cs["q"], cs["s"], cs["A"], cs["B"], c, cs["bias"], elt="f32")
    ref = oracle.lora_backward(cs["dy"], cs["x"], cs["q"], cs["s"], cs["A"], cs["B"], c, elt="f32")
    for hp in (p(h), None):
        _lib.check("bwd", L.reels_hip_i8lora_bwd_bias_f32(
            p(dy), p(x), hp, p(q), p(s), p(A), p(B), M, K, N, r, c, p(dx), p(dA), p(dB), p(db), p(ws), nb, st))
        torch.cuda.synchronize(dev)
        for name, a, b in (("y", y, yo), ("h", h, ho), ("dx", dx, ref["dx"]), ("dA", dA, ref["dA"]),
                           ("dB", dB, ref["dB"]), ("dbias", db, oracle.bias_gradient(cs["dy"], elt="f32"))):
            assert_parity(a.cpu().numpy(), b, f"generic {name}", tol=TOL)


def test_f32_results_near_the_end_of_the_range(dev):
    """y and dx of up to 3.2e38 from single terms, scales on both sides of a power of two: the scale's
    parts overflow on neither side of the products."""
    import torch
    from reels_amd import QuantizedMatrix, i8lora_backward, i8lora_forward
    print("[f32] near the end of the range", flush=True)
    K, N = 70, 9
    q = np.full((N, K), 127, np.int8)
    s = (np.float32(2.0 ** -7) * np.float32([1.0, 1.01, 1.3, 1.6, 1.99, 0.51, 0.75, 0.99, 1.0001])).astype(np.float32)
    W = QuantizedMatrix(todev(q, dev), todev(s, dev), torch.float32)
    x = np.zeros((N, K), np.float32)  # row n for scale n
    x[:, 5] = np.minimum(3.2e38 / (s.astype(np.float64) * 127), 3.3e38)
    dy = np.zeros((N, N), np.float32)
    dy[np.arange(N), np.arange(N)] = x[:, 5]
    y = i8lora_forward(todev(x, dev), W)[0].cpu().numpy()
    dx = i8lora_backward(todev(dy, dev), None, W, want_dA=False, want_dB=False)[0].cpu().numpy()
    want = x[:, 5].astype(np.float64) * 127 * s
    assert want.max() > 3e38
    d = np.arange(N)
    assert (np.abs(y[d, d] - want) <= 4 * 2.0 ** -24 * want).all()
    assert (np.abs(dx - want[:, None]) <= 4 * 2.0 ** -24 * want[:, None]).all()
