"""The LDS-fed FP8 weight kernels (csrc/dense_fp8.hip): the loader-wave kernel and the 128-row tiles behind dsv41_fp8_gemm
(5 to 64 rows) and dsv41_fp8_gemm_rows (any number), at the edges of their ranges: partial row blocks and token tiles, odd
chunk counts, one chunk per wave or none, every K split, column groups, unaligned operands (which keep the older kernel).

Products of bf16 and E4M3 x 2^e are exact in fp32, so only the order of the fp32 sums differs from the 64-bit result. A chain of n
sums of random sign rounds partial sums of rms sqrt(k), k = 1 .. n; rounding errors of 2^-24 / sqrt(3) of them add up to 2^-24 sqrt(n / 6) of
the result's rms. An accumulator takes one product of 32 k at a time, so n = K / 32: 3.6e-7 at the longest K here (7168). Measured:
at most 2.7e-7. REL is about four times that."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
REL = 1e-6


def _operands(M, N, K, seed, G=1):
    g = torch.Generator(device=DEV).manual_seed(seed)
    w = torch.randn(N, K, generator=g, device=DEV).to(torch.float8_e4m3fn).view(torch.uint8)
    s = torch.randint(119, 124, ((N + 31) // 32, K // 32), generator=g, device=DEV, dtype=torch.uint8)
    x = torch.randn(M * G, K, generator=g, device=DEV).to(torch.bfloat16)
    deq = w.view(torch.float8_e4m3fn).double() * torch.pow(2.0, s.double() - 127).repeat_interleave(32, 0)[:N].repeat_interleave(32, 1)
    return w, s, x, deq


def _close(got, ref, what):
    err = ((got.double() - ref).norm() / ref.norm()).item()
    print(f"{what}: rel {err:.1e}", flush=True)
    assert err <= REL, f"{what}: {err:.2e}"


# (M, N, K, group columns): one, two and four row blocks per workgroup and the tiles; K chunks 16 .. 129
UP_TO_64 = [(5, 1280, 2048, 0), (16, 1000, 4160, 0), (17, 2064, 1024, 0), (33, 4080, 1088, 0), (64, 3328, 7168, 0), (48, 512, 5120, 0),
            (9, 4112, 2304, 0), (16, 7168, 1664, 0), (31, 4104, 1280, 0), (49, 8192, 1024, 0), (64, 5128, 2112, 0),
            (16, 10240, 4096, 0), (33, 8208, 1024, 0), (64, 12296, 1088, 0), (17, 24576, 1024, 0), (40, 24600, 1088, 0), (64, 32768, 192, 0),
            (20, 4096, 1024, 32), (20, 4096, 1024, 16), (50, 16384, 1024, 64), (20, 24576, 1024, 128),
            (5, 1280, 4096, 0), (8, 3072, 2112, 0), (12, 3344, 2112, 0), (11, 24592, 4160, 0), (33, 16400, 768, 0)]


def _layouts(cases):
    """Each case row-major and, where its rows fill the 16-row blocks of the tile order, tiled."""
    return [(*c, tiled) for c in cases for tiled in ((False, True) if c[1] % 16 == 0 else (False,))]


@pytest.mark.parametrize("M,N,K,gc,tiled", _layouts(UP_TO_64))
def test_fp8_up_to_64_rows(M, N, K, gc, tiled):
    from dsv41_amd import hipkern, w8
    print(f"fp8 M={M} N={N} K={K} gc={gc} tiled={tiled}", flush=True)
    G = N // gc if gc else 1
    w, s, x, deq = _operands(M, N, K, M + N + K, G)
    if gc:
        ref = torch.stack([x.double().view(M, G, K)[:, q] @ deq[q * gc:(q + 1) * gc].t() for q in range(G)], 1).reshape(M, N)
    else:
        ref = x.double() @ deq.t()
    wk = w8.tile(w) if tiled else w
    y = hipkern.fp8_gemm_tc(x, wk, s, group_cols=gc, out_dtype=torch.float32, tiled=tiled)
    _close(y, ref, "fp32")
    assert torch.equal(hipkern.fp8_gemm_tc(x, wk, s, group_cols=gc, tiled=tiled), y.to(torch.bfloat16))
    if not gc:   # operands off the 16-byte grid keep the older kernel, with the same values up to summation order
        off = torch.empty(M * K + 3, device=DEV, dtype=torch.bfloat16)[3:].view(M, K).copy_(x)
        _close(hipkern.fp8_gemm_tc(off, wk, s, out_dtype=torch.float32, tiled=tiled), ref, "unaligned x")


@pytest.mark.parametrize("M,N,K,tiled", _layouts([(65, 1280, 1088), (128, 136, 192), (129, 400, 2048), (333, 1040, 4160), (64, 512, 64), (1, 264, 320)]))
def test_fp8_gemm_rows(M, N, K, tiled):
    from dsv41_amd import _lib, w8
    w, s, x, deq = _operands(M, N, K, M + N + K)
    ref = x.double() @ deq.t()
    wk = w8.tile(w) if tiled else w
    for tile in (64, 128):
        for splits in sorted({1, 2, min(5, K // 64), K // 64}):
            if splits > K // 64:
                continue
            print(f"fp8 rows M={M} N={N} K={K} tiled={tiled} tile={tile} splits={splits}", flush=True)
            out = torch.empty(M, N, device=DEV)
            outb = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
            part = torch.empty(splits * M * N, device=DEV)
            _lib.call("dsv41_fp8_gemm_rows", _lib.ptr(wk), K, 1 if tiled else 0, _lib.ptr(s), s.stride(0), N, K, _lib.ptr(x), K, M, _lib.ptr(out), N,
                      _lib.ptr(outb), N, tile, splits, _lib.ptr(part), part.numel(), _lib.stream(DEV))
            _close(out, ref, f"tile {tile} splits {splits}")
            assert torch.equal(outb, out.to(torch.bfloat16))
    bad = lambda **kw: _lib.lib().dsv41_fp8_gemm_rows(
        _lib.ptr(wk), K, 1 if tiled else 0, _lib.ptr(s), s.stride(0), N, K, kw.get("x", _lib.ptr(x)), kw.get("ldx", K), M, _lib.ptr(out), N, None, 0,
        kw.get("tile", 64), kw.get("splits", 2), _lib.ptr(part), kw.get("floats", part.numel()), _lib.stream(DEV))
    assert bad(tile=32) == -1 and bad(splits=0) == -1 and bad(splits=K // 64 + 1) == -1 and bad(ldx=K + 4) == -1
    if K >= 128:
        assert bad(floats=2 * M * N - 1) == -1


@pytest.mark.parametrize("M", [40, 70, 400])
def test_every_code_and_scale(M):
    """Each E4M3 code (NaN among them) under each scale byte 0 .. 255 (products below the normal range, infinities), picked by one-hot
    rows on the loader-wave kernel and both tile heights: the dequantised weight, as the library product of it gives it. A NaN
    or infinite weight makes NaN of its whole row (0 times it) on either side."""
    from dsv41_amd import hipkern, w8
    K, N, c0 = 1024, 256 * 32, 8 * (M // 10)
    code = 8 * (torch.arange(N) % 32)[:, None] + torch.arange(8)
    w = torch.zeros(N, K, dtype=torch.uint8)
    w[:, c0:c0 + 8] = code.to(torch.uint8)            # row n of a scale block: codes 8 (n % 32) ..
    W = w8.W8(w.to(DEV), torch.arange(256, dtype=torch.uint8)[:, None].expand(256, K // 32).contiguous().to(DEV))
    assert M <= 64 or hipkern.fp8_rows_plan(M, N, K) == ((64, 1) if M == 70 else (128, 1))
    x = torch.zeros(M, K, dtype=torch.bfloat16, device=DEV)
    for j in range(8):
        x[M - 1 - j, c0 + j] = 1.0
    y, lib = w8.linear_w(x, W), torch.nn.functional.linear(x, W.bf16())
    assert torch.equal(y.isnan(), lib.isnan()) and torch.equal(y[~y.isnan()], lib[~lib.isnan()])
    assert bool(y.isnan().any()) and bool((y == 0).any()) and bool((y.abs() > 1e38).any())


def test_linear_w_rows_plan_and_watchers():
    """linear_w past 64 rows: the tiles give the library route's values; calls that something watches keep the library."""
    from dsv41_amd import hipkern, w8
    M, N, K = 200, 768, 2048
    w, s, x, deq = _operands(M, N, K, 3)
    W = w8.W8(w, s)
    assert hipkern.fp8_rows_plan(M, N, K) is not None and w8._tiles_ok(x, W)
    lib = torch.nn.functional.linear(x, W.bf16())
    y = w8.linear_w(x, W)
    ref = x.double() @ deq.t()
    err = lambda v: ((v.double() - ref).norm() / ref.norm()).item()
    assert err(y) <= 1.01 * err(lib)                                   # one bf16 rounding each
    strided = torch.zeros(M, K + 8, device=DEV, dtype=torch.bfloat16)[:, :K].copy_(x)
    assert torch.equal(w8.linear_w(strided, W), y)
    xg = x.clone().requires_grad_(True)
    w8.linear_w(xg, W).float().sum().backward()
    assert xg.grad is not None
    out = torch.func.vmap(lambda r: w8.linear_w(r, W))(x.view(2, M // 2, K))
    assert torch.allclose(out.reshape(M, N).float(), lib.float(), rtol=2 ** -7, atol=1e-2 * lib.float().std().item())
    from torch.utils.flop_counter import FlopCounterMode
    with FlopCounterMode(display=False) as flops:
        assert torch.equal(w8.linear_w(x, W), lib)
    assert flops.get_total_flops() == 2 * M * N * K
    with torch.autocast("cuda", dtype=torch.float16):
        assert w8.linear_w(x, W).dtype == torch.float16
    g = torch.cuda.CUDAGraph()
    w8.linear_w(x, W)
    with torch.cuda.graph(g):
        yg = w8.linear_w(x, W)
    for _ in range(3):
        yg.zero_()
        g.replay()
        assert torch.equal(yg, y)
