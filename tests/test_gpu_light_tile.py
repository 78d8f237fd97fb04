"""The 64-pair tile of the prefill kernels (dsv41_prefill_up_g64 / _down_g64, dsv41_fp4_grouped_gemm_t64 / _scatter_g64) at
the edges of its range: group sizes either side of a token block and of the tile (larger groups in passes), experts with one
group and with several, both weight layouts, the shortest k-loops; and with the pairs' scale bytes in one load for four k-steps
(K % 512 == 0) over one, two, three and four such loads, whose two buffers switch at the second and are filled again from the third on. Every pair's row is the same sum in the same order as on
the larger tiles (which are checked against the oracle in test_gpu_moe.py), so the results are equal bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")

#        expert, pairs: an expert's groups lie together, as a dispatch leaves them
GROUPS = [(0, 1), (1, 15), (2, 16), (3, 17), (4, 63), (5, 64), (5, 33), (6, 65), (7, 128), (8, 32), (9, 48), (9, 64), (9, 2), (11, 5)]


def _setup(H, I, tiled, seed):
    from dsv41_amd import moe, quant
    E, T = 12, 77
    g = torch.Generator(device=DEV).manual_seed(seed)
    b = lambda *s: torch.randint(0, 256, s, generator=g, dtype=torch.uint8, device=DEV)
    sc = lambda *s: torch.randint(119, 124, s, generator=g, dtype=torch.uint8, device=DEV)
    w13, s13, w2, s2 = b(E, 2 * I, H // 2), sc(E, 2 * I, H // 32), b(E, H, I // 2), sc(E, H, I // 32)
    if tiled:
        w13, w2, s13, s2 = quant.tile_fp4(w13), quant.tile_fp4(w2), quant.tile_fp4_scales(s13), quant.tile_fp4_scales(s2)
    P = sum(n for _, n in GROUPS)
    x = torch.randn(T, H, generator=g, device=DEV).to(torch.bfloat16)
    i32 = lambda a: torch.tensor(a, dtype=torch.int32, device=DEV)
    tab = (i32([e for e, _ in GROUPS] + [-1]), i32(np.concatenate([[0], np.cumsum([n for _, n in GROUPS]), [P]])))
    tok = torch.randint(0, T, (P,), generator=g, device=DEV, dtype=torch.int32)
    wt = torch.rand(P, generator=g, device=DEV)
    return moe.ExpertWeights(w13, s13, w2, s2, tiled), x, tab, tok, wt, P


@pytest.mark.parametrize("tiled", [True, False])
@pytest.mark.parametrize("H,I", [(512, 384), (768, 640), (1024, 1536), (1536, 1024), (2048, 512)])
def test_light_tile_equals_the_larger_tiles(H, I, tiled):
    from dsv41_amd import _lib, hipkern, quant
    print(f"light tile H={H} I={I} tiled={tiled}", flush=True)
    ex, x, (ge, gs), tok, wt, P = _setup(H, I, tiled, H + I)
    G, dev = ge.numel(), x.device
    xc, xs = quant.quant_fp8_e8m0(x)
    got = {}
    for suffix in ("", "_g64"):
        hc = torch.zeros(P, I, dtype=torch.uint8, device=dev)
        hs = torch.zeros(P, I // 32, dtype=torch.uint8, device=dev)
        y2 = torch.zeros(P, H, device=dev)
        _lib.call("dsv41_prefill_up" + suffix, _lib.ptr(xc), xc.stride(0), _lib.ptr(xs), xs.stride(0), x.shape[0], _lib.ptr(ex.w13),
                  ex.w13.stride(0), _lib.ptr(ex.s13), ex.s13.stride(0), 1 if tiled else 0, ex.E, H, I, _lib.ptr(ge), _lib.ptr(gs), G,
                  _lib.ptr(tok), _lib.ptr(wt), 10.0, _lib.ptr(hc), hc.stride(0), _lib.ptr(hs), hs.stride(0), None, _lib.stream(dev))
        _lib.call("dsv41_prefill_down" + suffix, _lib.ptr(hc), hc.stride(0), _lib.ptr(hs), hs.stride(0), P, _lib.ptr(ex.w2), ex.w2.stride(0),
                  _lib.ptr(ex.s2), ex.s2.stride(0), 1 if tiled else 0, ex.E, H, I, _lib.ptr(ge), _lib.ptr(gs), G, _lib.ptr(y2), y2.stride(0),
                  None, _lib.stream(dev))
        # the general grouped GEMM with both FP8 terms of x (the second pass adds), and its scatter form
        hi, his, lo, los, flag = quant.quant_fp8_split(x)
        yt = torch.zeros(P, H, device=dev)
        n = H // 256 * 256
        hipkern.grouped_gemm_t128(hi, his, ex.w13[:, :n], ex.s13[:, :n], ge, gs, tok, yt, P, tiled, lo=(lo, los, flag),
                                  max_tokens=64 if suffix else 128)
        out = torch.zeros(P, n, device=dev)
        rows = torch.arange(P - 1, -1, -1, dtype=torch.int32, device=dev)
        one = torch.ones(1, dtype=torch.int32, device=dev)
        hipkern.grouped_gemm_scatter(hi, his, ex.w13[:, :n], ex.s13[:, :n], ge, gs, tok, rows, wt, one, False, out, P, tiled,
                                     lo=(lo, los, flag), gmax=64 if suffix else 256)
        # FP8-grid x (no second term): the light tile stores the weighted rows of a new output itself; rows out of range are
        # skipped, a given output is added to, shared rows take the atomic form (integers here: any order gives the same sums)
        flag0 = torch.zeros(1, dtype=torch.int32, device=dev)
        rows2 = rows.clone()
        rows2[5], rows2[70] = -1, P
        outs = []
        for accum, distinct, ro, w in ((False, one, rows2, wt), (True, one, rows, wt), (False, flag0, rows // 4, None)):
            o = torch.ones(P, n, device=dev) if accum else torch.zeros(P, n, device=dev)
            sc = his if w is not None else torch.full_like(his, 127)
            ws = ex.s13[:, :n] if w is not None else torch.full_like(ex.s13, 128)[:, :n]
            ints = hi if w is not None else torch.randint(0, 2, hi.shape, generator=torch.Generator(device=dev).manual_seed(9), device=dev,
                                                          dtype=torch.uint8) * 0x38      # 0 or 1.0
            hipkern.grouped_gemm_scatter(ints, sc, ex.w13[:, :n], ws, ge, gs, tok, ro, wt if w is not None else torch.ones_like(wt), distinct, accum, o,
                                         P, tiled, lo=(torch.zeros_like(lo), los, flag0), gmax=64 if suffix else 256)
            outs.append(o)
        got[suffix] = (hc, hs, y2, yt, out, *outs)
    names = ("h codes", "h scales", "y2", "grouped", "scatter", "stored", "added", "atomic")
    for name, a, b in zip(names, got[""], got["_g64"]):
        assert torch.equal(a, b), name
    assert all(bool(t.any()) for t in got["_g64"])
