"""FP4 expert kernels with the call surface of the reference's cukern.py (fp4_gemv_pairs, fp4_gemm_tc,
permute_x, moe_dispatch), on the HIP library instead of libcuda-launched cubins.

Activations are bf16, as the reference's kernels take them (fp4_gemv.cu and fp4_tcw.cu multiply bf16 x by bf16-decoded
weights). The kernels take x in the MFMA operand format as two FP8 terms, x = hi + lo (E4M3 codes + E8M0 bytes per 32
each, quant.quant_fp8_split's encoding). hi + lo reproduces every bf16 value (up to 2^-21 of its 32-group's amax for
residuals below the lo term's normal range), so the products equal the reference's bf16 products to fp32 accumulation
order. At decode sizes (bf16_in_kernel) the kernel splits the bf16 rows itself while staging them
(dsv41_fp4_grouped_gemm_bf16: one launch); otherwise the wrappers run the split quantiser first. FP8-grid input
(fake_quant_fp8 / swiglu_quant outputs, what the reference's own callers pass) has lo = 0: the result is bit for bit
the one-term computation (a device flag skips the lo pass where it would be a second weight pass).
Outputs are allocated with torch.empty on the input's device (cukern.py:67, 251, 328-332); kernels never
allocate. All launches go to torch's current stream and can be captured in a hipGraph.
"""
from __future__ import annotations

import os

import torch

from . import _lib
from .quant import attached_codes, quant_fp8_split

FP4_TILED = os.environ.get("DSV41_FP4_TILED", "1") == "1"  # experts stored in the tile_fp4 layout (cukern.py:231)
FP4_W_MAX = 64                                              # tokens per group of the dispatch (cukern.py:232)


def permute_x(x: torch.Tensor) -> torch.Tensor:
    """bf16 [M, K] -> the 8-k permuted layout fp4_gemm_tc accepts (within every 8 k: 0,4,2,6,1,5,3,7),
    cukern.py:224-227, kept for drop-in compatibility (the HIP kernels take natural order). The order swaps the outer two
    of three bits of k, so it is one strided copy: an index list would be uploaded on every call, and the host would wait
    for it behind the work in flight."""
    M, K = x.shape
    return x.view(M, K // 8, 2, 2, 2).permute(0, 1, 4, 3, 2).reshape(M, K).contiguous()


def _quant_x(x: torch.Tensor, permuted: bool, flag: bool = True):
    """(hi codes, hi scales, (lo codes, lo scales, lo flag or None)) of bf16 x; the flag only where a kernel path skips
    a second weight pass with it (its clearing costs a launch). x carrying the codes it was written from
    (quant.attach_codes: swiglu_quant's result) needs no quantisation and no lo term: (codes, scales, None)."""
    pre = attached_codes(x, permuted)
    if pre is not None:
        return pre[0], pre[1], None
    hc, hs, lc, ls, f = quant_fp8_split(x, permuted=permuted, flag=flag)
    return hc, hs, (lc, ls, f)


B_LDS_MAX_BYTES = 48 * 1024   # the grouped kernel's activation staging (csrc/gemm_fp4.hip)


def lo_in_lds(K: int, max_tokens: int) -> bool:
    """Whether dsv41_fp4_grouped_gemm runs both FP8 terms in one launch (their rows staged in LDS, passes of up to 8
    pairs whose hi and lo rows share one MFMA): then the lo term costs no second weight pass and needs no flag."""
    rows = min(min(max(1, int(max_tokens)), 16), 8)
    one = rows * (K + 16) + rows * (K // 32)
    return (one + 15) // 16 * 16 + one <= B_LDS_MAX_BYTES


def _lo_args(lo, xc: torch.Tensor, xs: torch.Tensor):
    if lo is None:
        return None, None, None
    lc, ls, flag = lo
    assert lc.shape == xc.shape and ls.shape == xs.shape and lc.stride() == xc.stride() and ls.stride() == xs.stride()
    assert flag is None or (flag.dtype == torch.int32 and flag.numel() == 1)
    return _lib.ptr(lc), _lib.ptr(ls), _lib.ptr(flag)


def grouped_gemm_codes(xc: torch.Tensor, xs: torch.Tensor, w: torch.Tensor, s: torch.Tensor, grp_expert: torch.Tensor,
                       grp_start: torch.Tensor, pair_tok: torch.Tensor, out: torch.Tensor, max_tokens: int, tiled: bool,
                       pair_wt: torch.Tensor | None = None, out_row: torch.Tensor | None = None, accum: int = 0,
                       shard_start: int = 0, shard_n: int = 1 << 30, zero_out: bool = False, n_cols: int | None = None,
                       min_tok: int = 0, max_tok: int = 1 << 30, n_pairs: int | None = None, lo=None) -> torch.Tensor:
    """Core launcher: out[out_row[p], :N] (=, +=, atomic +=) wt[p] * codes(x)[pair_tok[p]] . deq(W[e_g])^T.
    xc/xs: FP8 codes [rows, K] / E8M0 [rows, K/32]; w/s: [E, N, K/2] / [E, N, K/32] (may be a column slice);
    lo: (codes, scales, flag) of x's second FP8 term (quant_fp8_split), or None."""
    dev = _lib.require_cuda(xc, xs, w, s, grp_expert, grp_start, pair_tok, out)
    E, N, Kh = w.shape
    K = Kh * 2
    if n_cols is not None:
        N = n_cols
    assert w.stride(2) == 1 and w.stride(1) == Kh and s.stride(2) == 1 and s.stride(1) == K // 32, "weights must be row-contiguous"
    assert xc.dtype == torch.uint8 and xs.dtype == torch.uint8 and xc.shape[-1] == K and xs.shape[-1] == K // 32
    assert out.dtype == torch.float32 and out.stride(-1) == 1
    for t in (grp_expert, grp_start, pair_tok):
        assert t.dtype == torch.int32 and t.is_contiguous()
    G = grp_expert.numel()
    n_pairs = pair_tok.numel() if n_pairs is None else min(int(n_pairs), pair_tok.numel())
    assert grp_start.numel() >= G + 1 and (pair_wt is None or pair_wt.numel() >= n_pairs)
    assert out_row is not None or out.shape[0] >= n_pairs
    # W holds experts shard_start .. shard_start + E - 1 of the sharded id space (all E when unsharded)
    _lib.call("dsv41_fp4_grouped_gemm", _lib.ptr(w), w.stride(0), _lib.ptr(s), s.stride(0), 1 if tiled else 0, N, K,
              _lib.ptr(xc), xc.stride(0), _lib.ptr(xs), xs.stride(0), xc.shape[0], *_lo_args(lo, xc, xs), _lib.ptr(grp_expert),
              _lib.ptr(grp_start), G,
              _lib.ptr(pair_tok), n_pairs, _lib.ptr(out), out.stride(0), out.shape[0], _lib.ptr(out_row), _lib.ptr(pair_wt), accum,
              max(1, int(max_tokens)), shard_start, min(shard_n, E), 1 if zero_out else 0, min_tok, max_tok, _lib.stream(dev))
    return out


def bf16_in_kernel(x: torch.Tensor, K: int, max_tokens: int) -> bool:
    """Whether dsv41_fp4_grouped_gemm_bf16 takes x as it is: bf16 rows of 16-byte pieces whose two FP8 terms the kernel
    splits while staging them (lo_in_lds: both terms fit its LDS), so no quantiser launch runs first."""
    return (x.dtype == torch.bfloat16 and x.dim() == 2 and x.stride(1) == 1 and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0
            and lo_in_lds(K, max_tokens))


def grouped_gemm_bf16(x: torch.Tensor, permuted: bool, w: torch.Tensor, s: torch.Tensor, grp_expert: torch.Tensor,
                      grp_start: torch.Tensor, pair_tok: torch.Tensor, out: torch.Tensor, max_tokens: int, tiled: bool,
                      pair_wt: torch.Tensor | None = None, out_row: torch.Tensor | None = None, accum: int = 0,
                      shard_start: int = 0, shard_n: int = 1 << 30, zero_out: bool = False, n_cols: int | None = None,
                      n_pairs: int | None = None) -> torch.Tensor:
    """grouped_gemm_codes on bf16 rows x (bf16_in_kernel(x, K, max_tokens) must hold; 8-k permuted rows with
    `permuted`): dsv41_fp4_grouped_gemm_bf16, whose workgroups split the rows into the two FP8 terms themselves."""
    dev = _lib.require_cuda(x, w, s, grp_expert, grp_start, pair_tok, out)
    E, N, Kh = w.shape
    K = Kh * 2
    if n_cols is not None:
        N = n_cols
    assert w.stride(2) == 1 and w.stride(1) == Kh and s.stride(2) == 1 and s.stride(1) == K // 32, "weights must be row-contiguous"
    assert x.shape[-1] == K and bf16_in_kernel(x, K, max_tokens)
    assert out.dtype == torch.float32 and out.stride(-1) == 1
    for t in (grp_expert, grp_start, pair_tok):
        assert t.dtype == torch.int32 and t.is_contiguous()
    G = grp_expert.numel()
    n_pairs = pair_tok.numel() if n_pairs is None else min(int(n_pairs), pair_tok.numel())
    assert grp_start.numel() >= G + 1 and (pair_wt is None or pair_wt.numel() >= n_pairs)
    assert out_row is not None or out.shape[0] >= n_pairs
    _lib.call("dsv41_fp4_grouped_gemm_bf16", _lib.ptr(w), w.stride(0), _lib.ptr(s), s.stride(0), 1 if tiled else 0, N, K,
              _lib.ptr(x), x.stride(0), x.shape[0], 1 if permuted else 0, _lib.ptr(grp_expert), _lib.ptr(grp_start), G,
              _lib.ptr(pair_tok), n_pairs, _lib.ptr(out), out.stride(0), out.shape[0], _lib.ptr(out_row), _lib.ptr(pair_wt), accum,
              max(1, int(max_tokens)), shard_start, min(shard_n, E), 1 if zero_out else 0, 0, 1 << 30, _lib.stream(dev))
    return out


T128_MAX = 128   # pairs per group the 128-pair tile kernel computes
LIGHT_GROUP = 64  # pairs per group of the light tile (two workgroups per CU, csrc/prefill.hip)
TILE_GROUP = 256  # pairs per group of the larger tiles (128-pair tiles, 256-pair tiles for larger groups)
LIGHT_PAIRS_PER_EXPERT = 48
LIGHT_PAIRS = 2048


def tile_group(n_pairs: int, n_experts: int | None) -> int:
    """Pairs per group for the tile kernels: LIGHT_GROUP while the pairs average at most LIGHT_PAIRS_PER_EXPERT per expert,
    else TILE_GROUP. With few pairs per expert the launch is bound by the weight stream, which the light tile runs faster;
    with more of them an expert's pairs fill several 64-pair groups that each stream its weights. w13 + w2, larger tiles /
    light tile in us, uniform and Zipf routing: 7168 x 1664, 384 experts, top-8 at 40 pairs per expert 1650 / 1525 and 1728 /
    1665, 60 1926 / 1802 and 1957 / 1976, 90 2408 / 2623 and 2427 / 2463; 5120 x 2304, 384 experts, top-6 at 40 1632 / 1489 and
    1678 / 1599, 60 1904 / 1745 and 1948 / 1940, 90 2293 / 2586; 4096 x 2048, 128 experts, top-8 at 48 440 / 364 and 470 / 423, 90
    567 / 625.
    n_experts None (not counted; the tables' bound of 512 says nothing): LIGHT_GROUP up to LIGHT_PAIRS pairs, where it is the
    faster one for 2 to 384 experts and every form of output (7168 x 1664 over 2 experts 183 / 153, 4096 x 2048 over 128 325 /
    270); 24,576 pairs added into a given output take 765 / 935 over 128 experts, 880 / 1047 over 2."""
    few = n_pairs <= (LIGHT_PAIRS if n_experts is None else LIGHT_PAIRS_PER_EXPERT * n_experts)
    return LIGHT_GROUP if few else TILE_GROUP


def t128_ok(N: int, K: int, max_tokens: int) -> bool:
    """Shapes for which groups of more than 16 pairs go to the 256-row x 128-pair tile kernel (the prefill w2 kernel as a
    general grouped GEMM: the weights of a group are read once for all its pairs) instead of the 16-pair passes."""
    return 16 < max_tokens <= T128_MAX and N % 256 == 0 and K % 128 == 0 and K >= 384


def grouped_gemm_t128(xc: torch.Tensor, xs: torch.Tensor, w: torch.Tensor, s: torch.Tensor, grp_expert: torch.Tensor,
                      grp_start: torch.Tensor, row_of_pair: torch.Tensor | None, y: torch.Tensor, n_pairs: int, tiled: bool,
                      n_cols: int | None = None, lo=None, max_tokens: int = T128_MAX) -> torch.Tensor:
    """y[p, :N] = codes(x)[row_of_pair[p]] . deq(W[e_g])^T for the pairs p of every group (<= 128 pairs each);
    dsv41_fp4_grouped_gemm_t128, or _t64 (the light tile, the same results) when the groups hold at most 64 pairs."""
    dev = _lib.require_cuda(xc, xs, w, s, grp_expert, grp_start, row_of_pair, y)
    E, N, Kh = w.shape
    N = n_cols if n_cols is not None else N
    K = Kh * 2
    assert w.stride(2) == 1 and w.stride(1) == Kh and s.stride(2) == 1 and s.stride(1) == K // 32
    assert y.dtype == torch.float32 and y.stride(-1) == 1 and y.shape[0] >= n_pairs
    _lib.call("dsv41_fp4_grouped_gemm_t64" if max_tokens <= LIGHT_GROUP else "dsv41_fp4_grouped_gemm_t128", _lib.ptr(xc), xc.stride(0), _lib.ptr(xs), xs.stride(0), xc.shape[0], *_lo_args(lo, xc, xs),
              _lib.ptr(row_of_pair),
              _lib.ptr(w), w.stride(0), _lib.ptr(s), s.stride(0), 1 if tiled else 0, E, N, K, _lib.ptr(grp_expert), _lib.ptr(grp_start),
              grp_expert.numel(), n_pairs, _lib.ptr(y), y.stride(0), _lib.stream(dev))
    return y


def grouped_gemm_scatter(xc: torch.Tensor, xs: torch.Tensor, w: torch.Tensor, s: torch.Tensor, grp_expert: torch.Tensor,
                         grp_start: torch.Tensor, row_of_pair: torch.Tensor | None, row_out: torch.Tensor, wt: torch.Tensor,
                         distinct: torch.Tensor | None, accum: bool, out: torch.Tensor, n_pairs: int, tiled: bool,
                         n_groups: int | None = None, y2: torch.Tensor | None = None, lo=None,
                         gmax: int = TILE_GROUP) -> torch.Tensor:
    """out[row_out[p]] += wt[p] * codes(x)[row_of_pair[p]] . deq(W[e_g])^T over the pairs p of the first n_groups
    groups (<= gmax <= 256 pairs each, LIGHT_GROUP taking the light tile; default every table entry); distinct: device int32
    scalar, non-zero when no two pairs share an output row (then stores when not accum, else read-add-write; otherwise fp32
    atomics); y2: fp32 [n_pairs, N] workspace (allocated when None; not written where the light tile stores the output rows
    itself); dsv41_fp4_grouped_gemm_scatter / _scatter_g64."""
    dev = _lib.require_cuda(xc, xs, w, s, grp_expert, grp_start, row_of_pair, row_out, wt, distinct, out, y2)
    E, N, Kh = w.shape
    K = Kh * 2
    assert w.stride(2) == 1 and w.stride(1) == Kh and s.stride(2) == 1 and s.stride(1) == K // 32
    assert out.dtype == torch.float32 and out.stride(-1) == 1 and out.shape[1] >= N
    assert row_out.dtype == torch.int32 and wt.dtype == torch.float32 and row_out.numel() >= n_pairs and wt.numel() >= n_pairs
    assert distinct is None or (distinct.dtype == torch.int32 and distinct.numel() == 1)
    G = grp_expert.numel() if n_groups is None else min(n_groups, grp_expert.numel())
    if y2 is None:
        y2 = torch.empty(max(n_pairs, 1), N, device=dev, dtype=torch.float32)
    assert y2.dtype == torch.float32 and y2.stride(-1) == 1 and y2.shape[0] >= n_pairs and y2.shape[1] >= N
    _lib.call("dsv41_fp4_grouped_gemm_scatter_g64" if gmax <= LIGHT_GROUP else "dsv41_fp4_grouped_gemm_scatter", _lib.ptr(xc), xc.stride(0), _lib.ptr(xs), xs.stride(0), xc.shape[0], *_lo_args(lo, xc, xs),
              _lib.ptr(row_of_pair),
              _lib.ptr(w), w.stride(0), _lib.ptr(s), s.stride(0), 1 if tiled else 0, E, N, K, _lib.ptr(grp_expert), _lib.ptr(grp_start),
              G, n_pairs, _lib.ptr(row_out), _lib.ptr(wt), _lib.ptr(distinct), 1 if accum else 0, _lib.ptr(out),
              out.stride(0), out.shape[0], _lib.ptr(y2), y2.stride(0), _lib.stream(dev))
    return out


def rows_distinct(row_out: torch.Tensor, n: int, n_placed: torch.Tensor | None, out_rows: int) -> torch.Tensor:
    """Device int32 [1]: 1 when no two of the first n_placed (device int32, or n) entries of row_out inside
    [0, out_rows) are equal; dsv41_rows_distinct."""
    dev = _lib.require_cuda(row_out, n_placed)
    assert row_out.dtype == torch.int32 and row_out.numel() >= n and (n_placed is None or n_placed.dtype == torch.int32)
    flag = torch.empty(1, dtype=torch.int32, device=dev)
    _lib.call("dsv41_rows_distinct", _lib.ptr(row_out), n, _lib.ptr(n_placed), out_rows, _lib.ptr(flag), _lib.stream(dev))
    return flag


_STARTS = {}


def _pair_starts(n: int, dev) -> torch.Tensor:
    """0..n (int32): the group table of one group per pair, a constant kept per (device, n) and only read by the
    kernels. Made outside any graph capture (a tensor made inside one lives in the graph's memory pool); inside a
    capture an uncached table is made for that call."""
    key = (dev.index if dev.index is not None else torch.cuda.current_device(), n)
    t = _STARTS.get(key)
    if t is None:
        t = torch.arange(n + 1, device=dev, dtype=torch.int32)
        if not torch.cuda.is_current_stream_capturing():
            _STARTS[key] = t
    return t


def fp4_gemv_pairs(x: torch.Tensor, w: torch.Tensor, s: torch.Tensor, row_in: torch.Tensor, expert: torch.Tensor,
                   wt: torch.Tensor, n_pairs: int, tiled: bool = False) -> torch.Tensor:
    """One output row per (row, expert, weight) pair, no atomics (cukern.py:60-77): for pair p, the fp32 N-vector
    wt[p] * x[row_in[p]] . dequant(W[expert[p]])^T, with x the bf16 activations (K per row), W the packed E2M1 bytes
    (E x N x K/2) and their E8M0 bytes (E x N x K/32), row_in / expert int32 and wt fp32 per pair. Weights row-major
    as the reference's kernel reads them, or in the tile_fp4 layout with `tiled`."""
    dev = _lib.require_cuda(x, w, s, row_in, expert, wt)
    assert x.dtype == torch.bfloat16 and x.stride(1) == 1
    E, N, Kh = w.shape
    out = torch.empty(n_pairs, N, device=dev, dtype=torch.float32)
    if n_pairs == 0:
        return out
    starts = _pair_starts(n_pairs, dev)
    ge, pt, pw = expert.to(torch.int32).contiguous(), row_in.to(torch.int32).contiguous(), wt.to(torch.float32).contiguous()
    if attached_codes(x, False) is None and bf16_in_kernel(x, Kh * 2, 1):
        return grouped_gemm_bf16(x, False, w, s, ge, starts, pt, out, 1, tiled, pair_wt=pw)
    xc, xs, lo = _quant_x(x, False, flag=not lo_in_lds(Kh * 2, 1))
    grouped_gemm_codes(xc, xs, w, s, ge, starts, pt, out, 1, tiled, pair_wt=pw, lo=lo)
    return out


def fp4_gemm_tc(xp: torch.Tensor, w: torch.Tensor, s: torch.Tensor, grp_expert: torch.Tensor, grp_start: torch.Tensor,
                pair_tok: torch.Tensor, n_pairs: int, max_tokens: int, shard_start: int = 0, shard_n: int = 1 << 30,
                zero_out: bool = False, out: torch.Tensor | None = None, out_col: int = 0) -> torch.Tensor:
    """Grouped expert GEMM (cukern.py:238-276): group g is expert grp_expert[g] over the pairs grp_start[g] up to
    grp_start[g+1] - 1, and pair p multiplies activation row pair_tok[p] of xp (bf16, K per row, in the 8-k order of
    permute_x) by that expert's dequantised packed weights; the result has one fp32 row of N per pair. Experts outside
    [shard_start, shard_start + shard_n) are left out (their rows zeroed with zero_out); `out` / `out_col` place the
    N columns inside a wider buffer. Groups of any size run (passes of 64 pairs)."""
    dev = _lib.require_cuda(xp, w, s)
    E, N, Kh = w.shape
    K = Kh * 2
    assert xp.dtype == torch.bfloat16 and xp.is_contiguous() and K % 128 == 0 and N % 16 == 0
    if out is None:
        out = torch.empty(n_pairs, N, device=dev, dtype=torch.float32)
    assert out.shape[1] >= out_col + N
    target = out[:, out_col:] if out_col else out
    ge, gs, pt = grp_expert.to(torch.int32).contiguous(), grp_start.to(torch.int32).contiguous(), pair_tok.to(torch.int32).contiguous()
    tile = t128_ok(N, K, max_tokens) and shard_start == 0 and shard_n >= E
    if not tile and attached_codes(xp, True) is None and bf16_in_kernel(xp, K, max_tokens):
        grouped_gemm_bf16(xp, True, w, s, ge, gs, pt, target, max_tokens, FP4_TILED, shard_start=shard_start, shard_n=shard_n,
                          zero_out=zero_out, n_cols=N, n_pairs=n_pairs)
        return out
    xc, xs, lo = _quant_x(xp, True, flag=tile or not lo_in_lds(K, max_tokens))
    if tile:
        # groups of up to 64 pairs (cukern.FP4_W_MAX): one weight read per group on the light or the 128-pair tile kernel
        grouped_gemm_t128(xc, xs, w, s, ge, gs, pt, target, n_pairs, FP4_TILED, n_cols=N, lo=lo, max_tokens=max_tokens)
        return out
    grouped_gemm_codes(xc, xs, w, s, ge, gs, pt, target, max_tokens, FP4_TILED, shard_start=shard_start,
                       shard_n=shard_n, zero_out=zero_out, n_cols=N, n_pairs=n_pairs, lo=lo)
    return out


def moe_dispatch(eid: torch.Tensor, wt: torch.Tensor, topk: int, n_experts: int, gmax: int, device: torch.device,
                 n_groups: torch.Tensor | None = None):
    """Buckets n (expert id, weight) pairs by expert in one launch (cukern.py:323-337). Returns, in expert order, each
    pair's token and weight, the inverse permutation, and the group tables (expert per group, -1 padded, and the
    n + 1 group starts); groups hold at most gmax pairs. Pairs of one expert stay in ascending pair order (the
    reference leaves that order open)."""
    n = eid.numel()
    assert n_experts <= 512
    eid = eid.reshape(-1).to(torch.int32).contiguous()
    wt = wt.reshape(-1).to(torch.float32).contiguous()
    _lib.require_cuda(eid, wt)
    tok_sorted = torch.empty(n, dtype=torch.int32, device=device)
    wt_sorted = torch.empty(n, dtype=torch.float32, device=device)
    inv = torch.empty(n, dtype=torch.int32, device=device)
    grp_expert = torch.empty(n, dtype=torch.int32, device=device)
    grp_start = torch.empty(n + 1, dtype=torch.int32, device=device)
    _lib.call("dsv41_moe_dispatch", _lib.ptr(eid), _lib.ptr(wt), n, topk, n_experts, gmax, _lib.ptr(tok_sorted), _lib.ptr(wt_sorted),
              _lib.ptr(inv), _lib.ptr(grp_expert), _lib.ptr(grp_start), _lib.ptr(n_groups), _lib.stream(device))
    return tok_sorted, wt_sorted, inv, grp_expert, grp_start


# --------------------------------------------------------------------------- FP8-weight GEMM (M <= 64 rows per pass)
FP8_ROWS = 64  # output rows one launch handles; the weights are read once for all of them

def _fp8_launch(x: torch.Tensor, w8: torch.Tensor, s8: torch.Tensor, Mo: int, N: int, K: int, group_cols: int, tiled: bool,
                out: torch.Tensor | None, outb: torch.Tensor | None) -> None:
    # the kernels read scale row n // 32 for every weight row n < N and byte k // 32 for every k < K
    if s8.dim() != 2 or s8.shape[0] < (N + 31) // 32 or s8.shape[1] < K // 32 or s8.stride(1) != 1:
        raise ValueError(f"fp8 scales: need [>= {(N + 31) // 32}, >= {K // 32}] bytes with unit column stride, got {tuple(s8.shape)}")
    if w8.shape[0] < N or (w8.numel() < N * K):
        raise ValueError(f"fp8 weights: need {N} x {K} bytes, got {tuple(w8.shape)}")
    _lib.call("dsv41_fp8_gemm", _lib.ptr(w8), w8.stride(0), 1 if tiled else 0, _lib.ptr(s8), s8.stride(0), N, K,
              _lib.ptr(x), x.stride(0), Mo, group_cols, _lib.ptr(out), out.stride(0) if out is not None else 0,
              _lib.ptr(outb), outb.stride(0) if outb is not None else 0, _lib.stream(x.device))


def fp8_gemm_tc(x: torch.Tensor, w8: torch.Tensor, s8: torch.Tensor, group_cols: int = 0, out_dtype=torch.bfloat16,
                tiled: bool = False) -> torch.Tensor:
    """Dense FP8 weights times bf16 rows (cukern.py:114-173): x (M contiguous rows of K) against the E4M3 bytes w8
    (N x K, in w8.permute_k's order, and w8.tile's with `tiled`) with one E8M0 byte per 32 x 32 block (s8); the M x N
    result is accumulated in fp32 and rounded to out_dtype. group_cols > 0: block-diagonal use (x [B * N/group_cols, K]; output
    row b, column n uses x row b * (N/group_cols) + n // group_cols) -> [B, N]. More than 64 output rows run in
    passes of 64 (the reference also chunks, cukern.py:129-132)."""
    dev = _lib.require_cuda(x, w8, s8)
    M, K = x.shape
    N = w8.shape[0]
    assert x.dtype == torch.bfloat16 and x.is_contiguous() and w8.is_contiguous() and s8.is_contiguous()
    assert w8.dtype == torch.uint8 and s8.dtype == torch.uint8
    assert K % 64 == 0 and N % 8 == 0 and (group_cols == 0 or group_cols % 16 == 0 and N % group_cols == 0)
    G = N // group_cols if group_cols else 1
    Mo = M // G
    assert Mo * G == M
    if Mo > FP8_ROWS:
        return torch.cat([fp8_gemm_tc(x[i * G:(i + FP8_ROWS) * G], w8, s8, group_cols, out_dtype, tiled)
                          for i in range(0, Mo, FP8_ROWS)], dim=0)
    if out_dtype == torch.bfloat16:
        y = torch.empty(Mo, N, device=dev, dtype=torch.bfloat16)
        _fp8_launch(x, w8, s8, Mo, N, K, group_cols, tiled, None, y)
        return y
    y = torch.empty(Mo, N, device=dev, dtype=torch.float32)
    _fp8_launch(x, w8, s8, Mo, N, K, group_cols, tiled, y, None)
    return y if out_dtype == torch.float32 else y.to(out_dtype)


def fp8_rows_plan(M: int, N: int, K: int):
    """(activation rows per tile, K ranges) with which dsv41_fp8_gemm_rows multiplies M > 64 rows, or None where dequantising
    the weights and the library GEMM are faster. A tile's time is its chain over K, the library's the product's size.
    us below: medians of graph replays over weights larger than the last-level cache.
      * Small weights have too few tiles for their chains, unless K is short or falls into several ranges. dequantised + library /
        tiles: 856 x 1280 at 65 rows 11.0 / 14.2, 856 x 2560 at 160 15.5 / 18.1, 2048 x 1280 at 160 13.3 / 14.8, 512 x 1984 at 333
        17.4 / 18.8, 656 x 1216 at 640 14.7 / 15.3; on the other side of the lines 3000 x 1280 at 65 14.6 / 14.4, 2048 x 1280 at 333
        16.3 / 15.1, 1280 x 1280 at 420 17.1 / 15.3, 4096 x 768 at 65 14.1 / 11.9, 512 x 5120 at 160 18.1 / 17.2.
      * Tiles of 64 rows while they are at most 256, K in ranges of at least 1024 k. The weight tiles are dealt out to 8 XCDs of 32
        CUs, and the ranges are as many as leave one tile to a CU on the XCD with the most of them: 1280 x 5120 (10 weight
        tiles, two on two XCDs) at 256 rows in 5 / 4 ranges 25.6 / 20.3, 1280 x 2560 at 640 in 2 / 1 26.9 / 22.8, 2176 x 4096 at
        160 in 4 / 3 23.9 / 20.5, 3328 x 7168 at 160 in 3 / 2 35.8 / 32.7. From K = 6144 on two ranges pay also where they put
        two tiles on a CU: 5120 x 8192 at 256 in 1 / 2 56.9 / 52.1, 3000 x 7168 at 333 49.2 / 46.7 (6952 x 7232 at 160 52.5 / 55.8,
        so up to 40 weight tiles).
      * Tiles of 128 up to 512 rows while at most three go to a CU (dequantised + library / tiles: 32768 x 1280 at 333 55 / 52, 420 59 /
        66; 16384 x 5120 at 512 117 / 91), and beyond them up to 1024 rows while one per CU covers the product. Beyond 512 rows with
        long weight rows they have to fill two thirds of the CUs (5120 x 8192 at 700 89 / 78, 900 101 / 116; 1280 x 5120 at 768
        34 / 38), and 64-row tiles may not share one (2176 x 7168 at 768 50.2 / 65.1).
    The line is not the best one everywhere: 4608 x 5120 at 420 / 640 rows 52.3 / 53.2 and 55.0 / 58.6, 2992 x 5376 at 900 51.1 /
    60.1, 8672 x 2112 at 512 40.4 / 47.4; three ranges of 128-row tiles, which it does not use, take 65 for 5120 x 8192 at 420
    against 76 in one."""
    if K % 64 or N % 8 or M > 1024:
        return None
    if 1088 < K <= 3072 and N * K < (2_700_000 if M <= 192 else 1_570_000 if M <= 384 else 1_050_000):
        return None
    tn = (N + 127) // 128
    t64, t128 = (M + 63) // 64, (M + 127) // 128
    if tn * t64 <= 256:
        xcd = (tn + 7) // 8 * t64   # tiles of the XCD with the most of them
        fit = 2 if 16 < xcd <= 32 and K >= 6144 and tn <= 40 else 32 // xcd
        tile, splits = 64, max(1, min(fit, K // 1024, 8))
        filled = tn * t64 >= 176 and xcd <= 32
    elif (M <= 512 and tn * t128 <= 768) or tn * t128 <= 256:
        tile, splits, filled = 128, 1, tn * t128 >= 176
    else:
        return None
    if M > 512 and K > 4096 and not filled:
        return None
    # a range's scale bytes fit the kernel's 512
    return (tile, splits) if 2 * (-(-(K // 64) // splits)) <= 512 else None


def fp8_gemm_rows(x: torch.Tensor, w8: torch.Tensor, s8: torch.Tensor, tiled: bool, plan) -> torch.Tensor:
    """bf16 [M, N] = x . deq(w8)^T for M rows of contiguous bf16 x with plan = fp8_rows_plan(M, N, K); the values of
    fp8_gemm_tc up to the order of the fp32 sums. dsv41_fp8_gemm_rows."""
    dev = _lib.require_cuda(x, w8, s8)
    M, K = x.shape
    N = w8.shape[0]
    tile, splits = plan
    assert x.dtype == torch.bfloat16 and x.is_contiguous() and w8.is_contiguous() and w8.dtype == torch.uint8 and s8.dtype == torch.uint8
    assert x.data_ptr() % 16 == 0 and w8.data_ptr() % 16 == 0
    if s8.dim() != 2 or s8.shape[0] < (N + 31) // 32 or s8.shape[1] < K // 32 or s8.stride(1) != 1 or w8.shape[1] != K:
        raise ValueError(f"fp8 operands: {tuple(w8.shape)} weights with {tuple(s8.shape)} scales for K = {K}")
    y = torch.empty(M, N, device=dev, dtype=torch.bfloat16)
    part = torch.empty(splits * M * N, device=dev, dtype=torch.float32) if splits > 1 else None
    _lib.call("dsv41_fp8_gemm_rows", _lib.ptr(w8), K, 1 if tiled else 0, _lib.ptr(s8), s8.stride(0), N, K, _lib.ptr(x), K, M, None, 0,
              _lib.ptr(y), N, tile, splits, _lib.ptr(part), splits * M * N if splits > 1 else 0, _lib.stream(dev))
    return y


def fp8_gemv(x: torch.Tensor, w_fp8: torch.Tensor, s_u8: torch.Tensor) -> torch.Tensor:
    """x: bf16 [M, K]; w_fp8: float8_e4m3fn / uint8 [N, K] row-major (any N); s_u8: uint8 [ceil(N/32), K/32] (E8M0).
    fp32 [M, N] (cukern.py:78-93; the reference takes M == 1, this takes M <= 64). K % 32 == 0: a K that is not a
    multiple of 64 is padded with 32 zero columns (weights and activations) for the 64-k chunks of the kernel."""
    dev = _lib.require_cuda(x, w_fp8, s_u8)
    M, K = x.shape
    N = w_fp8.shape[0]
    assert x.stride(1) == 1 and K % 32 == 0 and 1 <= M <= FP8_ROWS
    w = w_fp8.view(torch.uint8)
    s = s_u8.view(torch.uint8)
    assert w.stride(1) == 1 and s.stride(1) == 1 and s.shape[0] * 32 >= N and s.shape[1] * 32 >= K
    if K % 64:
        w = torch.nn.functional.pad(w, (0, 32))
        x = torch.nn.functional.pad(x, (0, 32))
        s = torch.nn.functional.pad(s, (0, 1), value=127)
        K += 32
    out = torch.empty(M, N, device=dev, dtype=torch.float32)
    _fp8_launch(x.to(torch.bfloat16), w, s, M, N, K, 0, False, out, None)
    return out
