"""The launches around the experts: the fp32 router with the quantiser's workgroups beside it, the FP8 operand that a prefill
layer quantises once, and the dispatch over several chunks of pairs, against the separate launches and the oracle."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("M,H,E", [(1, 1024, 384), (3, 5120, 40), (16, 7168, 384), (7, 2048, 16)])
def test_router_f32w_with_quantised_rows(M, H, E):
    """part equals the router's own launch and xq the quantiser's, bit for bit, also with zero groups, infinities and NaN."""
    from dsv41_amd import _lib, moe, quant
    print(f"router M={M} H={H} E={E}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M + E)
    x = (torch.randn(M, H, generator=g, device=DEV) * torch.logspace(-4, 3, H, device=DEV)).to(torch.bfloat16)
    x[0, :32] = 0
    G = torch.randn(E, H, generator=g, device=DEV)
    xq = torch.full((M, H), -1.0, dtype=torch.bfloat16, device=DEV)
    part = moe.router_logits_f32w(x, G, xq=xq)
    assert torch.equal(part, moe.router_logits_f32w(x, G)) and torch.equal(xq, quant.fake_quant_fp8(x))
    x[M - 1, 64:67] = torch.tensor([float("inf"), float("nan"), -float("inf")], device=DEV, dtype=torch.bfloat16)
    moe.router_logits_f32w(x, G, xq=xq)
    assert torch.equal(xq.view(torch.int16), quant.fake_quant_fp8(x).view(torch.int16))
    L = _lib.lib()
    args = lambda q, ld: (_lib.ptr(x), H, _lib.ptr(G), H, E, H, M, _lib.ptr(part), q, ld, _lib.stream(DEV))
    assert L.dsv41_router_logits_f32w_quant(*args(_lib.ptr(x), H)) == -1 and L.dsv41_router_logits_f32w_quant(*args(None, H)) == -1
    assert L.dsv41_router_logits_f32w_quant(*args(_lib.ptr(xq), H - 8)) == -1


def test_prefill_operand_quantised_once():
    """fake_quant_codes' operand gives what prefill_up quantises from its values, and prefill_up reads the values it is given: a
    record left on a tensor whose bytes changed without a new version (library entry points write their `out` so) plays no part."""
    from dsv41_amd import moe, quant
    g = torch.Generator(device=DEV).manual_seed(5)
    E, H, I, k, T = 8, 512, 384, 2, 40
    b = lambda *s: torch.randint(0, 256, s, generator=g, dtype=torch.uint8, device=DEV)
    sc = lambda *s: torch.randint(119, 124, s, generator=g, dtype=torch.uint8, device=DEV)
    ex = moe.ExpertWeights(b(E, 2 * I, H // 2), sc(E, 2 * I, H // 32), b(E, H, I // 2), sc(E, H, I // 32), True)
    x = torch.randn(T, H, generator=g, device=DEV).to(torch.bfloat16)
    eid = torch.randint(0, E, (T, k), generator=g, device=DEV, dtype=torch.int32)
    wt = torch.rand(T, k, generator=g, device=DEV)
    xq, xc, xs = quant.fake_quant_codes(x)
    assert torch.equal(xq, quant.fake_quant_fp8(x))
    y = moe.prefill_experts(xq, eid, wt, ex, 10.0)
    assert torch.equal(y, moe.prefill_down(moe._prefill_up_codes(xc, xs, eid, wt, ex, 10.0), ex))
    quant.attach_codes(xq, xc, xs)
    xq.data.zero_()
    assert quant.attached_codes(xq, False) is not None and not moe.prefill_experts(xq, eid, wt, ex, 10.0).any()


@pytest.mark.parametrize("n,E,gmax", [(5000, 512, 64), (4096, 3, 256), (4097, 512, 1), (1025, 1, 7), (20000, 384, 256)])
def test_dispatch_over_several_chunks(n, E, gmax):
    from dsv41_amd import hipkern
    rng = np.random.default_rng(n)
    eid = np.minimum(rng.zipf(1.3, n) - 1, E + 1).astype(np.int32)     # popular experts, some ids out of range
    eid[rng.integers(0, n, 20)] = -1
    wt = rng.random(n).astype(np.float32)
    ref = O.moe_dispatch(eid, wt, 4, E, gmax)
    got = hipkern.moe_dispatch(torch.from_numpy(eid).to(DEV), torch.from_numpy(wt).to(DEV), 4, E, gmax, DEV)
    for a, r in zip(got, ref):
        assert np.array_equal(a.cpu().numpy(), r)
