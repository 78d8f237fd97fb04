"""The rules on sizes that choose a kernel, where they are Python."""


def test_tile_group_counts_experts():
    """64-pair groups while the pairs average at most 48 per expert. Without a count (GroupedPairs takes n_experts as an option) the
    tables' bound of 512 must not stand in for it: 24,576 pairs over 8 experts would stream each expert's weights 48 times."""
    from dsv41_amd.hipkern import LIGHT_GROUP, LIGHT_PAIRS, LIGHT_PAIRS_PER_EXPERT as most, TILE_GROUP, tile_group
    for E in (1, 8, 128, 384, 512):
        assert tile_group(most * E, E) == LIGHT_GROUP and tile_group(most * E + 1, E) == TILE_GROUP
    assert tile_group(LIGHT_PAIRS, None) == LIGHT_GROUP
    assert tile_group(LIGHT_PAIRS + 1, None) == tile_group(most * 512, None) == TILE_GROUP


def test_linear_w_sees_what_watches_a_call():
    """w8._watched: what follows torch operations keeps w8.linear_w on F.linear; a default device does not."""
    import torch
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    from dsv41_amd.w8 import _watched

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    x = torch.ones(2, 4)
    seen = []
    note = lambda v: (seen.append(_watched(v)), v + 1)[1]
    assert not _watched(x)
    with torch.device("cpu"):
        assert not _watched(x)
        with Function():
            assert _watched(x)
    with Dispatch():
        assert _watched(x)
    torch.func.vmap(note)(x)
    torch.func.jvp(note, (x,), (x,))
    torch.jit.trace(note, x, check_trace=False)
    torch.fx.experimental.proxy_tensor.make_fx(note)(x)
    assert len(seen) == 4 and all(seen)
    assert _watched(torch.nn.Parameter(x)) and _watched(x.clone().requires_grad_(True))
    with torch.no_grad():
        assert not _watched(x.clone().requires_grad_(True))


def test_fp8_rows_plan():
    """The tiles of w8.linear_w past 64 rows: not for small weights with an unsplit chain over K, and as many K ranges as leave
    one 64-row tile to a CU of the XCD (of 8, with 32 CUs) that has the most weight tiles; two where K is long."""
    from dsv41_amd.hipkern import fp8_rows_plan
    for M, N, K in ((65, 856, 1280), (160, 856, 2560), (333, 512, 1984), (640, 656, 1216), (160, 2048, 1280)):
        assert fp8_rows_plan(M, N, K) is None
    for (M, N, K), plan in {(640, 1280, 2560): (64, 1), (256, 1280, 5120): (64, 4), (160, 3328, 7168): (64, 2), (160, 2176, 4096): (64, 3),
                            (256, 5120, 8192): (64, 2), (65, 4096, 768): (64, 1), (160, 512, 5120): (64, 5)}.items():
        assert fp8_rows_plan(M, N, K) == plan
    for M in (65, 100, 192, 193, 320, 500, 640, 1000):
        for N in range(256, 9000, 424):
            for K in range(512, 16384, 704):
                plan = fp8_rows_plan(M, N, K)
                if plan is None or plan[0] == 128:
                    continue
                tn, nk = (N + 127) // 128, K // 64
                load = (tn + 7) // 8 * ((M + 63) // 64) * plan[1]
                assert 1 <= plan[1] <= 8 and 2 * -(-nk // plan[1]) <= 512
                assert plan[1] == 1 or load <= 32 or (plan[1] == 2 and K >= 6144 and load <= 64)
