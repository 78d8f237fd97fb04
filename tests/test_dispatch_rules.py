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
