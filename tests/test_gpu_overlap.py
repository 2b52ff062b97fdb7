"""The selected solve with the block inversions beside the lesser and greater products
(the default) and without, against the dense oracle at 1e-10 per block, the bound of the
other parity tests: one block, two, unequal neighbours (V of block i and Q of block j share a launch),
boundary blocks at both ends, the current, eager and captured.  The products of
either order are the same ones, so the results agree to the last bit."""

import numpy as np
import pytest

from quatrex_amd import _lib
from quatrex_amd import solve as S
from tests.helpers import edge_case
from tests.test_gpu_products import _check, _dense

pytestmark = pytest.mark.gpu


def _device_case(bs, E, device):
    import torch

    g, A, SL, SG, obc = edge_case(bs, seed=sum(bs) + E, E=E)
    t = lambda x: torch.as_tensor(np.ascontiguousarray(x), device=device)  # noqa: E731
    ob = [[None if x is None else t(x) for x in row] for row in obc]
    return g, (A, SL, SG, obc), [tuple(map(t, m)) for m in (A, SL, SG)], ob


@pytest.mark.parametrize("bs,E", [((33,), 2), ((40, 65), 3), ((65, 33, 96, 34), 5), ((128, 97, 130), 40), ((300, 64, 257), 2)])
def test_overlap_on_and_off_agree(device, bs, E):
    import torch

    print(f"overlap bs={bs} E={E}", flush=True)
    g, host, (A, SL, SG), ob = _device_case(bs, E, device)
    ctx = S.default_context(device)
    got = {}
    for on in (0, 1):
        out = [S.packed_empty(g, E, device) for _ in range(3)]
        cur = torch.empty((E, len(bs) + 1), dtype=torch.complex128, device=device) if len(bs) > 1 else None
        ctx.set_option(_lib.RGF_OPT_OVERLAP, on)
        try:
            S.selected_solve(g, A, SL, SG, g_lesser=out[1], g_greater=out[2], g_retarded=out[0], obc=ob, current=cur)
            ctx.status()
        finally:
            ctx.set_option(_lib.RGF_OPT_OVERLAP, 1)
        got[on] = [tuple(x.cpu().numpy() for x in o) for o in out]
        if cur is not None:
            got[on].append((cur.cpu().numpy(),))
    _check(g, got[1][:3], _dense(g, *host))
    for x, y in zip(got[0], got[1]):
        for p, q in zip(x, y):
            np.testing.assert_array_equal(p, q)


def test_captured_overlap_replays_the_eager_result(device):
    import torch

    bs, E = (65, 40, 96), 6
    g, _, (A, SL, SG), ob = _device_case(bs, E, device)
    eager = [S.packed_empty(g, E, device) for _ in range(3)]
    S.selected_solve(g, A, SL, SG, g_lesser=eager[1], g_greater=eager[2], g_retarded=eager[0], obc=ob)
    out = [S.packed_empty(g, E, device) for _ in range(3)]
    graph = S.SolveGraph(g, A, SL, SG, g_lesser=out[1], g_greater=out[2], g_retarded=out[0], obc=ob)
    for _ in range(4):
        for o in out:
            for p in o:
                p.zero_()
        torch.cuda.synchronize()
        graph.launch()
        torch.cuda.synchronize()
        for o, e in zip(out, eager):
            for p, q in zip(o, e):
                assert torch.equal(p, q)
        eager[0][0].abs().sum().item()  # eager work between the replays
    graph.close()


def _launches(g, mats, ob, E, ctx, on, device):
    """Product launches of one solve: the order with overlap has one more per step."""
    A, SL, SG = mats
    out = [S.packed_empty(g, E, device) for _ in range(3)]
    ctx.set_option(_lib.RGF_OPT_OVERLAP, on)
    ctx.profile(True)
    try:
        ctx.profile_read()
        S.selected_solve(g, A, SL, SG, g_lesser=out[1], g_greater=out[2], g_retarded=out[0], obc=ob)
        ctx.status()
        return ctx.profile_read()["gemm_launches"], out
    finally:
        ctx.profile(False)
        ctx.set_option(_lib.RGF_OPT_OVERLAP, 1)


@pytest.mark.parametrize("bs,E,two_streams", [
    ((40, 40, 200), 8, False),           # one wide block: most steps are small
    ((33, 33, 33, 256), 8, False),
    ((48, 48, 48), 78, False), ((48, 48, 48), 79, True),  # 179712 and 182016 elements
    ((65, 33, 96, 34), 70, True), ((40, 65), 80, True), ((512, 512), 1, True),
])
def test_second_stream_only_for_products_that_fill_the_chip(device, bs, E, two_streams):
    import torch

    print(f"overlap rule bs={bs} E={E}", flush=True)
    n = len(bs)
    assert (E * sum(a * b for a, b in zip(bs, bs[1:])) / (n - 1) >= 1.8e5) == two_streams
    g, A, SL, SG, obc = edge_case(bs, seed=sum(bs), E=min(E, 4))
    t = lambda x: torch.as_tensor(np.ascontiguousarray(np.resize(x, (E, *x.shape[1:]))), device=device)  # noqa: E731
    mats = [tuple(map(t, m)) for m in (A, SL, SG)]
    ob = [[None if x is None else t(x) for x in row] for row in obc]
    ctx = S.default_context(device)
    plain, ref = _launches(g, mats, ob, E, ctx, 0, device)
    got, out = _launches(g, mats, ob, E, ctx, 1, device)
    assert got - plain == (n - 1 if two_streams else 0)
    for o, r in zip(out, ref):
        for p, q in zip(o, r):
            assert torch.equal(p, q)


def test_captured_two_stream_sweep_with_current(device):
    """Large enough that the eager solve runs on two streams too."""
    import torch

    bs, E = (65, 40, 96), 60
    assert E * (65 * 40 + 40 * 96) / 2 >= 1.8e5
    g, _, (A, SL, SG), ob = _device_case(bs, E, device)
    ref = [S.packed_empty(g, E, device) for _ in range(3)]
    out = [S.packed_empty(g, E, device) for _ in range(3)]
    cur = [torch.empty((E, len(bs) + 1), dtype=torch.complex128, device=device) for _ in range(2)]
    ctx = S.default_context(device)
    ctx.set_option(_lib.RGF_OPT_OVERLAP, 0)
    try:
        S.selected_solve(g, A, SL, SG, g_lesser=ref[1], g_greater=ref[2], g_retarded=ref[0], obc=ob, current=cur[0])
    finally:
        ctx.set_option(_lib.RGF_OPT_OVERLAP, 1)
    graph = S.SolveGraph(g, A, SL, SG, g_lesser=out[1], g_greater=out[2], g_retarded=out[0], obc=ob, current=cur[1])
    flat = lambda o, c: [p for x in o for p in x] + [c]  # noqa: E731
    for k in range(4):
        for p in flat(out, cur[1]):
            p.zero_()
        torch.cuda.synchronize()
        graph.launch()
        if k == 2:  # the same sweep, eager, right behind the replay
            S.selected_solve(g, A, SL, SG, g_lesser=out[1], g_greater=out[2], g_retarded=out[0], obc=ob, current=cur[1])
        torch.cuda.synchronize()
        for p, q in zip(flat(out, cur[1]), flat(ref, cur[0])):
            assert torch.equal(p, q)
        ref[0][0].abs().sum().item()  # eager work between the replays
    graph.close()
