"""Host-pointer calls on both sides of the pinned staging's limits (128 KB in,
64 KB out), against the device-pointer call on the same weights, bit for bit:
odd sizes, row ranges that start inside a 16-byte piece, and the untouched
rows around them."""
import numpy as np
import pytest
import torch

import zero_amd
from zero_amd import synth

pytestmark = pytest.mark.gpu

Q4_0 = 2


# out of 64 KB is 16,384 rows, in of 128 KB is in_dim 32,768
@pytest.mark.parametrize("rows,k", [(1, 32), (5, 544), (16384, 64), (16385, 64), (3, 32768), (3, 32800)])
def test_host_call_equals_device_call(ctx, rows, k):
    rng = np.random.default_rng(rows + k)
    w, x = synth.weight(rng, Q4_0, rows, k, 1), synth.activations(rng, k)
    y = torch.empty(rows, dtype=torch.float32, device="cuda")
    ctx.linear_dev(torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda(), y, k, rows, Q4_0, 1)
    torch.cuda.synchronize()
    want = y.cpu().numpy().view(np.uint32)
    ctx.register(w, Q4_0, 1)
    try:
        for _ in range(2):
            out = np.empty(rows, np.float32)
            ctx.linear_dispatch(x, w, out, k, rows, Q4_0)
            assert np.array_equal(out.view(np.uint32), want)
        # starts at every offset in a 16-byte piece, and ends around the staging's
        # limit of 16,384 rows counted from the piece that holds the start
        ends = {(min(1, rows - 1), min(e, rows)) for e in (16381, 16382, 16383, 16384)}
        for s, e in ends | {(0, 1), (rows - 1, rows), (min(2, rows - 1), rows), (min(3, rows - 1), rows), (rows // 2, rows // 2)}:
            out = np.full(rows, -7.0, np.float32)
            ctx.linear_range(x, w, out, k, rows, Q4_0, s, e)
            assert np.array_equal(out[s:e].view(np.uint32), want[s:e]) and np.all(out[:s] == -7.0) and np.all(out[e:] == -7.0)
    finally:
        ctx.clear()


def test_host_fused_call_with_odd_segments(ctx):
    rng = np.random.default_rng(4)
    k, ns = 544, (7, 1, 18)
    ws, x = [synth.weight(rng, Q4_0, n, k, 1) for n in ns], synth.activations(rng, k)
    for w in ws:
        ctx.register(w, Q4_0, 1)
    try:
        one = [np.empty(n, np.float32) for n in ns]
        for w, o, n in zip(ws, one, ns):
            ctx.linear_dispatch(x, w, o, k, n, Q4_0)
        outs = [np.empty(n, np.float32) for n in ns]
        ctx.linear_fused_dispatch(x, [(w, o, Q4_0) for w, o in zip(ws, outs)], k)
        assert all(np.array_equal(a.view(np.uint32), b.view(np.uint32)) for a, b in zip(one, outs))
    finally:
        ctx.clear()


def test_staging_begins_with_the_second_host_call(ctx):
    """A fresh context: device calls, then host calls on changing activations,
    with outputs that fit the staging and one that does not; each gives the
    device call's bits, so nothing of an earlier call's bytes is read again."""
    rng = np.random.default_rng(11)
    k = 64
    own = zero_amd.Context(0)
    try:
        for rows in (8, 16388, 12):
            w = synth.weight(rng, Q4_0, rows, k, 1)
            wd = torch.from_numpy(w).cuda()
            own.register(w, Q4_0, 1)
            for _ in range(4):
                x = synth.activations(rng, k)
                y = torch.empty(rows, dtype=torch.float32, device="cuda")
                own.linear_dev(torch.from_numpy(x).cuda(), wd, y, k, rows, Q4_0, 1)
                out = np.empty(rows, np.float32)
                own.linear_dispatch(x, w, out, k, rows, Q4_0)
                assert np.array_equal(out.view(np.uint32), y.cpu().numpy().view(np.uint32))
    finally:
        own.close()
