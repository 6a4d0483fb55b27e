"""The wide GEMV (zg_gemv_wide.hip): Q4_0 / Q8_0 shapes outside the strip
kernel's range, against the oracle's row kernels and float64.

Edges of its tiles: in_dims of one block, one chunk of 16 blocks and one
block more, one, two and three chunks per wave, and a partial last round;
row counts around the groups of four and the one- and two-group batches;
row ranges that start inside a group.
"""
import numpy as np
import pytest
import torch

from zero_amd import synth

pytestmark = pytest.mark.gpu

Q4_0, Q8_0 = 2, 8

# (interleave, rows, k): k / 32 blocks in chunks of 16; four waves up to
# in_dim 2048, eight above it
SHAPES = [
    (1, 1, 32), (1, 5, 480), (1, 7, 544), (4, 8, 96), (4, 4, 2016), (1, 6, 2080), (1, 4097, 2048), (1, 2049, 4128),
    (4, 2044, 4160), (4, 2052, 8256), (1, 33, 8224), (1, 513, 11008), (4, 4096, 11008), (1, 9, 12320), (1, 3, 20512),
]


@pytest.mark.parametrize("quant", [Q4_0, Q8_0])
@pytest.mark.parametrize("il,rows,k", SHAPES)
def test_wide_gemv_parity_and_ranges(ctx, zo, quant, il, rows, k):
    rng = np.random.default_rng(rows + 7 * k + quant)
    w = synth.weight(rng, quant, rows, k, il)
    x = synth.activations(rng, k)
    ctx.register(w, quant, il)
    try:
        out = np.empty(rows, np.float32)
        ctx.linear_dispatch(x, w, out, k, rows, quant)
        ref = zo.linear_range(x, w, k, rows, quant, il)
        f64 = zo.linear_f64(x, w, k, rows, quant, il)
        top = np.max(np.abs(f64))
        # fp32 sums of k products in two orders: both within the oracle's own
        # distance to float64, with room for the smaller of the two
        assert np.max(np.abs(out - f64)) / top <= 4 * np.max(np.abs(ref - f64)) / top + 1e-6
        # a row's bits do not depend on the range it is computed in
        for s, e in {(0, rows), (rows // 3, rows), (1 if rows > 1 else 0, max(1, rows - 1)), (rows - 1, rows)}:
            part = np.full(rows, -7.0, np.float32)
            ctx.linear_range(x, w, part, k, rows, quant, s, e)
            assert np.array_equal(part[s:e].view(np.uint32), out[s:e].view(np.uint32)), (s, e)
            assert np.all(part[:s] == -7.0) and np.all(part[e:] == -7.0), (s, e)
    finally:
        ctx.clear()


@pytest.mark.parametrize("quant,rows,k", [(Q4_0, 10001, 1056), (Q8_0, 4097, 2048)])
def test_wide_gemv_argmax(ctx, quant, rows, k):
    """The argmax form: the row of the largest output, ties to the first."""
    rng = np.random.default_rng(rows + k)
    w = synth.weight(rng, quant, rows, k, 1)
    x = synth.activations(rng, k)
    wd, xd = torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda()
    y = torch.empty(rows, dtype=torch.float32, device="cuda")
    best = torch.empty(1, dtype=torch.int64, device="cuda")
    for _ in range(2):
        ctx.lm_head_dev(xd, wd, y, k, rows, quant, 1, best)
        torch.cuda.synchronize()
        ok, idx, v = ctx.argmax_unpack(int(best.item()) & ((1 << 64) - 1))
        got = y.cpu().numpy()
        assert ok and idx == int(np.argmax(got)) and v == got[idx]
        # the winner's bytes again at the end of the tensor: the first wins
        rb = w.size // rows
        wd[(rows - 1) * rb:] = wd[idx * rb:(idx + 1) * rb].clone()


def rows_of(quant, q, d_bits):
    """Plain block bytes of the integer quants q [rows][k], one fp16 scale."""
    rows, k = q.shape
    b = q.reshape(rows, k // 32, 32)
    if quant == Q4_0:
        u = (b + 8).astype(np.uint8)
        body = u[..., :16] | (u[..., 16:] << 4)
    else:
        body = b.astype(np.int8).view(np.uint8)
    w = np.empty((rows, k // 32, 2 + body.shape[-1]), np.uint8)
    w[..., :2] = np.frombuffer(np.uint16(d_bits).tobytes(), np.uint8)
    w[..., 2:] = body
    return w.reshape(-1)


def wide(ctx, x, w, rows, k, quant, il):
    if il == 4:
        w = synth.interleave_x4(w, rows, k, quant)
    y = torch.empty(rows, dtype=torch.float32, device="cuda")
    ctx.linear_dev(torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda(), y, k, rows, quant, il)
    return y.cpu().numpy()


# plain rows, and X4 groups of in_dims that the segment kernel does not take
FORMS = [(1, 9, 480), (1, 33, 11008), (4, 8, 96), (4, 12, 14400)]


@pytest.mark.parametrize("quant", [Q4_0, Q8_0])
@pytest.mark.parametrize("il,rows,k", FORMS)
def test_wide_gemv_sums_the_products_alone(ctx, quant, il, rows, k):
    """Activations with a large common part and quants of +1, -1 in turn:
    every partial sum of the products x (d q) is an integer below 2^24 and the
    result exact, while a sum of x with offset quants (8 or 128 times the
    common part) would round."""
    rng = np.random.default_rng(k + quant)
    x = (2.0 ** 20 + rng.integers(0, 64, k)).astype(np.float32)
    q = np.empty((rows, k), np.int64)
    q[:, 0::2] = rng.choice([-1, 1], size=(rows, 1))
    q[:, 1::2] = -q[:, :1]
    want = (q @ x.astype(np.float64)).astype(np.float32)
    got = wide(ctx, x, rows_of(quant, q, 0x3C00), rows, k, quant, il)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("quant", [Q4_0, Q8_0])
@pytest.mark.parametrize("il,rows,k", FORMS)
def test_wide_gemv_infinite_and_huge_activations(ctx, quant, il, rows, k):
    """An infinite activation gives +-Inf by its quant's sign, NaN where the
    quant is 0; activations of 1e37 stay finite while their products do."""
    rng = np.random.default_rng(2 * k + quant)
    top = 7 if quant == Q4_0 else 127
    q = rng.integers(-top, top + 1, (rows, k))
    at = k // 2 + 1
    q[:3, at] = (5, -5, 0)
    x = synth.activations(rng, k)
    w = rows_of(quant, q, 0x0C00)  # d = 2^-12
    xi = x.copy()
    xi[at] = np.inf
    got = wide(ctx, xi, w, rows, k, quant, il)
    s = np.sign(q[:, at])
    assert np.array_equal(got[s != 0], np.where(s[s != 0] > 0, np.float32(np.inf), np.float32(-np.inf)))
    assert np.all(np.isnan(got[s == 0]))
    xh = (np.float32(1e37) * np.sign(x)).astype(np.float32)
    ref = q @ xh.astype(np.float64) * 2.0 ** -12
    got = wide(ctx, xh, w, rows, k, quant, il).astype(np.float64)
    # an fp32 sum of k products: k roundings of at most sum |x d q| * 2^-24
    bound = k * 2.0 ** -24 * np.sum(np.abs(q * xh.astype(np.float64)), 1) * 2.0 ** -12
    assert np.all(np.isfinite(got)) and np.all(np.abs(got - ref) <= bound)


# one wide launch of the segments; wide segments around one that the segment
# kernel takes (more than 4,096 rows, or 2,048 above in_dim 2560); an in_dim
# that only the wide kernel takes (a launch per segment)
@pytest.mark.parametrize("quant,k,ns", [(Q4_0, 2176, (8, 4, 2052)), (Q8_0, 5056, (1028, 4, 512)), (Q4_0, 5056, (4, 2048)),
                                        (Q4_0, 2560, (4, 4096)), (Q4_0, 2176, (4, 4100, 12)), (Q8_0, 2624, (2052, 8)),
                                        (Q8_0, 96, (8, 12, 4))])
def test_fused_call_gives_the_bits_of_single_calls(ctx, quant, k, ns):
    rng = np.random.default_rng(k + quant)
    x = torch.from_numpy(synth.activations(rng, k)).cuda()
    ws = [torch.from_numpy(synth.weight(rng, quant, n, k, 4)).cuda() for n in ns]
    one = [torch.empty(n, dtype=torch.float32, device="cuda") for n in ns]
    for w, y, n in zip(ws, one, ns):
        ctx.linear_dev(x, w, y, k, n, quant, 4)
    y = torch.full((sum(ns) + 4,), -7.0, dtype=torch.float32, device="cuda")
    parts = list(torch.split(y[:-4], ns))
    ctx.linear_fused_dev(x, [(w, p, n, quant, 4) for w, p, n in zip(ws, parts, ns)], k)
    got = y.cpu().numpy()
    assert np.array_equal(got[:-4].view(np.uint32), torch.cat(one).cpu().numpy().view(np.uint32))
    assert np.all(got[-4:] == -7.0)
