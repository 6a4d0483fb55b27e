"""The prefill GEMMs' tile forms, bit for bit against the oracle, at sizes
around their dispatch rules: the Q8_0-activation GEMM's 32 x 32 tiles (at most
half a 32 x 64 tile per CU) and its 64-row tile with the scales' outer
product by MFMA, with subnormal, zero and large fp16 scales; the K-quant
GEMM's 32-row and 64-row tiles with two superblock groups per workgroup."""
import numpy as np
import pytest
import torch

from zero_amd import synth

pytestmark = pytest.mark.gpu

Q4_0, Q8_0, Q4K, Q6K = 2, 8, 12, 14


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def same_bits(a, b):
    return np.array_equal(a.view(np.uint32), b.view(np.uint32))


# few tiles: whole ones whose width is no multiple of 64, partial rows and
# columns, one stage and a partial last stage, on the 32-row tile; then in_dims
# from the narrow tile's 1024 (Q4_0) and 2048 (Q8_0) on, and the first below;
# and the first width past the narrow tile
@pytest.mark.parametrize("wt", [Q4_0, Q8_0])
@pytest.mark.parametrize("il,m,n,k", [(4, 32, 96, 256), (1, 33, 100, 544), (4, 1, 4, 32), (1, 64, 1340, 512),
                                      (4, 16, 8192, 256), (4, 16, 8256, 256), (4, 32, 96, 2048), (1, 33, 100, 2080),
                                      (4, 1, 4, 2080), (1, 64, 1340, 2048), (4, 33, 100, 1024), (1, 17, 36, 1056),
                                      (4, 33, 100, 992), (1, 17, 36, 2016), (4, 16, 8192, 2048), (4, 16, 8256, 2048)])
def test_q8act_narrow_tiles(ctx, zo, wt, il, m, n, k):
    rng = np.random.default_rng(m + n + k + wt)
    w, x = synth.weight(rng, wt, n, k, il), synth.activations(rng, m * k).reshape(m, k)
    check_q8act(ctx, zo, w, x, wt, il, m, n, k)


# 768 and more 64 x 64 tiles: the 64-row form, whole and with partial tiles
@pytest.mark.parametrize("wt,il,m,n", [(Q4_0, 4, 64, 49152), (Q8_0, 1, 65, 24640), (Q4_0, 1, 64, 49156)])
def test_q8act_scales_by_mfma(ctx, zo, wt, il, m, n):
    k = 128
    rng = np.random.default_rng(n + wt)
    w = synth.weight(rng, wt, n, k, 1).reshape(n * (k // 32), -1)
    # weight scales over fp16's range: zeros, subnormals, ordinary, near the top
    d = rng.choice(np.array([0x0000, 0x0001, 0x03FF, 0x0400, 0x1C00, 0x2E66, 0x3C00, 0x7BFF, 0x8001, 0xBC00], np.uint16),
                   size=w.shape[0])
    w[:, :2] = d.view(np.uint8).reshape(-1, 2)
    w = w.reshape(-1)
    if il == 4:
        w = synth.interleave_x4(w, n, k, wt)
    x = synth.activations(rng, m * k).reshape(m, k)
    x[0] *= np.float32(1e-6)   # activation scales below the smallest normal fp16
    x[1, :32] = 0.0
    x[2] *= np.float32(1e4)
    check_q8act(ctx, zo, w, x, wt, il, m, n, k)


# the same kernel on split-scale groups (in_dims a multiple of 512), as a
# model's long prefill runs it: whole tiles, and partial ones in both directions
@pytest.mark.parametrize("wt", [Q4_0, Q8_0])
@pytest.mark.parametrize("m,n", [(64, 49152), (65, 24644)])
def test_q8act_scales_by_mfma_split_groups(ctx, wt, m, n):
    k = 512
    rng = np.random.default_rng(m + n + wt)
    w = synth.weight(rng, wt, n, k, 4)
    qs = torch.empty((m, k), dtype=torch.int8, device="cuda")
    d = torch.empty((m, k // 32), dtype=torch.int16, device="cuda")
    ctx.quantize_q8_0_split_dev(dev(synth.activations(rng, m * k).reshape(m, k)), qs, d, m, k)
    ys = []
    for il, wb in ((4, w), (5, synth.x4_split(w, n, k, wt))):
        ys.append(torch.full((m, n), -3.0, dtype=torch.float32, device="cuda"))
        ctx.gemm_q8act_dev(qs, d, dev(wb), ys[-1], m, n, k, wt, il)
    assert same_bits(ys[0].cpu().numpy(), ys[1].cpu().numpy())


def check_q8act(ctx, zo, w, x, wt, il, m, n, k):
    qs = torch.empty((m, k), dtype=torch.int8, device="cuda")
    d = torch.empty((m, k // 32), dtype=torch.int16, device="cuda")
    y = torch.full((m, n), -3.0, dtype=torch.float32, device="cuda")
    ctx.quantize_q8_0_split_dev(dev(x), qs, d, m, k)
    ctx.gemm_q8act_dev(qs, d, dev(w), y, m, n, k, wt, il)
    ref = zo.gemm_q8act(zo.quantize_q8_0(x.reshape(-1)), w, m, n, k, wt, il)
    assert same_bits(y.cpu().numpy(), ref)


# two groups per workgroup need an even superblock count: 32-row tiles around
# their edge, 64-row ones once the 32-row tiles outnumber the CUs, one group
# for an odd count
@pytest.mark.parametrize("wt", [Q4K, Q6K])
@pytest.mark.parametrize("m,n,k", [(31, 64, 512), (32, 12288, 512), (33, 128, 1024), (97, 4096, 512), (150, 4096, 512),
                                   (33, 128, 768)])
def test_q8k_tile_forms(ctx, zo, wt, m, n, k):
    rng = np.random.default_rng(m + n + k + wt)
    w, x = synth.weight(rng, wt, n, k, 1), synth.activations(rng, m * k).reshape(m, k)
    qs = torch.empty((m, k), dtype=torch.int8, device="cuda")
    d8 = torch.empty((m, k // 256), dtype=torch.float32, device="cuda")
    bs = torch.empty((m, k // 32), dtype=torch.int16, device="cuda")
    ctx.quantize_q8k_split_dev(dev(x), qs, d8, bs, m, k)
    y = torch.full((m, n), -3.0, dtype=torch.float32, device="cuda")
    ctx.gemm_q8k_dev(qs, d8, bs, dev(w), y, m, n, k, wt)
    f = zo.linear_q4k_q8k if wt == Q4K else zo.linear_q6k_q8k
    rows = range(m) if m * n <= 1 << 16 else [0, 15, 16, m // 2, m - 2, m - 1]
    got = y.cpu().numpy()
    for i in rows:
        assert same_bits(got[i], f(zo.quantize_q8k(x[i]), w, k, n)), i
    y0 = synth.activations(rng, m * n).reshape(m, n)
    y = dev(y0)
    ctx.gemm_q8k_dev(qs, d8, bs, dev(w), y, m, n, k, wt, accumulate=True)
    assert same_bits(y.cpu().numpy(), y0 + got)
