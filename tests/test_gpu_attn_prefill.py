"""The batched prefill's attention (zg_attn_prefill.hip) at the edges of its
tiles: 16-key tiles, 32 query columns (16 rows of two heads of a KV head, or
32 rows of one), eight waves that take the tiles in turn.

A row's bits depend on its own position and keys only, so any split of a
prompt into calls gives the same final rows bit for bit; against the oracle
(fp32 attention in its own order) the prefill differs by single roundings of
the 8-bit activations.  The attention on its own is compared with float64.
"""
import numpy as np
import pytest
import torch

from zero_amd import _lib, synth
from zero_amd.model import GpuModel
from zero_amd.ops import ZgError

pytestmark = pytest.mark.gpu


def model(n_q, n_kv, hd, seed, o_kq=False):
    lq = None
    if o_kq:  # a Q4_K O projection reads the attention's fp32 rows
        lq = tuple(tuple((synth.Q4K, 1) if p == 3 else (synth.Q4_0, 4) for p in range(7)) for _ in range(2))
    cfg = synth.ModelConfig(n_layers=2, hidden=256, ffn=512, n_q_heads=n_q, n_kv_heads=n_kv, head_dim=hd,
                            vocab_padded=512, vocab_real=500, max_ctx=330, layer_quants=lq)
    return synth.random_model(cfg, seed=seed)


# query heads per KV head 1, 2, 3 and 4; both head dims
@pytest.mark.parametrize("n_q,n_kv,hd,o_kq", [(4, 4, 64, False), (4, 2, 128, False), (6, 2, 128, False), (8, 2, 64, True)])
def test_prefill_attention_tile_edges(ctx, zo, n_q, n_kv, hd, o_kq):
    m = model(n_q, n_kv, hd, seed=n_q + hd, o_kq=o_kq)
    gm, om = GpuModel(ctx, m), zo.OracleModel(m)
    try:
        prompt = synth.prompt(hd, 300, m.cfg.vocab_real)
        for n in (1, 15, 16, 17, 32, 33, 127, 129, 257):
            gm.reset()
            tok, mx, hid = gm.prefill(prompt[:n], want_hidden=True)
            ref = om.prefill_q8(prompt[:n])
            # the roundings of 8-bit activations that another summation order
            # flips move a tiny model's hidden state by up to 5e-3 each: this
            # bar sees a wrong layout or row, not a single key (those are
            # pinned against float64 below)
            assert np.max(np.abs(hid - ref)) / np.max(np.abs(ref)) <= 2e-2, n
            for cut in {1, 7, 16, n // 2, n - 1}:
                if 0 < cut < n:
                    gm.reset()
                    gm.prefill(prompt[:cut])
                    t2, m2, h2 = gm.prefill(prompt[cut:n], pos0=cut, want_hidden=True)
                    assert t2 == tok and m2 == mx and np.array_equal(h2, hid), (n, cut)
    finally:
        gm.close()
        om.close()
        ctx.clear()


@pytest.mark.parametrize("row", [0, 20, 31, 39])
def test_prefill_attention_nonfinite_row_stays_its_own(ctx, row):
    """A NaN embedding row makes that position's K and V NaN; the rows before
    it, in the same tiles, stay finite: the latch names that row first."""
    m = model(4, 2, 64, seed=3)
    w = m.token_embd.reshape(m.cfg.vocab_padded, -1)
    w[499, :2] = np.frombuffer(np.uint16(0x7E00).tobytes(), np.uint8)
    gm = GpuModel(ctx, m)
    try:
        prompt = synth.prompt(1, 40, 499)
        prompt[row] = 499
        with pytest.raises(ZgError) as ei:
            gm.prefill(prompt)
        assert ei.value.code == _lib.ZG_ERR_ATTENTION
        assert gm.first_nonfinite() == f"L00 k_cache[{row}] n1 i0"
        # a clean prompt afterwards is not touched by what the cache held
        gm.reset()
        clean = synth.prompt(2, 40, 499)
        a = gm.prefill(clean, want_hidden=True)
        gm.reset()
        b = gm.prefill(clean, want_hidden=True)
        assert np.all(np.isfinite(a[2])) and np.array_equal(a[2], b[2])
        gm.prefill(clean[:9])  # rows 9.. of the cache hold other data
        c = gm.prefill(clean[9:], pos0=9, want_hidden=True)
        assert np.array_equal(a[2], c[2])
    finally:
        gm.close()
        ctx.clear()


def test_prefill_across_a_chunk_boundary(ctx):
    """A prompt of more rows than a chunk holds (2,048) gives the bits of the
    same prompt in two calls that cut elsewhere."""
    cfg = synth.ModelConfig(n_layers=1, hidden=256, ffn=256, n_q_heads=4, n_kv_heads=2, head_dim=64, vocab_padded=512,
                            vocab_real=500, max_ctx=2100)
    gm = GpuModel(ctx, synth.random_model(cfg, seed=8))
    try:
        prompt = synth.prompt(5, 2081, cfg.vocab_real)
        a = gm.prefill(prompt, want_hidden=True)
        gm.reset()
        gm.prefill(prompt[:1500])
        b = gm.prefill(prompt[1500:], pos0=1500, want_hidden=True)
        assert a[0] == b[0] and a[1] == b[1] and np.array_equal(a[2], b[2])
    finally:
        gm.close()
        ctx.clear()


def test_prefill_row_buffers_follow_the_prompt_and_the_memory(ctx):
    """The row buffers hold the longest prompt so far in steps of 512 rows;
    where they do not fit, fewer rows run the prompt in more chunks with the
    same bits, down to 512, below which the call fails and a later one runs."""
    cfg = synth.ModelConfig(n_layers=2, hidden=256, ffn=256, n_q_heads=4, n_kv_heads=2, head_dim=64, vocab_padded=512,
                            vocab_real=500, max_ctx=2100)
    gm = GpuModel(ctx, synth.random_model(cfg, seed=9))
    rows, fit = ctx.lib.zg_model_prefill_rows, ctx.lib.zg_model_test_prefill_fit
    try:
        prompt = synth.prompt(6, 2081, cfg.vocab_real)
        assert fit(gm.h, 100) == _lib.ZG_OK and rows(gm.h) == 0
        with pytest.raises(ZgError) as ei:
            gm.prefill(prompt[:10])
        assert ei.value.code == _lib.ZG_ERR_OUT_OF_MEMORY and rows(gm.h) == 0
        assert fit(gm.h, 0) == _lib.ZG_OK
        seen = []
        for n in (10, 512, 513, 10, 1500, 2081):
            gm.reset()
            want = gm.prefill(prompt[:n], want_hidden=True)
            seen.append(rows(gm.h))
        assert seen == [512, 512, 1024, 1024, 1536, 2048]
        gm.close()
        ctx.clear()
        gm = GpuModel(ctx, synth.random_model(cfg, seed=9))
        assert fit(gm.h, 1000) == _lib.ZG_OK
        got = gm.prefill(prompt, want_hidden=True)
        assert rows(gm.h) == 512
        assert got[0] == want[0] and got[1] == want[1] and np.array_equal(got[2], want[2])
    finally:
        gm.close()
        ctx.clear()


def attention(ctx, q, k, v, n_q, n_kv, hd, pos0, q8=False, scratch=True):
    """zg_prefill_attention_dev on host arrays: rows, or (int8, scale) rows."""
    n, ctx_rows = q.shape[0], pos0 + q.shape[0]
    pad = lambda a: np.concatenate([a, np.full((-ctx_rows % 16, n_kv * hd), np.nan, np.float32)])  # noqa: E731
    qd, kd, vd = (torch.from_numpy(a).cuda() for a in (q, pad(k), pad(v)))
    out = torch.full((n + 1, n_q * hd), -7.0, dtype=torch.float32, device="cuda")
    qs = torch.full((n + 1, n_q * hd), 77, dtype=torch.int8, device="cuda")
    d = torch.full((n + 1, n_q * hd // 32), -1, dtype=torch.int16, device="cuda")
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    nb = ctx.lib.zg_prefill_attention_scratch(n_q, n_kv, hd, n) if scratch else 0
    sc = torch.full((nb + 16,), 255, dtype=torch.uint8, device="cuda")  # NaNs, and a guard behind them
    torch.cuda.synchronize()
    ctx.check(ctx.lib.zg_prefill_attention_dev(ctx.h, qd.data_ptr(), kd.data_ptr(), vd.data_ptr(),
                                               None if q8 else out.data_ptr(), qs.data_ptr(), d.data_ptr(), err.data_ptr(),
                                               n_q, n_kv, hd, n, pos0, sc.data_ptr() if nb else None, nb, None))
    torch.cuda.synchronize()
    assert torch.all(sc[nb:] == 255)
    out, qs, d = out.cpu().numpy(), qs.cpu().numpy(), d.cpu().numpy()
    # nothing past the last row, and only the asked-for form
    assert np.all(out[n if not q8 else 0:] == -7.0) and np.all(qs[n if q8 else 0:] == 77) and np.all(d[n if q8 else 0:] == -1)
    return (qs[:n], d[:n].view(np.float16), int(err)) if q8 else (out[:n], int(err))


def attention_f64(q, k, v, n_q, n_kv, hd, pos0):
    n, g = q.shape[0], n_q // n_kv
    q, k, v = (a.astype(np.float64) for a in (q, k, v))
    out = np.empty((n, n_q * hd))
    seen = np.arange(pos0 + n)[None] <= pos0 + np.arange(n)[:, None]
    for h in range(n_q):
        kv = slice(h // g * hd, (h // g + 1) * hd)
        s = q[:, h * hd:(h + 1) * hd] @ k[:, kv].T / np.sqrt(hd)
        s = np.where(seen, s, -np.inf)
        p = np.exp(s - s.max(1, keepdims=True))
        out[:, h * hd:(h + 1) * hd] = p / p.sum(1, keepdims=True) @ v[:, kv]
    return out


# query heads per KV head 1, 2, 3 and 8, both head dims; contexts of one tile,
# four (the short form's most), five, a tile edge and a row either side, more
# than one round of the eight waves, at the start of the cache and behind rows
@pytest.mark.parametrize("n,pos0", [(1, 0), (16, 0), (17, 0), (64, 0), (65, 0), (127, 0), (128, 0), (129, 0), (257, 0),
                                    (1, 63), (1, 64), (15, 17), (33, 128), (40, 250), (1, 127), (1, 128), (5, 400), (33, 300)])
@pytest.mark.parametrize("n_q,n_kv,hd", [(2, 2, 128), (4, 2, 64), (4, 2, 128), (6, 2, 64), (3, 1, 128), (8, 1, 64)])
def test_attention_against_float64(ctx, n_q, n_kv, hd, n, pos0):
    """With scratch (few rows behind more than four tiles share their slots
    over workgroups) and without, the same bits.  Scores of spread about 1, values of spread 1: an fp32 score is off by at
    most hd * 2^-24 * sum |q k| / sqrt(hd) (under 1e-5 here, most of it far
    below), which moves the weights by as much relatively and the row by 1e-5
    of the largest value.  A key dropped, doubled or let past the mask moves
    it by its weight, 1 / 405 and more."""
    rng = np.random.default_rng(n + 7 * pos0 + 100 * n_q + hd)
    rows = pos0 + n
    q = rng.standard_normal((n, n_q * hd)).astype(np.float32)
    k, v = (rng.standard_normal((rows, n_kv * hd)).astype(np.float32) for _ in range(2))
    want = attention_f64(q, k, v, n_q, n_kv, hd, pos0)
    got, err = attention(ctx, q, k, v, n_q, n_kv, hd, pos0)
    assert err == 0 and np.max(np.abs(got - want)) <= 1e-5 * np.max(np.abs(v))
    one, err = attention(ctx, q, k, v, n_q, n_kv, hd, pos0, scratch=False)
    assert err == 0 and np.array_equal(one.view(np.uint32), got.view(np.uint32))
    qs, d, err = attention(ctx, q, k, v, n_q, n_kv, hd, pos0, q8=True)
    # a block's scale is max / 127 rounded to fp16 (2^-11), its values rounded
    # to half a step and clipped at 127 of them
    b, dd = want.reshape(n, -1, 32), d.astype(np.float64)[..., None]
    step = np.max(np.abs(b), 2, keepdims=True) / 127
    assert err == 0 and np.all(np.abs(dd - step) <= step * 2.0 ** -10)
    assert np.all(np.abs(qs.reshape(b.shape) * step - b) <= step * 0.5 + 1e-5 * np.max(np.abs(v)))


# more than 64 units of five to eight tiles, and of nine: the long form
@pytest.mark.parametrize("n,pos0", [(113, 0), (128, 0), (113, 16)])
def test_attention_of_many_units(ctx, n, pos0):
    test_attention_against_float64(ctx, 24, 12, 64, n, pos0)


@pytest.mark.parametrize("n_q,n_kv,hd,n,pos0", [(2, 2, 128, 150, 0), (4, 2, 64, 40, 100), (3, 1, 64, 60, 0)])
def test_attention_single_keys(ctx, n_q, n_kv, hd, n, pos0):
    """Every row's query picks one key (the first, its own, tile edges, ...),
    whose score is far above the others': the row is that key's value row."""
    rng = np.random.default_rng(hd + n)
    rows, g = pos0 + n, n_q // n_kv
    k = rng.choice([-1.0, 1.0], size=(rows, n_kv * hd)).astype(np.float32)
    v = rng.standard_normal((rows, n_kv * hd)).astype(np.float32)
    pick = np.empty((n, n_q), np.int64)
    q = np.empty((n, n_q * hd), np.float32)
    for z in range(n):
        p = pos0 + z
        edges = [c for c in (0, p, p - 1, p // 16 * 16, p // 16 * 16 - 1, p // 128 * 128, p // 2) if c >= 0]
        for h in range(n_q):
            pick[z, h] = edges[(z + h) % len(edges)]
            q[z, h * hd:(h + 1) * hd] = 8 * k[pick[z, h], h // g * hd:(h // g + 1) * hd]
    got, err = attention(ctx, q, k, v, n_q, n_kv, hd, pos0)
    # the picked score is 8 sqrt(hd) and another's below 0.7 of it (keys of
    # random signs): their weights are under exp(-19) each
    for h in range(n_q):
        want = v[pick[:, h], h // g * hd:(h // g + 1) * hd]
        assert err == 0 and np.max(np.abs(got[:, h * hd:(h + 1) * hd] - want)) <= 1e-5, h
