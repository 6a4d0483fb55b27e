"""The batched prefill's attention (zg_attn_prefill.hip) at the edges of its
tiles: 16-key tiles, 32 query columns (16 rows of two heads of a KV head, or
32 rows of one), eight waves that take the tiles in turn.

A row's bits depend on its own position and keys only, so any split of a
prompt into calls gives the same final rows bit for bit; against the oracle
(fp32 attention in its own order) the prefill differs by single roundings of
the 8-bit activations.
"""
import numpy as np
import pytest

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
            # flips move a tiny model's hidden state by up to 5e-3 each; an
            # attention mistake by the size of the state
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
