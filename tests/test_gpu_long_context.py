"""Decode steps on both sides of the long-context switch (position 640: more
attention splits and, in the fused Q|K|V + attention launch, longer rounds):
greedy tokens and hidden states against the oracle across it, and the same
bits from single steps and from the device loop."""
import ctypes as C

import numpy as np
import pytest

from zero_amd import synth
from zero_amd.model import GpuModel

pytestmark = pytest.mark.gpu

REL_TOL = 1e-3  # parity bar of the decode path


# fused launch (in_dim 2048) with Q4_0X4 and with Q4_K weights; separate launches
@pytest.mark.parametrize("hidden,lin,n_q,n_kv,hd", [(2048, (synth.Q4_0, 4), 8, 4, 128), (2048, (synth.Q4K, 1), 4, 2, 64),
                                                    (256, (synth.Q4_0, 4), 8, 2, 128)])
def test_decode_across_the_long_context_switch(ctx, zo, hidden, lin, n_q, n_kv, hd):
    cfg = synth.ModelConfig(n_layers=1, hidden=hidden, ffn=512, n_q_heads=n_q, n_kv_heads=n_kv, head_dim=hd,
                            vocab_padded=512, vocab_real=500, max_ctx=720, lin_type=lin[0], lin_interleave=lin[1])
    model = synth.random_model(cfg, seed=hidden + hd)
    gm, om = GpuModel(ctx, model), zo.OracleModel(model)
    try:
        prompt = synth.prompt(hd, 600, cfg.vocab_real)
        toks, _, _ = gm.generate(prompt, 120)
        assert np.array_equal(toks, om.generate(prompt, 120))
        # the same rows again, step by step around the switch
        for pos in list(range(634, 648)) + [704, 718]:
            t = int(toks[pos - 600])
            nxt, _, hid, _ = gm.step(t, pos, want_hidden=True)
            assert nxt == int(toks[pos - 599])
            ref = om.forward(t, pos)
            assert np.max(np.abs(hid - ref)) / np.max(np.abs(ref)) <= REL_TOL
    finally:
        gm.close()
        om.close()
        ctx.clear()


# the fused long form's second round of 128 rows: eight splits hold 128 rows
# each at position 1,023 and 136 from 1,024 on
@pytest.mark.parametrize("lin,n_q,n_kv,hd", [((synth.Q4_0, 4), 8, 4, 128), ((synth.Q4K, 1), 4, 2, 64)])
def test_decode_across_the_second_round(ctx, zo, lin, n_q, n_kv, hd):
    cfg = synth.ModelConfig(n_layers=1, hidden=2048, ffn=512, n_q_heads=n_q, n_kv_heads=n_kv, head_dim=hd, vocab_padded=512,
                            vocab_real=500, max_ctx=1100, lin_type=lin[0], lin_interleave=lin[1])
    model = synth.random_model(cfg, seed=3 * hd)
    gm, om = GpuModel(ctx, model), zo.OracleModel(model)
    try:
        prompt = synth.prompt(hd + 1, 1016, cfg.vocab_real)
        toks, _, _ = gm.generate(prompt, 80)
        assert np.array_equal(toks, om.generate(prompt, 80))
        for pos in list(range(1020, 1030)) + [1060, 1094]:
            t = int(toks[pos - 1016])
            nxt, _, hid, _ = gm.step(t, pos, want_hidden=True)
            assert nxt == int(toks[pos - 1015])
            ref = om.forward(t, pos)
            assert np.max(np.abs(hid - ref)) / np.max(np.abs(ref)) <= REL_TOL
    finally:
        gm.close()
        om.close()
        ctx.clear()


# (query heads, KV heads, head dim): splits of the steps past the switch
@pytest.mark.parametrize("n_q,n_kv,hd,splits", [(16, 8, 128, 8), (22, 11, 128, 8), (24, 8, 128, 6), (32, 8, 128, 6),
                                                (31, 31, 64, 8), (32, 8, 64, 6)])
def test_waiting_workgroups_leave_slots_for_the_gemv(ctx, n_q, n_kv, hd, splits):
    """The attention workgroups of the fused launch wait for its GEMV: those of
    four such launches at once (four contexts) have to be fewer than the
    device holds, or the launch keeps the base form's six splits."""
    cfg = synth.ModelConfig(n_layers=1, hidden=2048, ffn=512, n_q_heads=n_q, n_kv_heads=n_kv, head_dim=hd, vocab_padded=512,
                            vocab_real=500, max_ctx=720)
    gm = GpuModel(ctx, synth.random_model(cfg, seed=n_q))
    try:
        for pos in (0, 639, 640, 719):
            w, slots = C.c_uint32(), C.c_uint32()
            ctx.check(ctx.lib.zg_model_step_waiters(gm.h, pos, C.byref(w), C.byref(slots)))
            assert w.value == n_q * (splits if pos >= 640 else 6)
            assert 4 * w.value < slots.value, pos
    finally:
        gm.close()
        ctx.clear()
