"""Launch-plan choices of the runtime that lossless speculation relies on,
checked without a GPU: everything that changes a row's arithmetic must be
the same for the plain and the speculative state of one batch."""

import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "dryft-challenge_amd"))


@pytest.mark.parametrize("batch", list(range(1, 65)))
@pytest.mark.parametrize("group", [1, 2, 4, 5, 8, 16])
def test_attention_waves_fit_every_state_of_a_batch(batch, group):
    from engine import spec_k
    from qdec.runtime import attn_waves, max_rows_per_seq
    waves = attn_waves(batch)
    assert waves in (4, 8)

    def max_t(requested):  # DecodeState's clamp
        return max_rows_per_seq(batch, requested, group)

    k = spec_k(batch, group)
    plain, spec = max_t(16), max_t(k + 1 if k else 16)
    if waves == 8:  # the 8-wave body takes at most 8 rows per sequence
        assert plain <= 8 and spec <= 8
    # query rows per kv head within what the attention takes (qdec_attn)
    assert plain * group <= (32 if waves == 8 else 64) and spec * group <= (32 if waves == 8 else 64)
    assert k + 1 <= max_t(16) or k == 0
    # verify rows of a speculative state stay on the one-M-tile GEMM path
    assert batch * (k + 1) <= 16 or k == 0


@pytest.mark.parametrize("batch,nkv,head_dim,cap,waves", [
    (1, 8, 128, 1024, 4), (8, 8, 128, 1024, 8), (32, 8, 128, 4384, 8), (33, 8, 128, 1024, 4), (64, 8, 128, 512, 4),
    (64, 8, 128, 480, 8), (33, 4, 128, 1024, 8), (64, 4, 128, 2080, 8), (64, 2, 128, 1024, 8), (48, 16, 128, 1024, 4),
    (8, 2, 64, 128, 4), (64, 8, 64, 1024, 4)])
def test_state_attention_waves(batch, nkv, head_dim, cap, waves):
    """4 waves above batch 32 only where batch x kv heads are more workgroups
    than CUs."""
    from qdec.runtime import state_attn_waves
    assert state_attn_waves(batch, nkv, head_dim, cap) == waves


def test_lm_head_grouping_divides_the_vocab():
    from qdec.checkpoint import qwen3_config
    from qdec.runtime import LM_TILES_BATCHED, role_plan
    vocab, hidden = qwen3_config()["vocab_size"], qwen3_config()["hidden_size"]
    assert (vocab // 16) % LM_TILES_BATCHED == 0
    assert (vocab // 16) % role_plan(vocab, hidden, "lm")[2] == 0


@pytest.mark.parametrize("hidden,vocab", [(1024, 151936), (2560, 151936), (640, 151936), (320, 151936), (1344, 151936),
                                          (2080, 151936), (2560, 4096), (320, 1024), (2560, 16896 + 16)])
def test_lm_head_grouping_is_accepted(hidden, vocab):
    """Every lm_head call of a state plans, with and without a split update to
    merge, and from 9 rows takes the grouping measured faster."""
    from qdec import capi
    from qdec.runtime import LM_TILES_BATCHED, lm_tiles, role_plan
    lib = capi.lib()
    waves = role_plan(vocab, hidden, "lm")[1]
    got = {}
    for rows in range(2, 65):
        for merges in (False, True):
            t = got[rows, merges] = lm_tiles(rows, vocab, hidden, waves, merges)
            a = capi.GemmArgs(x=16, w=16, norm_w=16, ids_out=16, eps=1e-6, rows=rows, n=vocab, k=hidden, ksplit=1, waves=waves,
                              flags=capi.NORM_IN | capi.ARGMAX, tiles_per_wg=t)
            if merges:
                if rows < 9:  # states of 9 or more sequences split the down projection
                    continue
                a.x_parts, a.x_nparts, a.x_merged = 16, 4, 32
            lib.gemm_workspace(a)
    small = vocab < 151936
    for rows, want in ((8, 8), (9, 8 if hidden in (320, 1344, 2080) and not small else 1),
                       (24, 8 if hidden in (320, 640, 1024, 2080) and not small else 1), (33, 1), (64, 1)):
        if (vocab // 16) % LM_TILES_BATCHED == 0:
            assert got[rows, False] == want, rows
        else:
            assert got[rows, False] == 1


@pytest.mark.parametrize("n,k", [(2560, 4096), (2560, 9728), (2048, 6144), (1024, 3072), (1024, 2048), (4096, 12288),
                                 (5120, 25600), (320, 704), (1152, 1152)])
def test_prefill_split_fills_one_round(n, k):
    """k parts of a short prompt's O and down: whole 64-element stages in each
    part, and no more tiles than one round of the CUs."""
    from qdec.runtime import prefill_split, round_up
    for rows in range(129, 2049):
        parts, tiles = prefill_split(rows, n, k), round_up(rows, 256) // 256 * (n // 128)
        assert 1 <= parts <= 8 and (parts == 1 or (n % 128 == 0 and k % (64 * parts) == 0 and parts * tiles <= 256))
        if n % 128 == 0 and parts < 8 and k % (128 * parts) == 0:
            assert 2 * parts * tiles > 256  # the most that fit
