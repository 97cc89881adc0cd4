"""Prefill launches that carry the f16 row prepass of the matmul after them: the batched
attention merge (attention_merge_half) and silu_mul in sixteen waves (silu_half_rows_wide, rows
of more than 4096 values).  The same f32 and f16 rows as the separate launches, so the same
logits bit for bit, over chunks with a ragged end and contexts of several splits, and in a Q8_0
model whose rows pass f16's range."""
import dataclasses

import numpy as np
import pytest

from helpers import tactics
from skyla_hip import engine as E
from skyla_hip import synth

pytestmark = pytest.mark.gpu

CFG = "test-prefill-joins"


def _logits(ctx, c, tensors, prompt, **tactic):
    with tactics(**tactic):
        eng = E.Engine(ctx, tensors, c, 40 * E.ATTENTION_CHUNK, E.KvPrecision.F16_KEYS_Q8_VALUES)
        try:
            rows = [eng.prefill(prompt).copy(), eng.step(int(prompt[0])).copy()]
            return np.stack(rows).view(np.uint32), eng.recording(True, E.BATCH).launches()
        finally:
            eng.free()


# one chunk of one row; a ragged second chunk; more than 16 splits (the merge's other loop)
@pytest.mark.parametrize("n_prompt", [2, E.BATCH + 22, 17 * E.ATTENTION_CHUNK + 5])
def test_merge_with_prepass_same_logits(ctx, n_prompt):
    c = synth.qwen3_config("tiny")
    tensors = synth.qwen3(CFG, c, "q4_k_m", "random")
    prompt = synth.prompt(f"{CFG}-{n_prompt}", n_prompt, c.n_vocab)
    got, n1 = _logits(ctx, c, tensors, prompt)
    want, n0 = _logits(ctx, c, tensors, prompt, merge_join="0")
    assert n0 - n1 == c.n_layer and np.array_equal(got, want)


# either side of the line at 4096 values, and the longest rows (12288: three full passes)
@pytest.mark.parametrize("n_ff", [4096, 4352, 12288])
def test_wide_silu_with_prepass_same_logits(ctx, n_ff):
    c = dataclasses.replace(synth.qwen3_config("tiny"), n_ff=n_ff)
    tensors = synth.qwen3(f"{CFG}-{n_ff}", c, "q4_k_m", "random")
    prompt = synth.prompt(f"{CFG}-ff", 45, c.n_vocab)
    got, n1 = _logits(ctx, c, tensors, prompt)
    want, n0 = _logits(ctx, c, tensors, prompt, xhalf_join="0")
    assert n0 > n1 and np.array_equal(got, want)


# rows below and above the line at 4096 values
@pytest.mark.parametrize("n_ff", [3072, 4384])
def test_joins_past_f16_range_same_logits(ctx, n_ff):
    """Norm weights of 1e5 put the rows that q, k, v, o, gate, up and down read past 2^15: each
    run of 128 values then has an exponent, written by the joined launches as by x_half_rows."""
    c = dataclasses.replace(synth.qwen3_config("tiny"), n_ff=n_ff)
    tensors = synth.qwen3(f"{CFG}-range-{n_ff}", c, "q8_0", "random")
    for i in range(c.n_layer):
        for name in ("attn_norm", "ffn_norm"):
            tensors[f"blk.{i}.{name}.weight"] = tensors[f"blk.{i}.{name}.weight"] * np.float32(1e5)
    prompt = synth.prompt(f"{CFG}-range", E.BATCH + 22, c.n_vocab)
    got, n1 = _logits(ctx, c, tensors, prompt)
    want, n0 = _logits(ctx, c, tensors, prompt, xhalf_join="0", merge_join="0")
    assert n0 > n1 and np.array_equal(got, want) and np.isfinite(got.view(np.float32)).all()
    tile, _ = _logits(ctx, c, tensors, prompt, ring="0")
    g, w = got.view(np.float32)[0].astype(np.float64), tile.view(np.float32)[0].astype(np.float64)
    assert np.linalg.norm(g - w) <= 1e-2 * np.linalg.norm(w)


@pytest.mark.parametrize("n_head,n_kv,n_split,joined", [(16, 2, 64, True), (16, 2, 65, False), (32, 4, 8, True),
                                                        (32, 4, 9, False), (40, 5, 2, False)])
def test_merge_keeps_to_itself_past_its_heads_and_splits(ctx, n_head, n_kv, n_split, joined):
    """The merge carries the prepass only where one workgroup a token is no slower than the two
    launches (up to 16 heads over 64 splits, 32 over 8); elsewhere it is a launch of its own."""
    c = dataclasses.replace(synth.qwen3_config("tiny"), n_head=n_head, n_head_kv=n_kv, n_layer=1)
    tensors = synth.qwen3(f"{CFG}-{n_head}", c, "q4_k_m", "random")
    n = {}
    for join in ("1", "0"):
        with tactics(merge_join=join):
            eng = E.Engine(ctx, tensors, c, n_split * E.ATTENTION_CHUNK, E.KvPrecision.F16)
            try:
                n[join] = eng.recording(True, n_split * E.ATTENTION_CHUNK).launches()
            finally:
                eng.free()
    assert n["0"] - n["1"] == (1 if joined else 0)
