"""The F32-KV attention kernel (and F16 KV at the small head dims it also serves) against the
oracle at the edges of its 32-key tiles and 256-key splits, for every head dim, with query
groups that fill a kernel's head group, leave it partly empty, or take several groups.

A one-layer model prefills prompts of 1, 31, 33 and 256 tokens in one ragged pass (rows at
every position of a tile), then three decode passes take the rows
across the next tile and split boundaries. F32 execution: logits within 2e-4 + 1e-4 |ref|, the
suite's F32 bound (22-bit activation splits, another summation order)."""
import numpy as np
import pytest

import oracle
from hllm_amd import capi, model, synthetic
from tests import helpers_parity as hp
from tests import models

pytestmark = pytest.mark.gpu
LENGTHS, STEPS, VOCAB = (1, 31, 33, 256), 3, 300


def shape_of(head_dim, heads, kv_heads, dtype):
    return synthetic.ModelShape(f"d{head_dim}-g{heads // kv_heads}", 1, 64, 96, heads, kv_heads, head_dim, VOCAB,
                                eps=1e-6, theta=1e4, qk_norm=head_dim >= 64, tied=False, dtype=dtype, max_seq=512)


@pytest.mark.parametrize("head_dim,heads,kv_heads,execution", [
    (4, 8, 1, "f32"), (8, 3, 3, "f32"), (16, 4, 2, "f32"), (32, 6, 2, "f32"), (64, 8, 2, "f32"),
    (128, 4, 2, "f32"), (128, 5, 1, "f32"), (256, 6, 2, "f32"), (4, 4, 2, "f16"), (32, 6, 2, "f16")])
def test_tile_and_split_edges_match_the_oracle(head_dim, heads, kv_heads, execution):
    shape = shape_of(head_dim, heads, kv_heads, "f32" if execution == "f32" else "f16")
    rng = np.random.default_rng(3)
    prompts = [rng.integers(0, VOCAB, n).astype(np.uint64) for n in LENGTHS]
    ids = rng.integers(0, VOCAB, (STEPS, len(LENGTHS))).astype(np.uint64)
    st = capi.Stage(model.stage_config(shape, execution=execution, kv_cache_bytes=16 << 20, max_sequences=4,
                                       max_pass_rows=512))
    model.synthesize(st, shape, seed=5, norm_sigma=0.1)
    ost = oracle.OracleStage(models.synthetic_stage(shape, seed=5, norm_sigma=0.1))
    seqs = [st.allocate(n + STEPS) for n in LENGTHS]
    oseqs = [ost.allocate_sequence(n + STEPS) for n in LENGTHS]

    def check(out, inputs, positions, what):
        for i, (o, x, pos) in enumerate(zip(oseqs, inputs, positions)):
            trace = []
            ost.execute(np.atleast_1d(x), pos, o, trace)
            error = np.abs(out["logits"][i] - trace[-1])
            bound = 2e-4 + 1e-4 * np.abs(trace[-1]) if execution == "f32" else hp.MAX_ABS
            assert (error <= bound).all(), (what, i, error.max())

    hp.say(shape.name, execution, "prefill")
    out = st.execute([capi.item(s, n, 0) for s, n in zip(seqs, LENGTHS)], token_ids=np.concatenate(prompts),
                     want_logits=True)
    check(out, prompts, [0] * len(LENGTHS), "prefill")
    for step in range(STEPS):
        positions = [n + step for n in LENGTHS]
        out = st.execute([capi.item(s, 1, p) for s, p in zip(seqs, positions)], token_ids=ids[step], want_logits=True)
        check(out, ids[step], positions, f"decode {step}")
    st.close()
