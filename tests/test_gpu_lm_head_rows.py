"""The LM head of 65 to 128 sampled rows (the decode GEMM's eight row tiles, unsplit): logits and the five
best log-probabilities against the oracle, and the fused greedy token against the first maximum
of the logits. Vocabulary just wide enough for that kernel and not a multiple of its tiles; hidden
sizes whose 128 rows fit in LDS whole (up to 576) and whose chunks of four k-steps are staged in turn.

Logits within max-abs 2e-2 and cosine 0.9999 (F16 slices); log-probabilities against the
64-bit log-softmax of the GPU's own logits to 1e-12 (a few roundings of 64-bit sums)."""
import numpy as np
import pytest

import oracle
from hllm_amd import capi, model, synthetic
from tests import helpers_parity as hp
from tests import models

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden", [96, 608])
def test_head_of_65_to_128_rows(hidden):
    shape = synthetic.ModelShape(f"head-rows-h{hidden}", 1, hidden, 64, 4, 2, 64, 16500, eps=1e-6, theta=1e4, qk_norm=False,
                                 tied=False, max_seq=128)
    st = capi.Stage(model.stage_config(shape, execution="f16", kv_cache_bytes=16 << 20, max_sequences=128,
                                       max_pass_rows=128))
    model.synthesize(st, shape, seed=5, norm_sigma=0.1)
    ost = oracle.OracleStage(models.synthetic_stage(shape, seed=5, norm_sigma=0.1))
    ids = np.random.default_rng(3).integers(0, shape.vocab, 128).astype(np.uint64)
    expect = []
    for i in ids:
        trace = []
        ost.execute(np.array([i], np.uint64), 0, ost.allocate_sequence(1), trace)
        expect.append(trace[-1])
    for rows in (64, 65, 113, 128):
        hp.say(shape.name, "rows", rows)

        def run(**options):
            seqs = [st.allocate(1) for _ in range(rows)]
            out = st.execute([capi.item(s, 1, 0, logprobs=options.get("top", 0) > 0, top_logprobs=options.get("top", 0))
                              for s in seqs], token_ids=ids[:rows], want_logits=options.get("logits", True))
            for s in seqs:
                st.release(s)
            return out

        out = run(top=5)
        hp.check_rows(out["logits"], np.stack(expect[:rows]), ("logits", rows))
        z = out["logits"].astype(np.float64)
        z -= z.max(1, keepdims=True)
        best = np.sort(z - np.log(np.exp(z).sum(1, keepdims=True)), axis=1)[:, :-6:-1]
        assert np.abs(out["top_logprobs"] - best).max() < 1e-12
        greedy = run(logits=False)
        assert np.array_equal(greedy["tokens"].astype(np.int64), out["logits"].argmax(1))
    st.close()


def test_fused_argmax_of_128_rows_with_a_ragged_last_tile():
    """A vocabulary with 32 features in its last 128-feature tile: the candidates of 128 greedy rows fit,
    so the passes keep the argmax epilogue (no logits, no argmax_partial_kernel) up to 128 rows."""
    shape = synthetic.ModelShape("head-ragged", 1, 96, 64, 4, 2, 64, 128 * 128 + 32, eps=1e-6, theta=1e4, qk_norm=False,
                                 tied=False, max_seq=128)
    st = capi.Stage(model.stage_config(shape, execution="f16", kv_cache_bytes=16 << 20, max_sequences=128,
                                       max_pass_rows=128))
    model.synthesize(st, shape, seed=5, norm_sigma=0.1)
    ids = np.random.default_rng(3).integers(0, shape.vocab, 128).astype(np.uint64)
    tokens = {}
    for logits in (True, False):
        hp.say(shape.name, "logits", logits)
        seqs = [st.allocate(1) for _ in range(128)]
        st.profile("argmax")
        out = st.execute([capi.item(s, 1, 0) for s in seqs], token_ids=ids, want_logits=logits)
        kernels = [r for r in st.profile_records() if r.startswith("argmax/")]
        st.profile(None)
        assert ("argmax/argmax_partial_kernel" in kernels) == logits, kernels
        tokens[logits] = out["tokens"].astype(np.int64)
        if logits:
            assert np.array_equal(tokens[True], out["logits"].argmax(1))
        for s in seqs:
            st.release(s)
    assert np.array_equal(tokens[True], tokens[False])
    st.close()
