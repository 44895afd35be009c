"""Passes of one and two rows, whose RMSNorms are folded into q/k/v and gate+up, against the oracle
and beside passes of three rows (separate norms): row lengths around the chunk counts of both
kernels, several layers (the residual rows alternate between two buffers), and both ends (final
norm and head; boundary rows). Partials of o and of down, up to more than one round of loads of
each folded kernel, in test_partials_in_folded_norms, also bit for bit against separate norms.

Logits and boundary rows within max-abs 2e-2 and cosine 0.9999, as for the other F16 slices."""
import numpy as np
import pytest

import oracle
from hllm_amd import capi, model, synthetic
from tests import helpers_parity as hp
from tests import models

pytestmark = pytest.mark.gpu
PROMPT, STEPS, VOCAB = 5, 3, 300


@pytest.mark.parametrize("hidden,intermediate,final", [
    (64, 96, True), (1024, 160, False), (1056, 1600, True), (2048, 96, True), (2080, 352, False), (3104, 544, True),
    (4096, 2080, False)])
def test_folded_norms_match_the_oracle(hidden, intermediate, final):
    shape = synthetic.ModelShape(f"h{hidden}", 3, hidden, intermediate, 4, 2, 64, VOCAB, eps=1e-6, theta=1e4,
                                 qk_norm=False, tied=False, max_seq=64)
    end = 3 if final else 2
    st = capi.Stage(model.stage_config(shape, 0, end, first=True, final=final, execution="f16",
                                       kv_cache_bytes=16 << 20, max_sequences=8, max_pass_rows=64))
    model.synthesize(st, shape, seed=5, norm_sigma=0.1)
    ost = oracle.OracleStage(models.synthetic_stage(shape, 0, end, first=True, final=final, seed=5, norm_sigma=0.1))
    rng = np.random.default_rng(3)
    for rows in (1, 2, 3):
        ids = rng.integers(0, VOCAB, (PROMPT + STEPS, rows)).astype(np.uint64)
        seqs = [st.allocate(PROMPT + STEPS) for _ in range(rows)]
        oseqs = [ost.allocate_sequence(PROMPT + STEPS) for _ in range(rows)]
        for r in range(rows):
            st.execute([capi.item(seqs[r], PROMPT, 0, sample=False)], token_ids=ids[:PROMPT, r])
            ost.execute(np.ascontiguousarray(ids[:PROMPT, r]), 0, oseqs[r])
        for step in range(STEPS):
            hp.say(shape.name, "rows", rows, "step", step)
            position = PROMPT + step
            out = st.execute([capi.item(s, 1, position, sample=final) for s in seqs], token_ids=ids[position],
                             want_logits=final)
            expect = []
            for r in range(rows):
                trace = []
                result = ost.execute(ids[position, r:r + 1].copy(), position, oseqs[r], trace)
                expect.append(trace[-1] if final else oracle.f16_decode(result[1])[0])
            got = out["logits"] if final else oracle.f16_decode(out["boundary"])
            hp.check_rows(got, np.stack(expect), (shape.name, rows, step))
        for s in seqs:
            st.release(s)
    st.close()


# Shapes whose o and down leave partials to the folded norms (6 waves per CU of 256 over 128-feature
# workgroups of eight waves, whole chunks of four k-steps): hidden 896: o 4 and down 19, past the
# q/k/v kernel's 12 loads in flight; 1024: o 16, past the pair kernel's 12 (one chunk of columns
# per thread); 2080: o 11, past its 6 (two chunks); 3072: o 8 and down 8.
@pytest.mark.parametrize("hidden,intermediate,heads,head_dim", [
    (896, 4864, 16, 64), (1024, 1600, 32, 128), (2080, 352, 32, 128), (3072, 2048, 32, 128)])
def test_partials_in_folded_norms(monkeypatch, hidden, intermediate, heads, head_dim):
    """Against the oracle, and bit for bit against passes with separate norms."""
    shape = synthetic.ModelShape(f"h{hidden}", 2, hidden, intermediate, heads, 4, head_dim, VOCAB, eps=1e-6, theta=1e4,
                                 qk_norm=False, tied=False, max_seq=64)
    st = capi.Stage(model.stage_config(shape, execution="f16", kv_cache_bytes=16 << 20, max_sequences=8,
                                       max_pass_rows=64))
    model.synthesize(st, shape, seed=5, norm_sigma=0.1)
    ost = oracle.OracleStage(models.synthetic_stage(shape, seed=5, norm_sigma=0.1))
    rng = np.random.default_rng(3)
    steps = 2
    for rows in (1, 2):
        ids = rng.integers(0, VOCAB, (steps, rows)).astype(np.uint64)
        oseqs = [ost.allocate_sequence(steps) for _ in range(rows)]
        seqs = {fold: [st.allocate(steps) for _ in range(rows)] for fold in "10"}
        for step in range(steps):
            got = {}
            for fold in "10":
                hp.say(shape.name, "rows", rows, "step", step, "fold", fold)
                monkeypatch.setenv("HLLM_ROCM_NORM_FOLD", fold)
                st.profile("gemm")
                got[fold] = st.execute([capi.item(s, 1, step) for s in seqs[fold]], token_ids=ids[step],
                                       want_logits=True)["logits"]
                folded = "gemm_qkv/gemm_norm_kernel" in st.profile_records()
                st.profile(None)
                assert folded == (fold == "1" and rows * hidden <= 4096)
            assert np.array_equal(got["1"], got["0"]), (shape.name, rows, step)
            expect = []
            for r in range(rows):
                trace = []
                ost.execute(ids[step, r:r + 1].copy(), step, oseqs[r], trace)
                expect.append(trace[-1])
            hp.check_rows(got["1"], np.stack(expect), (shape.name, rows, step))
        for s in seqs["1"] + seqs["0"]:
            st.release(s)
    st.close()


def test_switch_is_part_of_a_captured_pass(monkeypatch):
    """With graphs enabled, a pass with HLLM_ROCM_NORM_FOLD=0 does not replay the folded pass's
    graph, nor the other way round, and every pass returns the bits of an eager stage."""
    shape = synthetic.ModelShape("graphs", 2, 1024, 1600, 4, 2, 64, VOCAB, eps=1e-6, theta=1e4, qk_norm=False,
                                 tied=False, max_seq=64)
    ids = np.random.default_rng(3).integers(0, VOCAB, 7).astype(np.uint64)
    stages = []
    for graphs in (False, True):
        st = capi.Stage(model.stage_config(shape, 0, 1, first=True, final=False, execution="f16",
                                           kv_cache_bytes=16 << 20, max_sequences=4, max_pass_rows=64))
        model.synthesize(st, shape, seed=5, norm_sigma=0.1)
        st.set_graphs(graphs)
        stages.append((st, st.allocate(len(ids))))
    stats = []
    for position, fold in enumerate("1110011"):
        hp.say("graphs", "position", position, "fold", fold)
        monkeypatch.setenv("HLLM_ROCM_NORM_FOLD", fold)
        eager, replayed = [st.execute([capi.item(seq, 1, position, sample=False)],
                                      token_ids=ids[position:position + 1])["boundary"] for st, seq in stages]
        assert np.array_equal(eager, replayed), position
        stats.append(stages[1][0].graph_stats())
    # (captured, replayed): folded eager, captured, replayed; unfolded eager, captured; folded replayed.
    assert stats == [(0, 0), (1, 1), (1, 2), (1, 2), (2, 3), (2, 4), (2, 5)], stats
    for st, _ in stages:
        st.close()
