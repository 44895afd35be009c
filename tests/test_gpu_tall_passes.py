"""F16 passes of 224 rows and more at the edges of the projection tiles chosen for them (128, 192
and 256 rows, with and without K splits): the choice by shape against the 64-row tiles of the
activation-staged kernel (checked against the oracle by the configuration tests), on one layer
of Falcon3-3B's and of Qwen3-0.6B's shape. Bounds per row as for the other F16 slices."""
import numpy as np
import pytest

import oracle
from hllm_amd import capi, model, synthetic
from tests import helpers_parity as hp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [synthetic.FALCON3_3B, synthetic.QWEN3_0_6B], ids=lambda s: s.name)
def test_choice_by_shape_matches_64_row_tiles(shape):
    st = capi.Stage(model.stage_config(shape, 0, 1, first=True, final=False, execution="f16", kv_cache_bytes=128 << 20,
                                       max_sequences=4, max_pass_rows=2048))
    model.synthesize(st, shape, seed=5, norm_sigma=0.1)
    rng = np.random.default_rng(3)
    for rows in (223, 224, 385, 577, 769, 1025, 1300, 1537, 2048):
        ids = rng.integers(0, shape.vocab, rows).astype(np.uint64)
        out = []
        for config in (-1, 12):
            hp.say(shape.name, "rows", rows, "config", config)
            seq, previous = st.allocate(rows), capi.set_gemm_config(config)
            try:
                out.append(st.execute([capi.item(seq, rows, 0, sample=False)], token_ids=ids)["boundary"])
            finally:
                capi.set_gemm_config(previous)
            st.release(seq)
        hp.check_rows(oracle.f16_decode(out[0]), oracle.f16_decode(out[1]), (shape.name, rows))
    st.close()


def run(st, rows, ids, family, items):
    """The boundary rows or logits of a pass, and the kernels of one family of projections."""
    seqs = [st.allocate(rows // items) for _ in range(items)]
    st.profile(family)
    out = st.execute([capi.item(s, rows // items, 0, sample=items > 1) for s in seqs], token_ids=ids,
                     want_logits=items > 1)
    kernels = [r.partition("/")[2] for r in st.profile_records() if r.startswith(family + "/")]
    st.profile(None)
    for s in seqs:
        st.release(s)
    return out["logits"] if items > 1 else oracle.f16_decode(out["boundary"]), kernels


@pytest.mark.parametrize("hidden,intermediate,rows", [(4096, 1024, 224), (4096, 1024, 1024), (2048, 1536, 256),
                                                      (2560, 256, 385), (8192, 512, 224)])
def test_narrow_gate_up_splits_k(hidden, intermediate, rows):
    """Gate/up projections whose tiles are too few for the chip split K (they took up to four times as
    long unsplit), with the rows of unsplit 128-row tiles."""
    shape = synthetic.ModelShape(f"h{hidden}-i{intermediate}", 2, hidden, intermediate, 4, 2, 64, 300, eps=1e-6,
                                 theta=1e4, qk_norm=False, tied=False, max_seq=rows)
    st = capi.Stage(model.stage_config(shape, 0, 1, first=True, final=False, execution="f16", kv_cache_bytes=16 << 20,
                                       max_sequences=4, max_pass_rows=rows))
    model.synthesize(st, shape, seed=5, norm_sigma=0.1)
    ids = np.random.default_rng(3).integers(0, shape.vocab, rows).astype(np.uint64)
    hp.say(shape.name, "rows", rows)
    got, kernels = run(st, rows, ids, "gemm_gate_up", 1)
    assert any(k.startswith("gemm_reduce_kernel") for k in kernels), kernels
    previous = capi.set_gemm_config(15)
    try:
        expect, _ = run(st, rows, ids, "gemm_gate_up", 1)
    finally:
        capi.set_gemm_config(previous)
    hp.check_rows(got, expect, (shape.name, rows))
    st.close()


def test_head_over_a_small_vocabulary_splits_k():
    """As above for the LM head: 256 sampled rows over 2000 features."""
    shape = synthetic.ModelShape("v2000", 1, 2560, 96, 4, 2, 64, 2000, eps=1e-6, theta=1e4, qk_norm=False, tied=False,
                                 max_seq=64)
    st = capi.Stage(model.stage_config(shape, execution="f16", kv_cache_bytes=16 << 20, max_sequences=256,
                                       max_pass_rows=256))
    model.synthesize(st, shape, seed=5, norm_sigma=0.1)
    ids = np.random.default_rng(3).integers(0, shape.vocab, 256).astype(np.uint64)
    hp.say(shape.name, "rows", 256)
    got, kernels = run(st, 256, ids, "gemm_lm_head", 256)
    assert any(k.startswith("gemm_reduce_kernel") for k in kernels), kernels
    previous = capi.set_gemm_config(15)
    try:
        expect, _ = run(st, 256, ids, "gemm_lm_head", 256)
    finally:
        capi.set_gemm_config(previous)
    hp.check_rows(got, expect, shape.name)
    st.close()
