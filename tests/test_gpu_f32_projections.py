"""F32 execution of 65 rows and more: which tiles the projections take, by the bytes of the resident
weights (F16 or F32), and their results against the 64-row activation-staged tiles
(checked against the oracle by the configuration tests).

Boundary rows within 5e-4 + 2^-10 |ref|. Both sides are F32 sums of 22-bit products in another order:
the layer's F32 output (rms about 1) under any two of the 16-, 32-, 64- and 128-row tiles differs by
1e-5 rms and 3.1e-4 at most on the largest of these shapes, because the input norm scales embedding
rows of rms 0.02, and with them their rounding, up fifty times; the second term is the F16 unit in the
last place by which a value next to a rounding boundary then moves."""
import numpy as np
import pytest

import oracle
from hllm_amd import capi, model, synthetic
from tests import helpers_parity as hp

pytestmark = pytest.mark.gpu
SMALL, STAGED64 = "gemm_kernel<1, 4, 1, 1, 4, 4, ", "gemm_xlds_kernel<4, 4, 8, 4, "
STAGED32, STAGED128 = "gemm_xlds_kernel<2, 4, 4, 4, ", "gemm_xlds_kernel<8, 4, 4, 2, "


def tiles_and_rows(weights, hidden, intermediate, heads, rows, families):
    """{family: its kernels} of the choice by shape, after comparing the rows with 64-row tiles."""
    shape = synthetic.ModelShape(f"h{hidden}-i{intermediate}", 2, hidden, intermediate, heads, heads // 2, 128, 300,
                                 eps=1e-6, theta=1e4, qk_norm=False, tied=False, max_seq=rows)
    st = capi.Stage(model.stage_config(shape, 0, 1, first=True, final=False, execution="f32", weights=weights,
                                       kv_cache_bytes=64 << 20, max_sequences=4, max_pass_rows=rows))
    model.synthesize(st, shape, seed=5, norm_sigma=0.1)
    ids = np.random.default_rng(3).integers(0, shape.vocab, rows).astype(np.uint64)
    out = []
    for config in (-1, 12):
        hp.say(shape.name, weights, "rows", rows, "config", config)
        seq, previous = st.allocate(rows), capi.set_gemm_config(config)
        try:
            st.profile("gemm")
            out.append(oracle.f16_decode(st.execute([capi.item(seq, rows, 0, sample=False)], token_ids=ids)["boundary"]))
            records = [r.split("/") for r in st.profile_records() if "/" in r]
            st.profile(None)
        finally:
            capi.set_gemm_config(previous)
        st.release(seq)
        if config < 0:
            kernels = {f: [k for family, k in records if family == f] for f in families}
    st.close()
    error = np.abs(out[0] - out[1])
    hp.say(shape.name, weights, "rows", rows, f"max-abs {error.max():.1e}")
    assert (error <= 5e-4 + 2.0 ** -10 * np.abs(out[1])).all(), error.max()
    return kernels


@pytest.mark.parametrize("weights,rows,tile", [("f16", 223, SMALL), ("f32", 192, SMALL), ("f32", 223, STAGED64)])
def test_tiles_by_resident_bytes(weights, rows, tile):
    """q/k/v of 223 rows: 117 MB of repeated weight reads as F16, 235 MB as F32 (201 MB at 192 rows);
    o: half of each. The 16-row tiles win up to 120 MB of F16 and 205 MB of F32 weights."""
    kernels = tiles_and_rows(weights, 1024, 256, 16, rows, ("gemm_qkv", "gemm_o"))
    assert any(k.startswith(tile) for k in kernels["gemm_qkv"]), kernels
    assert any(k.startswith(SMALL) for k in kernels["gemm_o"]), kernels


@pytest.mark.parametrize("weights,hidden,intermediate,heads,rows,gate_up,down", [
    ("f32", 2560, 9728, 32, 384, STAGED128, STAGED128),   # three whole 128-row tiles
    ("f32", 2560, 9728, 32, 1024, STAGED128, STAGED128),
    ("f16", 2560, 9728, 32, 512, STAGED32, STAGED32),
    ("f16", 4096, 1024, 32, 224, "gemm_reduce_kernel", ""),  # narrow and deep: a K split
    ("f32", 4096, 1024, 32, 512, "gemm_reduce_kernel", "")])
def test_tiles_by_estimated_time(weights, hidden, intermediate, heads, rows, gate_up, down):
    """224 to 1024 rows: 32-row tiles alone were up to 2.3 times slower than 64- or 128-row ones."""
    kernels = tiles_and_rows(weights, hidden, intermediate, heads, rows, ("gemm_gate_up", "gemm_down"))
    assert any(k.startswith(gate_up) for k in kernels["gemm_gate_up"]), kernels
    assert any(k.startswith(down) for k in kernels["gemm_down"]), kernels


@pytest.mark.parametrize("weights,rows,tile", [("f16", 223, STAGED128), ("f32", 223, STAGED128), ("f16", 33, SMALL),
                                               ("f32", 33, STAGED64)])
def test_wide_head(weights, rows, tile):
    """223 rows: 130 tiles of 128 rows, unsplit (splits would take a second round of workgroups); 33
    rows: the 16-row tiles with F16-resident weights only."""
    shape = synthetic.ModelShape("v16500", 1, 1024, 64, 4, 2, 64, 16500, eps=1e-6, theta=1e4, qk_norm=False, tied=False,
                                 max_seq=64)
    st = capi.Stage(model.stage_config(shape, execution="f32", weights=weights, kv_cache_bytes=64 << 20,
                                       max_sequences=rows, max_pass_rows=256))
    model.synthesize(st, shape, seed=5, norm_sigma=0.1)
    ids = np.random.default_rng(3).integers(0, shape.vocab, rows).astype(np.uint64)
    logits = []
    for config in (-1, 12):
        hp.say(shape.name, weights, "config", config)
        seqs, previous = [st.allocate(1) for _ in ids], capi.set_gemm_config(config)
        try:
            st.profile("gemm_lm_head")
            logits.append(st.execute([capi.item(s, 1, 0) for s in seqs], token_ids=ids, want_logits=True)["logits"])
            kernels = [r.partition("/")[2] for r in st.profile_records() if r.startswith("gemm_lm_head/")]
            st.profile(None)
        finally:
            capi.set_gemm_config(previous)
        for s in seqs:
            st.release(s)
        if config < 0:
            assert any(k.startswith(tile) for k in kernels) and (rows < 193 or len(kernels) == 1), kernels
    st.close()
    # F32 logits, the suite's bound for another order of summation.
    assert (np.abs(logits[0] - logits[1]) <= 2e-4 + 1e-4 * np.abs(logits[1])).all()
