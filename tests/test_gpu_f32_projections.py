"""F32 execution of 65 rows and more: which tiles the projections take, by the bytes of the resident
weights (F16 or F32), and their results against the 64-row activation-staged tiles
(checked against the oracle by the configuration tests).

Boundary rows within 2e-5 + 2^-10 |ref|: both sides are F32 sums of 22-bit products in another order
(2e-5 covers a layer's sums of order one over at most 8192 terms), so a value next to a rounding
boundary moves by one F16 unit in the last place, at most 2^-10 of it."""
import numpy as np
import pytest

import oracle
from hllm_amd import capi, model, synthetic
from tests import helpers_parity as hp

pytestmark = pytest.mark.gpu
SMALL, STAGED64 = "gemm_kernel<1, 4, 1, 1, 4, 4, ", "gemm_xlds_kernel<4, 4, 8, 4, "


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
    assert (error <= 2e-5 + 2.0 ** -10 * np.abs(out[1])).all(), error.max()
    return kernels


@pytest.mark.parametrize("weights,rows,tile", [("f16", 223, SMALL), ("f32", 192, SMALL), ("f32", 223, STAGED64)])
def test_tiles_by_resident_bytes(weights, rows, tile):
    """q/k/v of 223 rows: 117 MB of repeated weight reads as F16, 235 MB as F32 (201 MB at 192 rows);
    o: half of each. The 16-row tiles win up to 120 MB of F16 and 205 MB of F32 weights."""
    kernels = tiles_and_rows(weights, 1024, 256, 16, rows, ("gemm_qkv", "gemm_o"))
    assert any(k.startswith(tile) for k in kernels["gemm_qkv"]), kernels
    assert any(k.startswith(SMALL) for k in kernels["gemm_o"]), kernels
