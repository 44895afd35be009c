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
