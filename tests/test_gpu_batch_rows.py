"""A decode row's result does not depend on the rows beside it: the same sequence alone (folded
norms), with one more, and among 17, 33 and 64 rows gives the same boundary bits, on layers whose
gate/up runs on the pair kernel and on the decode kernel."""
import numpy as np
import pytest

from hllm_amd import capi, model, synthetic
from tests import helpers_parity as hp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,intermediate", [(1024, 3072), (2080, 352), (3072, 9216), (544, 4128)])
def test_rows_are_independent(hidden, intermediate):
    shape = synthetic.ModelShape(f"h{hidden}", 3, hidden, intermediate, 8, 4, 128, 300, eps=1e-6, theta=1e4,
                                 qk_norm=True, tied=False, max_seq=64)
    st = capi.Stage(model.stage_config(shape, 0, 2, first=True, final=False, execution="f16",
                                       kv_cache_bytes=128 << 20, max_sequences=64, max_pass_rows=64))
    model.synthesize(st, shape, seed=5, norm_sigma=0.1)
    ids = np.random.default_rng(3).integers(0, shape.vocab, 64).astype(np.uint64)
    ref = None
    for rows in (64, 33, 17, 2, 1):
        hp.say(shape.name, "rows", rows)
        seqs = [st.allocate(1) for _ in range(rows)]
        out = st.execute([capi.item(s, 1, 0, sample=False) for s in seqs], token_ids=ids[:rows])["boundary"]
        ref = out if ref is None else ref
        assert np.array_equal(out, ref[:rows]), (shape.name, rows)
        for s in seqs:
            st.release(s)
    st.close()
