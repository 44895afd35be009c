"""Gate/up projections of up to 128 rows (the pair kernel, and the decode kernel on wide outputs)
and the boundary encoding that sums the last down projection's K-split partials, against the
oracle at their edges: k-steps fewer than the waves, not a multiple of them and past one ring of
every row tile count (544 columns: four or five k-steps per wave of the pair kernel, three chunks of
the decode kernel's six and eight row tiles); an odd number of 32-feature groups; workgroups of one
pair and of two (more pairs than CUs); 1 to 128 rows around the 16-row tiles; row lengths that divide
by four and that do not, both with partials for the boundary (66 columns from 1600: five).

A one-layer first stage returns its boundary rows. Bounds per row as for the other F16 slices
(max-abs 2e-2, cosine 0.9999)."""
import numpy as np
import pytest

import oracle
from hllm_amd import capi, model, synthetic
from tests import helpers_parity as hp
from tests import models

pytestmark = pytest.mark.gpu
ROWS = (1, 15, 16, 17, 31, 33, 48, 49, 64, 65, 81, 96, 97, 128)


@pytest.mark.parametrize("hidden,intermediate", [(64, 32), (66, 96), (96, 160), (160, 4128), (544, 288), (64, 8224),
                                                 (66, 1600), (544, 4128), (544, 8224)])
def test_gate_up_and_boundary_match_the_oracle(hidden, intermediate):
    shape = synthetic.ModelShape(f"h{hidden}-i{intermediate}", 2, hidden, intermediate, 4, 2, 64, 300, eps=1e-6,
                                 theta=1e4, qk_norm=False, tied=False, max_seq=128)
    st = capi.Stage(model.stage_config(shape, 0, 1, first=True, final=False, execution="f16", kv_cache_bytes=16 << 20,
                                       max_sequences=4, max_pass_rows=128))
    model.synthesize(st, shape, seed=5, norm_sigma=0.1)
    ost = oracle.OracleStage(models.synthetic_stage(shape, 0, 1, first=True, final=False, seed=5, norm_sigma=0.1))
    rng = np.random.default_rng(3)
    for rows in ROWS:
        hp.say(shape.name, "rows", rows)
        ids = rng.integers(0, shape.vocab, rows).astype(np.uint64)
        seq, oseq = st.allocate(rows), ost.allocate_sequence(rows)
        got = st.execute([capi.item(seq, rows, 0, sample=False)], token_ids=ids)["boundary"]
        kind, expect = ost.execute(ids, 0, oseq)[:2]
        assert kind == "boundary"
        hp.check_rows(oracle.f16_decode(got), oracle.f16_decode(expect), (shape.name, rows))
        st.release(seq)
    st.close()


def gate_up_kernel(hidden, intermediate, rows):
    """The kernel that starts gate/up of one layer, after comparing its rows with 64-row staged tiles."""
    shape = synthetic.ModelShape(f"h{hidden}-i{intermediate}", 2, hidden, intermediate, 4, 2, 64, 300, eps=1e-6,
                                 theta=1e4, qk_norm=False, tied=False, max_seq=128)
    st = capi.Stage(model.stage_config(shape, 0, 1, first=True, final=False, execution="f16", kv_cache_bytes=16 << 20,
                                       max_sequences=4, max_pass_rows=128))
    model.synthesize(st, shape, seed=5, norm_sigma=0.1)
    ids = np.random.default_rng(3).integers(0, shape.vocab, rows).astype(np.uint64)
    out, kernels = [], []
    for config in (-1, 12):
        hp.say(shape.name, "rows", rows, "config", config)
        seq, previous = st.allocate(rows), capi.set_gemm_config(config)
        try:
            st.profile("gemm_gate_up")
            out.append(st.execute([capi.item(seq, rows, 0, sample=False)], token_ids=ids)["boundary"])
            kernels.append([r.partition("/")[2] for r in st.profile_records() if r.startswith("gemm_gate_up/")])
            st.profile(None)
        finally:
            capi.set_gemm_config(previous)
        st.release(seq)
    st.close()
    hp.check_rows(oracle.f16_decode(out[0]), oracle.f16_decode(out[1]), (shape.name, rows))
    return kernels[0]


@pytest.mark.parametrize("hidden,intermediate,rows,kernel", [
    (8192, 512, 64, "gemm_pair_kernel"), (8192, 512, 65, "gemm_xlds_kernel"), (4096, 1024, 128, "gemm_xlds_kernel"),
    (4096, 2048, 128, "gemm_pair_kernel"), (3072, 256, 128, "gemm_pair_kernel")])
def test_narrow_gate_up_of_a_long_k_above_64_rows(hidden, intermediate, rows, kernel):
    """The pair kernel up to 128 rows only where it beats the staged tiles' K splits."""
    kernels = gate_up_kernel(hidden, intermediate, rows)
    assert any(k.startswith(kernel) for k in kernels), kernels


@pytest.mark.parametrize("hidden,intermediate,rows,kernel", [
    (512, 18432, 96, "gemm_decode_kernel"), (512, 18432, 97, "gemm_xlds_kernel"), (2080, 16416, 96, "gemm_decode_kernel"),
    (2080, 16416, 128, "gemm_xlds_kernel"), (512, 16384, 128, "gemm_decode_kernel")])
def test_wide_gate_up_of_a_short_k_above_96_rows(hidden, intermediate, rows, kernel):
    """The decode kernel's eight row tiles only in one round of workgroups, or with a long K."""
    kernels = gate_up_kernel(hidden, intermediate, rows)
    assert any(k.startswith(kernel) for k in kernels), kernels
