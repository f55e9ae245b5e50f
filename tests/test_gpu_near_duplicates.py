"""Near-duplicate samples, generalized: every FP32 entry within 1e-6 of the FP64 oracle,
with no need of the reference's build."""
import pytest

from conftest import rel_err
from test_gpu_parity import inputs_from, near_duplicate_table, oracle_matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("alpha", [0.5, 0.3, 1.0])
def test_generalized_near_duplicates_against_the_oracle(ssu, O, synth, alpha):
    if not ssu.device_available():
        pytest.fail("no HIP device visible: the HIP path cannot run (no CPU fallback exists)")
    tree, table = near_duplicate_table(synth)
    s, m = ssu.matrix_inmem(inputs_from(ssu, tree, table), "generalized", alpha=alpha)
    assert s == ssu.OKAY, ssu.last_error()
    err = rel_err(m, oracle_matrix(O, tree, table, "generalized", alpha=alpha))
    print("[gpu-case] generalized near duplicates", alpha, "max rel err", err, flush=True)
    assert err <= 1e-6
