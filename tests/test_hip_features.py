"""The feature projection's two products (hidden = embedding + feature . W, dW = feature^T . gradient)
through the training step, against the float64 oracle."""

import numpy as np
import pytest

import hip_harness as H
import kge_cases as K
from oracle.kge_oracle import make_cfg

pytestmark = pytest.mark.gpu


def _first_moments(oracle, c, feature_dtype, seed, emb_scale=None):
    """One step from zero moments: the first moments are the gradients times (1 - beta_m).  Returns the
    engine's and the oracle's state."""
    import libpoplar_kge

    rng = np.random.default_rng(seed)
    state = K.make_state(c, rng, warm=False)
    if emb_scale:
        state["entity_data"][:, :c["dim"]] *= emb_scale * np.sqrt(c["dim"])
    if feature_dtype == "bfloat16":
        state["entity_data"][:, 3 * c["dim"]:] = oracle.round(state["entity_data"][:, 3 * c["dim"]:], "bfloat16_embedding")
    batch = K.random_batch(c, 1, rng)
    lr = np.full(c["n_shard"], 1e-3, np.float32)
    engine = libpoplar_kge.Engine(H.engine_settings(c, 1, **{"execution.feature_dtype": feature_dtype}), "")
    H.load_state(engine, c, state)
    loss = H.train(engine, c, lr, batch)
    got, want = H.read_state(engine, c), K.copy_state(state)
    np.testing.assert_allclose(loss, oracle.train_step_loop(make_cfg(**c), want, lr, batch), rtol=1e-6)
    return got, want


@pytest.mark.parametrize("feature_dtype", ["float32", "float16"])
def test_embeddings_larger_than_the_projection(oracle64, feature_dtype):
    """The embedding is added to the finished product: the hidden rows round at its size once (2^-24 / sqrt 3
    of it), which with the predicted tail's, the coefficients' and the sums' few roundings makes 1.3e-7
    of the gradients (measured; 4.6e-7 when all 240 instructions of a contraction over 768 features
    rounded at that size, as they do if the accumulators start from the embedding)."""
    c = K.cfg_dict(distance_fn="L2", n_shard=2, batch=64, a2a=32, dim=256, feature=768, n_entity=600, n_relation=6, gamma=4.0)
    got, want = _first_moments(oracle64, c, feature_dtype, 5, emb_scale=3.0)
    D = c["dim"]
    assert K.rel_l2(got["entity_data"][:, D:2 * D], want["entity_data"][:, D:2 * D]) < 2.5e-7
    # dW over 256 rows: the gradient's own error, and one rounding of the large terms per sixteen rows (1.5e-7;
    # 1.95e-7 when the small terms round into the same sum)
    assert K.rel_l2(got["feature_projection/adam_m"], want["feature_projection/adam_m"]) < 1.75e-7
