"""The feature projection's two products (hidden = embedding + feature . W, dW = feature^T . gradient)
through the training step, against the float64 oracle."""

import numpy as np
import pytest

import hip_harness as H
import kge_cases as K
from oracle.kge_oracle import make_cfg

pytestmark = pytest.mark.gpu


def _first_moments(oracle, c, feature_dtype, seed, emb_scale=None, all_distinct=False):
    """One step from zero moments: the first moments are the gradients times (1 - beta_m).  Returns the
    engine's and the oracle's state.  `all_distinct` (one shard): every head and tail a row of its own."""
    import libpoplar_kge

    rng = np.random.default_rng(seed)
    state = K.make_state(c, rng, warm=False)
    if emb_scale:
        state["entity_data"][:, :c["dim"]] *= emb_scale * np.sqrt(c["dim"])
    if feature_dtype == "bfloat16":
        state["entity_data"][:, 3 * c["dim"]:] = oracle.round(state["entity_data"][:, 3 * c["dim"]:], "bfloat16_embedding")
    batch = K.random_batch(c, 1, rng)
    if all_distinct:
        batch["head"][:] = np.arange(c["batch"])
        batch["a2a"][:] = c["batch"] + np.arange(c["a2a"])
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


def _small(dtype, F, D, rows):  # that many distinct rows, two of them tails
    return pytest.param(dtype, F, D, rows - 2, True, id=f"{dtype}-F{F}-D{D}-{rows}rows")


def _tall(dtype, F, D, batch):  # heads drawn with repeats: fewer distinct rows than the launches are sized for
    return pytest.param(dtype, F, D, batch, False, id=f"{dtype}-F{F}-D{D}-batch{batch}")


# Widths of two, four and eight waves (up to 64, 128, 256 columns) and of two workgroups; features that end in a
# slab of 32 or fill it up; rows around a tile of 32; features that take the loads a second round (all but the
# first line of either list: eight waves above 768 16-bit or 384 float32 features; fewer waves on tall
# tiles, four times as many chunks per thread, above 192 and 96).  Batches of 40k and 80k, 120k rows with four and
# two waves take tiles of 64 to 128 rows; eight waves take theirs by the distinct rows, 0.63 of a batch: 32, 64, 96 and 128
# for 10k, 20k, 30k and 40k, and for 25.5k 64 in more workgroups than the 128 of the batch itself (up to 8192 contributions
# in all there is nothing to choose); from 1152 rows on
# dW's contraction has more than eight parts.
@pytest.mark.parametrize("dtype,F,D,batch,all_distinct", [
    _small("float32", 4, 30, 31), _small("float16", 4, 66, 33), _small("bfloat16", 130, 66, 32), _small("float32", 36, 260, 33),
    _small("float16", 800, 130, 31), _small("float32", 388, 130, 33), _small("bfloat16", 800, 260, 65), _small("float32", 388, 256, 1200),
    _tall("float16", 36, 30, 40000), _tall("float32", 36, 30, 80000), _tall("float16", 228, 30, 120000),
    _tall("bfloat16", 36, 66, 20000), _tall("float16", 130, 66, 40000), _tall("float32", 132, 66, 60000),
    _tall("float32", 36, 130, 10000), _tall("bfloat16", 130, 130, 20000), _tall("float16", 36, 130, 30000), _tall("float32", 100, 260, 15000),
    _tall("float16", 36, 130, 25500), _tall("float16", 36, 130, 40000), _tall("float32", 36, 130, 40000),
    _tall("float16", 36, 130, 8190), _tall("float16", 36, 130, 8191),
])
def test_feature_shapes(oracle64, dtype, F, D, batch, all_distinct):
    c = K.cfg_dict(distance_fn="L2", n_shard=1, batch=batch, a2a=2, dim=D, feature=F, n_entity=batch + 5, n_relation=6, gamma=4.0)
    got, want = _first_moments(oracle64, c, dtype, 7, all_distinct=all_distinct)
    # A step's dozen roundings of 2^-24 and the contraction over the features (800: 3.1e-7 measured); and the two
    # tails' gradients, most of the norm on tall batches: one float32 sum over all positives, of 12 matrix
    # instructions per 32, whose N roundings (0.29 of 2^-24 each, at a partial sum that grows evenly)
    # add up to 0.29 / sqrt(3) 2^-24 sqrt(N): 2.1e-6 for 120000 positives.  Half as much again for the draw.
    bound = 5e-7 + 1.5 * 0.29 / np.sqrt(3) * 2.0**-24 * np.sqrt(12 * batch / 32)
    assert K.rel_l2(got["entity_data"][:, D:2 * D], want["entity_data"][:, D:2 * D]) < bound
    assert K.rel_l2(got["feature_projection/adam_m"], want["feature_projection/adam_m"]) < bound


# The loads of a row's last slab run on into the row behind it: nothing of that row may enter, a NaN included.
@pytest.mark.parametrize("dtype,F", [("float32", 4), ("float32", 36), ("float16", 8), ("float16", 40), ("bfloat16", 40)])
@pytest.mark.parametrize("D", [30, 66, 130])
def test_row_behind_stays_out(dtype, F, D):
    import libpoplar_kge

    c = K.cfg_dict(distance_fn="L2", n_shard=1, batch=40, a2a=2, dim=D, feature=F, n_entity=300, n_relation=6, gamma=4.0)
    rng = np.random.default_rng(3)
    state, batch = K.make_state(c, rng, warm=False), K.random_batch(c, 1, rng)
    used = np.unique(batch["remote"])
    unused = np.setdiff1d(np.arange(c["n_entity"]), used)
    assert np.isin(used + 1, unused).any()
    after = []
    for value in (0.0, np.nan):
        start = K.copy_state(state)
        start["entity_data"][unused] = value
        engine = libpoplar_kge.Engine(H.engine_settings(c, 1, **{"execution.feature_dtype": dtype}), "")
        H.load_state(engine, c, start)
        loss = H.train(engine, c, np.full(1, 1e-3, np.float32), batch)
        got = H.read_state(engine, c)
        after.append((loss, got["entity_data"][used], got["feature_projection/adam_m"], got["relation_embedding"]))
    for clean, beside in zip(*after):
        assert np.isfinite(clean).all()
        np.testing.assert_array_equal(clean, beside)
