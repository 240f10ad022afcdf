"""The scoring kernels away from whole tiles, against the float64 oracle through the training step:
sizes around the edges of tiles and groups, one row, splits of a side over several workgroups."""

import ctypes as C

import hip_harness as H
import kge_cases as K
import numpy as np
import pytest

from test_hip_step import run_case

pytestmark = pytest.mark.gpu


# (shards, positives, tails per shard pair, dim).  L1 backward: groups of at most 512 tails shared
# evenly in steps of 32, groups of heads in steps of 8, slices of 64 columns; a split side's sums
# come in pieces.
@pytest.mark.parametrize("merge", [True, False])
@pytest.mark.parametrize("S,B,A,D", [
    (1, 1, 2, 1),        # one head, two tails, one column
    (1, 7, 33, 63),      # below a chunk of heads, a tail over 32, below a slice
    (1, 129, 257, 65),   # both sides split; one over every edge
    (2, 64, 320, 68),    # 640 tails: over one group
    (1, 600, 128, 64),   # heads split eight ways and more, whole chunks
    (1, 264, 513, 32),   # a tail over a group, a chunk over 256 heads
    (16, 12, 96, 64),    # 1536 tails per block in four groups
])
def test_l1_shapes(oracle64, S, B, A, D, merge):
    run_case(oracle64, dict(distance_fn="L1", n_shard=S, batch=B, a2a=A, dim=D, feature=0, n_entity=4000,
                            n_relation=16, gamma=4.0), n_step=2, **{"execution.merge_tails": merge})


# L1 backward without bounds checks (tails in steps of 32, heads of 8, columns of 64): tails per wave that are
# and are not a multiple of four, one chunk of heads and several
@pytest.mark.parametrize("B,A,D", [(8, 32, 64), (16, 96, 128), (24, 160, 64), (64, 352, 64), (8, 512, 64), (264, 544, 64)])
def test_l1_whole_groups(oracle64, B, A, D):
    run_case(oracle64, dict(distance_fn="L1", n_shard=1, batch=B, a2a=A, dim=D, feature=0, n_entity=4000, n_relation=16,
                            gamma=4.0), n_step=2, **{"execution.merge_tails": False})


# L1 backward with bounds checks, one group of 512, 480, 448 and 416 tails: 32, 30, 28 and 26 per wave, whose heads'
# values are asked for two, four, four and eight heads ahead
@pytest.mark.parametrize("S,B,A,D", [(64, 9, 8, 200), (32, 19, 15, 452), (64, 12, 7, 250), (32, 9, 13, 450)])
def test_l1_wide_groups(oracle64, S, B, A, D):
    run_case(oracle64, dict(distance_fn="L1", n_shard=S, batch=B, a2a=A, dim=D, feature=0, n_entity=1500, n_relation=S,
                            gamma=4.0), n_step=1, **{"execution.merge_tails": False})


# the same with 4, 8, 10 and 16 tails per wave: one, one, two and two columns of coefficients per lane
@pytest.mark.parametrize("S,B,A,D", [(50, 9, 1, 250), (50, 17, 2, 250), (50, 9, 3, 250), (50, 8, 5, 250)])
def test_l1_narrow_groups(oracle64, S, B, A, D):
    run_case(oracle64, dict(distance_fn="L1", n_shard=S, batch=B, a2a=A, dim=D, feature=0, n_entity=1000, n_relation=S,
                            gamma=4.0), n_step=1, **{"execution.merge_tails": False})


# L1 forward: tiles of 64 heads x 32 tails, four waves over slabs of eight columns (from 64 columns on): around a tile's
# edges, a last slab of four columns, waves with and without one
@pytest.mark.parametrize("merge", [True, False])
@pytest.mark.parametrize("loss_fn", ["logsigmoid", "softmax"])
@pytest.mark.parametrize("S,B,A,D", [(1, 1, 2, 64), (1, 63, 31, 68), (2, 64, 16, 72), (1, 65, 33, 100), (3, 130, 43, 260), (1, 8, 96, 128)])
def test_l1_forward_tiles(oracle64, loss_fn, S, B, A, D, merge):
    run_case(oracle64, dict(distance_fn="L1", loss_fn=loss_fn, n_shard=S, batch=B, a2a=A, dim=D, feature=0, n_entity=1500,
                            n_relation=6, gamma=4.0), n_step=2, **{"execution.merge_tails": merge})


# Merged tails: limits are whole groups of 64 columns, the L1 forward's tiles are 32 wide, so the last 32 columns in front of
# a limit can lie behind the distinct tails.  The forward leaves zeros there; the vector backward, a launch per side, adds
# them up.  Fewer distinct tails from step to step: what the step before left there would show.
@pytest.mark.parametrize("B,T,D", [(70, 192, 64), (33, 180, 100)])
def test_l1_dead_columns_in_front_of_the_limit(oracle64, B, T, D):
    counts = [(T, T - 1), (160, 129), (96, 70), (32, 20)]  # distinct tails of the two blocks, step by step

    def batch_fn(c, n_step, rng):
        batch = K.raw_batch(c, n_step, rng, zipf=False)
        for step in range(n_step):
            for d in range(2):
                pool = rng.choice(np.arange(1, c["n_entity"]), counts[step][d], replace=False).astype(np.uint32)
                rows = np.concatenate([pool, pool[rng.integers(0, len(pool), T - len(pool))]])
                rng.shuffle(rows)
                # block d's tails: slots B + d A .. + A - 1 of either source shard's `remote`
                batch["remote"][:, step, B + d * T // 2:B + (d + 1) * T // 2] = rows.reshape(2, T // 2)
        return batch

    run_case(oracle64, dict(distance_fn="L1", n_shard=2, batch=B, a2a=T // 2, dim=D, feature=0, n_entity=1500, n_relation=6,
                            gamma=4.0, shared_table=True), n_step=4, batch_fn=batch_fn, **{"execution.scoring": "valu"})


# L1 forward in tiles of 64 x 64 over slabs of 32 columns: below 64 columns, and where short loops meet 2048 tiles or more
# (64 columns with merged tails, up to 160 without).  Fused, that takes whole tiles and the next slab's loads are in flight.
# (Softmax: where the head's rounding to float32 turns a difference's sign, a term of the gradient turns with it; the sequential
# float32 oracle is 2e-6 and 3e-6 off the float64 one here, and 1.1e-5, over the bar, with 510 positives, 512 tails and D = 128.)
@pytest.mark.parametrize("loss_fn,S,B,A,D,merge", [
    ("logsigmoid", 2, 64, 64, 32, True), ("logsigmoid", 1, 128, 64, 32, False), ("logsigmoid", 32, 256, 32, 64, True),
    ("logsigmoid", 32, 512, 16, 96, False), ("softmax", 32, 250, 32, 64, True), ("softmax", 32, 250, 32, 96, False),
])
def test_l1_forward_square_tiles(oracle64, loss_fn, S, B, A, D, merge):
    run_case(oracle64, dict(distance_fn="L1", loss_fn=loss_fn, n_shard=S, batch=B, a2a=A, dim=D, feature=0, n_entity=2000,
                            n_relation=S, gamma=4.0), n_step=1, **{"execution.merge_tails": merge})


# Columns in which every head equals every tail have signum 0 throughout: their gradients are exactly zero
@pytest.mark.parametrize("B,A,D", [(33, 90, 30), (64, 352, 64)])
def test_l1_equal_columns_have_zero_gradient(B, A, D):
    import libpoplar_kge

    c = K.cfg_dict(distance_fn="L1", n_shard=1, batch=B, a2a=A, dim=D, feature=0, n_entity=2000, n_relation=9, gamma=4.0)
    rng = np.random.default_rng(5)
    state = K.make_state(c, rng, warm=False)
    equal = np.arange(0, D, 3)
    state["entity_data"][:, equal] = 0.25
    state["relation_embedding"][:, equal] = 0.0
    engine = libpoplar_kge.Engine(H.engine_settings(c, 2, **{"execution.merge_tails": False}), "")
    H.load_state(engine, c, state)
    H.train(engine, c, 0.1, K.random_batch(c, 2, rng))
    after = H.read_state(engine, c)
    np.testing.assert_array_equal(after["entity_data"][:, equal], state["entity_data"][:, equal])
    np.testing.assert_array_equal(after["relation_embedding"][:, equal], state["relation_embedding"][:, equal])
    np.testing.assert_array_equal(after["entity_data"][:, D + equal], 0.0)


# L2 and dot on float16 halves: tiles of 64 x 64 over slabs of 32, matrices filled up to 32
@pytest.mark.parametrize("merge", [True, False])
@pytest.mark.parametrize("score_fn,distance_fn", [("TransE", "L2"), ("DistMult", "MatMul"), ("ComplEx", "L2")])
@pytest.mark.parametrize("loss_fn", ["logsigmoid", "softmax"])
@pytest.mark.parametrize("S,B,A,D", [
    (1, 1, 2, 2),         # one pair of rows and two columns
    (1, 31, 33, 30),      # around one 32 x 32 sub-block
    (2, 64, 32, 32),      # exactly a tile, exactly a slab
    (1, 65, 97, 66),      # one over a tile, a sub-block and two slabs
    (3, 130, 43, 100),    # several tiles, none of them whole
    (2, 128, 64, 64),     # whole tiles, few of them
])
def test_l2_and_dot_shapes(oracle64, score_fn, distance_fn, loss_fn, S, B, A, D, merge):
    run_case(oracle64, dict(score_fn=score_fn, distance_fn=distance_fn, loss_fn=loss_fn, n_shard=S, batch=B, a2a=A, dim=D,
                            feature=0, n_entity=1500, n_relation=6, gamma=4.0), n_step=2, **{"execution.merge_tails": merge})


def _first_moments(c, state, batch, loss_scale, oracle64, **extra):
    """One step from moments of zero: (engine, oracle) x (the loss, the entities' first moments, the relations'), which are
    the gradients times 1 - beta_m."""
    import libpoplar_kge
    from oracle.kge_oracle import make_cfg

    c = dict(c, loss_scale=float(loss_scale))
    lr = np.full(c["n_shard"], 0.01, np.float32)
    engine = libpoplar_kge.Engine(H.engine_settings(c, 1, **extra), "")
    H.load_state(engine, c, state)
    loss = H.train(engine, c, lr, batch)
    got, want = H.read_state(engine, c), K.copy_state(state)
    want_loss = oracle64.train_step_loop(make_cfg(**c), want, lr, batch)
    D = c["dim"]
    return [(l, s["entity_data"][:, D:2 * D].astype(np.float64), s["relation_embedding/adam_m"].astype(np.float64))
            for l, s in ((loss, got), (want_loss, want))]


def _assert_each_row(got, want, rel=1e-5):
    """1e-5, the bar of every float32 gradient here, of the whole and of every row by its own norm (and 2^-126, float32's
    smallest normal number: what lies below has fewer bits, as a softmax's e^-87 has)."""
    np.testing.assert_allclose(got[0], want[0], rtol=rel)
    for g, w in zip(got[1:], want[1:]):
        assert K.rel_l2(g, w) < rel
        norm, error = np.linalg.norm(w, axis=1), np.linalg.norm(g - w, axis=1)
        bar = rel * norm + 2.0**-126
        worst = np.argmax(error - bar)
        assert error[worst] <= bar[worst], (worst, error[worst], norm[worst])


@pytest.mark.parametrize("score_fn,distance_fn", [("TransE", "L2"), ("DistMult", "MatMul")])
@pytest.mark.parametrize("loss_fn", ["logsigmoid", "softmax"])
@pytest.mark.parametrize("S,B,A,D", [
    (1, 40, 2080, 260),    # more than 64 slabs of tails, rows of more than 256 columns
    (1, 2100, 40, 36),     # more than 64 slabs of heads
    (64, 129, 9, 66),      # tiles of 128 x 64, none of them whole
])
def test_halves_of_rows_of_many_sizes(oracle64, score_fn, distance_fn, loss_fn, S, B, A, D):
    """Rows whose lengths are spread over a factor of a thousand and more, so that the scales of rows and of sub-blocks of
    coefficients differ from one to the next."""
    c = K.cfg_dict(score_fn=score_fn, distance_fn=distance_fn, loss_fn=loss_fn, n_shard=S, batch=B, a2a=A, dim=D, feature=0,
                   n_entity=3000, n_relation=6, gamma=4.0, shared_table=True)
    rng = np.random.default_rng(S + B)
    state = K.make_state(c, rng, warm=False)
    state["entity_data"][:, :D] *= np.exp(rng.normal(0, 1.5, (c["n_entity"], 1))).astype(np.float32)
    _assert_each_row(*_first_moments(c, state, K.raw_batch(c, 1, rng), c["loss_scale"], oracle64))


# Coefficients times the scales of their rows far below 1 (a small initialisation, a loss scale that is not the default
# one): no slab of them may be left out of the sums
@pytest.mark.parametrize("score_fn,distance_fn", [("TransE", "L2"), ("DistMult", "MatMul"), ("ComplEx", "MatMul")])
@pytest.mark.parametrize("loss_fn", ["logsigmoid", "softmax"])
@pytest.mark.parametrize("S,B,A,D,sigma,loss_scale", [
    (64, 256, 8, 256, 1 / 256, 1),
    (16, 512, 96, 128, 1 / 128, 1),
    (4, 200, 64, 100, 1e-3, 1),
    (4, 200, 64, 100, 1e-4, 2.0**-12),
])
def test_small_coefficients_reach_the_gradient(oracle64, score_fn, distance_fn, loss_fn, S, B, A, D, sigma, loss_scale):
    c = K.cfg_dict(score_fn=score_fn, distance_fn=distance_fn, loss_fn=loss_fn, n_shard=S, batch=B, a2a=A, dim=D, feature=0,
                   n_entity=3000, n_relation=S * 6, gamma=4.0, shared_table=True)
    rng = np.random.default_rng(7)
    state = K.make_state(c, rng, warm=False, scale=sigma)
    _assert_each_row(*_first_moments(c, state, K.raw_batch(c, 1, rng), loss_scale, oracle64))


def _one_block(c, state, sizes, rng):
    """One block whose heads, and then tails in their slots' order, are rows 1 .. with standard deviations `sizes`
    ([B + A]); relations of size 1 of their own."""
    B, A, D = c["batch"], c["a2a"], c["dim"]
    state["entity_data"][1:1 + B + A, :D] = rng.normal(0, 1, (B + A, D)) * np.asarray(sizes)[:, None]
    return dict(remote=(1 + np.arange(B + A, dtype=np.uint32)).reshape(1, 1, B + A),
                a2a=(B + np.arange(A, dtype=np.uint32)).reshape(1, 1, 1, A), head=np.arange(B, dtype=np.uint32).reshape(1, 1, B),
                relation=np.arange(B, dtype=np.uint32).reshape(1, 1, B), tail=rng.integers(0, A, (1, 1, B)).astype(np.uint32))


# The first slab of heads and of tails is sixteen times shorter than the others: whatever the loss scale, it counts
@pytest.mark.parametrize("power", range(-40, 41, 4))
def test_short_first_slab_counts(oracle64, power):
    B, A, D = 96, 96, 64
    c = K.cfg_dict(score_fn="DistMult", distance_fn="MatMul", n_shard=1, batch=B, a2a=A, dim=D, feature=0, n_entity=300,
                   n_relation=B, gamma=4.0, shared_table=True)
    rng = np.random.default_rng(7)
    state = K.make_state(c, rng, warm=False, scale=2.0**-3)
    sizes = np.where(np.arange(B + A) % 96 < 32, 2.0**-7, 2.0**-3)
    batch = _one_block(c, state, sizes, rng)
    _assert_each_row(*_first_moments(c, state, batch, 2.0**power, oracle64, **{"execution.merge_tails": False}))


# Rows of zeros, one head and one tail, among others of one size: their gradients are as right as their neighbours'
@pytest.mark.parametrize("score_fn,distance_fn,loss_fn,sigma", [
    ("TransE", "L2", "logsigmoid", 1 / 16), ("TransE", "L2", "logsigmoid", 1), ("TransE", "L2", "logsigmoid", 64),
    ("TransE", "L2", "softmax", 1 / 16), ("DistMult", "MatMul", "logsigmoid", 1 / 16), ("DistMult", "MatMul", "logsigmoid", 1),
    ("DistMult", "MatMul", "logsigmoid", 64), ("DistMult", "MatMul", "softmax", 1), ("DistMult", "MatMul", "softmax", 64),
])
def test_rows_of_zeros(oracle64, score_fn, distance_fn, loss_fn, sigma):
    B, A, D = 70, 100, 64
    c = K.cfg_dict(score_fn=score_fn, distance_fn=distance_fn, loss_fn=loss_fn, n_shard=1, batch=B, a2a=A, dim=D, feature=0,
                   n_entity=300, n_relation=B, gamma=4.0, shared_table=True)
    rng = np.random.default_rng(7)
    state = K.make_state(c, rng, warm=False, scale=sigma)
    sizes = np.full(B + A, float(sigma))
    sizes[[3, B + 37]] = 0.0
    if score_fn == "DistMult":  # (scores of a few units)
        state["relation_embedding"] *= sigma**-3 / 4
    else:
        state["relation_embedding"][3] = 0.0
    _assert_each_row(*_first_moments(c, state, _one_block(c, state, sizes, rng), B * A, oracle64))


# One head and one tail much smaller or larger than the others (2^power), or rows of all sizes beside one another (None).
# L2 to 2^-50 only (below 2^-60 the square of the distance between the two leaves float32's range), and no softmax of distances
# between rows of all sizes (the sequential float32 oracle is 4e-4 and 2e-3 off the float64 one there).
@pytest.mark.parametrize("score_fn,distance_fn,loss_fn,power",
                         [("TransE", "L2", "logsigmoid", p) for p in (-50, -28, -20, 20, 40, None)] +
                         [("TransE", "L2", "softmax", p) for p in (-50, -28, -20)] +
                         [("DistMult", "MatMul", "logsigmoid", p) for p in (-90, -50, -28, -20, 20, 40, None)] +
                         [("DistMult", "MatMul", "softmax", p) for p in (-90, -50, -28, -20, None)])
@pytest.mark.parametrize("B,A,D", [(70, 100, 64), (600, 520, 68)])
def test_rows_of_other_sizes(oracle64, score_fn, distance_fn, loss_fn, power, B, A, D):
    c = K.cfg_dict(score_fn=score_fn, distance_fn=distance_fn, loss_fn=loss_fn, n_shard=1, batch=B, a2a=A, dim=D, feature=0,
                   n_entity=2000, n_relation=B, gamma=4.0, shared_table=True)
    rng = np.random.default_rng(7)
    state = K.make_state(c, rng, warm=False, scale=0.25)
    sizes = np.full(B + A, 0.25)
    odd = [3, B + 37]
    if power is None:
        sizes = 0.25 * 2.0**rng.uniform(-60, 0, B + A)
        odd = np.arange(B)
        state["relation_embedding"] *= (4 * sizes[:B, None] if score_fn == "TransE" else 1)
    else:
        sizes[odd] *= 2.0**power
        if score_fn == "TransE":
            state["relation_embedding"][3] *= 2.0**power
    _assert_each_row(*_first_moments(c, state, _one_block(c, state, sizes, rng), B * A, oracle64))


# Softmax of scores that differ by tens of units from column to column: tails that no head gives a probability worth
# mentioning have gradients as right as the others'.  The scores come from one column, in steps that float32 holds.
@pytest.mark.parametrize("most", [12, 30, 60])
@pytest.mark.parametrize("B,A", [(70, 100), (600, 520)])
def test_columns_of_small_probabilities(oracle64, B, A, most):
    D = 64
    c = K.cfg_dict(score_fn="DistMult", distance_fn="MatMul", loss_fn="softmax", n_shard=1, batch=B, a2a=A, dim=D, feature=0,
                   n_entity=2000, n_relation=B, gamma=4.0, shared_table=True)
    rng = np.random.default_rng(7)
    state = K.make_state(c, rng, warm=False)
    batch = _one_block(c, state, np.full(B + A, 2.0**-9), rng)
    state["relation_embedding"][:] = 1.0
    state["entity_data"][1:1 + B, 0] = 1.0
    state["entity_data"][1 + B:1 + B + A, 0] = rng.integers(-4 * most, 1, A) / 4
    batch["tail"][:] = np.argmax(state["entity_data"][1 + B:1 + B + A, 0])
    _assert_each_row(*_first_moments(c, state, batch, B * A, oracle64))


# Slabs whose coefficients lie 2^50 and more apart, either way round
@pytest.mark.parametrize("powers", [(0, -50, -100), (-100, -50, 0), (-100, 0, -50)])
@pytest.mark.parametrize("side", ["tails", "heads"])
@pytest.mark.parametrize("loss_power", [0, 40])
def test_slabs_far_apart(oracle64, powers, side, loss_power):
    B, A, D = 96, 96, 64
    c = K.cfg_dict(score_fn="DistMult", distance_fn="MatMul", n_shard=1, batch=B, a2a=A, dim=D, feature=0, n_entity=300,
                   n_relation=B, gamma=4.0, shared_table=True)
    rng = np.random.default_rng(7)
    state = K.make_state(c, rng, warm=False, scale=0.25)
    sizes = np.full(B + A, 0.25)
    sizes[(B if side == "tails" else 0):][:96] *= np.repeat(2.0**np.array(powers), 32)
    batch = _one_block(c, state, sizes, rng)
    _assert_each_row(*_first_moments(c, state, batch, 2.0**loss_power, oracle64, **{"execution.merge_tails": False}))


# The product of very long rows with very short ones is of an ordinary size
@pytest.mark.parametrize("power", [-105, -90, -70, 70, 90, 105])
def test_dot_of_long_and_short_rows(oracle64, power):
    B, A, D = 70, 100, 64
    c = K.cfg_dict(score_fn="DistMult", distance_fn="MatMul", n_shard=1, batch=B, a2a=A, dim=D, feature=0, n_entity=300,
                   n_relation=B, gamma=4.0, shared_table=True)
    rng = np.random.default_rng(7)
    state = K.make_state(c, rng, warm=False, scale=0.25)
    batch = _one_block(c, state, np.repeat([2.0**power, 2.0**-power], [B, A]), rng)
    _assert_each_row(*_first_moments(c, state, batch, 1, oracle64))


# Columns much smaller than their rows' largest element, in every row or in one head and one tail: the gradients of such
# columns by their own norm, as the rows' above
@pytest.mark.parametrize("score_fn,distance_fn,loss_fn", [("TransE", "L2", "logsigmoid"), ("TransE", "L2", "softmax"),
                                                          ("DistMult", "MatMul", "logsigmoid"), ("DistMult", "MatMul", "softmax")])
@pytest.mark.parametrize("power", [-24, -30, -40, -60])
@pytest.mark.parametrize("every", [True, False])
@pytest.mark.parametrize("B,A,D", [(70, 100, 62), (200, 1024, 260)])
def test_columns_of_other_sizes(oracle64, score_fn, distance_fn, loss_fn, power, every, B, A, D):
    c = K.cfg_dict(score_fn=score_fn, distance_fn=distance_fn, loss_fn=loss_fn, n_shard=1, batch=B, a2a=A, dim=D, feature=0,
                   n_entity=2000, n_relation=B, gamma=4.0, shared_table=True)
    rng = np.random.default_rng(7)
    state = K.make_state(c, rng, warm=False, scale=0.25)
    batch = _one_block(c, state, np.full(B + A, 0.25), rng)
    columns = [1, 34, D - 1]
    rows = 1 + np.arange(B + A) if every else np.array([1 + 3, 1 + B + 37])
    state["entity_data"][rows[:, None], columns] *= 2.0**power
    if score_fn == "TransE":
        state["relation_embedding"][(np.arange(B) if every else np.array([3]))[:, None], columns] *= 2.0**power
    got, want = _first_moments(c, state, batch, B * A, oracle64)
    _assert_each_row(got, want)
    _assert_each_row(*[(l, e[:, columns].T, r[:, columns].T) for l, e, r in (got, want)])


# Merged tails: the slots behind a block's distinct ones repeat its first row.  That one has a column far below its largest
# element, the last distinct ones have none: what the repeated slots hold is multiplied by zeros
@pytest.mark.parametrize("score_fn,distance_fn,loss_fn", [("TransE", "L2", "logsigmoid"), ("TransE", "L2", "softmax"),
                                                          ("DistMult", "MatMul", "logsigmoid"), ("DistMult", "MatMul", "softmax")])
@pytest.mark.parametrize("live", [33, 71, 127])
def test_repeated_tails_behind_small_columns(oracle64, score_fn, distance_fn, loss_fn, live):
    B, A, D = 70, 300, 64
    c = K.cfg_dict(score_fn=score_fn, distance_fn=distance_fn, loss_fn=loss_fn, n_shard=1, batch=B, a2a=A, dim=D, feature=0,
                   n_entity=2000, n_relation=B, gamma=4.0, shared_table=True)
    rng = np.random.default_rng(7)
    state = K.make_state(c, rng, warm=False, scale=0.25)
    batch = _one_block(c, state, np.full(B + A, 0.25), rng)
    batch["a2a"][:] = B + np.arange(A, dtype=np.uint32) % live
    state["entity_data"][1 + B:1 + B + 32, 1] *= 2.0**-40
    state["entity_data"][1 + B:1 + B + 32, 34] *= 2.0**-40
    _assert_each_row(*_first_moments(c, state, batch, B * A, oracle64))


def _two_disjoint_blocks(kind, loss_fn, B, A, D, bad, merge):
    """One step of two blocks that share no row (entity or relation); `bad`: (role, value) of block 1's
    first head or tail, or None.  Returns the losses and block 0's rows afterwards."""
    import libpoplar_kge

    c = K.cfg_dict(score_fn="TransE" if kind != "MatMul" else "DistMult", distance_fn=kind, loss_fn=loss_fn, shared_table=True,
                   n_shard=2, batch=B, a2a=A, dim=D, feature=0, n_entity=2 * (B + 2 * A) + 1, n_relation=2 * B, gamma=4.0)
    rng = np.random.default_rng(3)
    state = K.make_state(c, rng)
    N = B + 2 * A
    remote = (1 + np.arange(2 * N, dtype=np.uint32)).reshape(2, 1, N)
    a2a = np.broadcast_to((B + np.arange(2 * A, dtype=np.uint32)).reshape(2, A), (2, 1, 2, A))
    batch = dict(remote=remote, a2a=a2a, head=np.broadcast_to(np.arange(B, dtype=np.uint32), (2, 1, B)),
                 relation=np.arange(2 * B, dtype=np.uint32).reshape(2, 1, B),
                 tail=rng.integers(0, 2 * A, (2, 1, B)).astype(np.uint32))
    if bad:
        state["entity_data"][remote[1, 0, 0] if bad[0] == "head" else remote[0, 0, B + A], min(3, D - 1)] = bad[1]
    engine = libpoplar_kge.Engine(H.engine_settings(c, 1, **{"execution.merge_tails": merge}), "")
    H.load_state(engine, c, state)
    loss = H.train(engine, c, 0.1, batch)
    after = H.read_state(engine, c)
    rows = np.concatenate([remote[0, 0, :B], remote[0, 0, B:B + A], remote[1, 0, B:B + A]])  # block 0's heads, its tails
    return loss, after["entity_data"][rows], after["relation_embedding"][:B]


# A block's last slab of 32 rows may reach into the next block's: nothing of that block may enter.
# (33, 42): both sides ragged, the head slab of block 0 reads block 1's heads, its tail slab block 1's tails
# (64, 42), (33, 64): one side whole
@pytest.mark.parametrize("kind", ["L2", "MatMul", "L1"])
@pytest.mark.parametrize("loss_fn,merge", [("logsigmoid", True), ("softmax", True), ("logsigmoid", False)])
@pytest.mark.parametrize("B,A,D", [(33, 21, 30), (64, 21, 64), (33, 32, 64), (1, 1, 2)])
def test_nonfinite_row_stays_in_its_block(kind, loss_fn, merge, B, A, D):
    clean = _two_disjoint_blocks(kind, loss_fn, B, A, D, None, merge)
    assert all(np.isfinite(x).all() for x in clean)
    for role in ("head", "tail"):
        for value in (np.inf, -np.inf, np.nan):
            got = _two_disjoint_blocks(kind, loss_fn, B, A, D, (role, value), merge)
            assert got[0][0] == clean[0][0]
            np.testing.assert_array_equal(got[1], clean[1])
            np.testing.assert_array_equal(got[2], clean[2])


# An infinite element must show in the block's loss (L2: distances to it are infinite, dot: products
# are; logsigmoid's sum holds 0 x infinity), and with whole columns that stand for no tail (repeats of the
# block's first tail) the gradients' other columns stay finite
@pytest.mark.parametrize("kind", ["L2", "MatMul"])
@pytest.mark.parametrize("B,A,D", [(33, 21, 30), (8, 100, 64), (130, 65, 100),
                                   (512, 512, 64)])  # whole tiles
def test_infinite_row_shows_in_the_loss(kind, B, A, D):
    for role in ("head", "tail"):
        for value in (np.inf, -np.inf):
            loss = _two_disjoint_blocks(kind, "logsigmoid", B, A, D, (role, value), True)[0]
            assert np.isfinite(loss[0]) and not np.isfinite(loss[1]), (role, value, loss)


def test_infinite_first_tail_keeps_to_its_column(oracle64):
    import libpoplar_kge

    S, B, A, D = 1, 20, 70, 24
    c = K.cfg_dict(score_fn="DistMult", distance_fn="MatMul", shared_table=True, n_shard=S, batch=B, a2a=A, dim=D, feature=0,
                   n_entity=100, n_relation=20, gamma=4.0)
    state = K.make_state(c, np.random.default_rng(3))
    remote = np.concatenate([np.arange(60, 60 + B), np.resize(np.arange(1, 11), A)]).astype(np.uint32).reshape(1, 1, B + A)
    batch = dict(remote=remote, a2a=(B + np.arange(A, dtype=np.uint32)).reshape(1, 1, 1, A),
                 head=np.arange(B, dtype=np.uint32).reshape(1, 1, B), relation=np.arange(B, dtype=np.uint32).reshape(1, 1, B),
                 tail=np.zeros((1, 1, B), np.uint32) + 3)
    state["entity_data"][1, 5] = np.inf  # ten distinct tails of 70: the columns behind them repeat row 1
    engine = libpoplar_kge.Engine(H.engine_settings(c, 1), "")
    H.load_state(engine, c, state)
    H.train(engine, c, 0.1, batch)
    heads = H.read_state(engine, c)["entity_data"][60:60 + B, :D]
    assert np.isfinite(np.delete(heads, 5, axis=1)).all()


class _ScoreShape(C.Structure):  # kge::ScoreShape, kge::RowSource
    _fields_ = ([(k, C.c_int) for k in ("S", "B", "T", "Dp", "score_fn", "dist_fn", "loss_fn")] +
                [(k, C.c_float) for k in ("gamma", "loss_scale", "softmax_correction", "negative_adversarial_scale")] +
                [("use_mfma", C.c_int), ("operands_dense", C.c_int), ("tcount", C.c_void_p), ("tmult", C.c_void_p),
                 ("tpad", C.c_int)])


class _RowSource(C.Structure):
    _fields_ = [("base", C.c_void_p), ("pitch", C.c_int64), ("etype", C.c_int), ("index", C.c_void_p), ("count", C.c_int),
                ("vec", C.c_int)]


# The parts of the loss that the fused L1 forward leaves are as many as score_fwd_parts says, whichever kernel
# takes the operands: prepared ones, or the table's rows with the relation still to be added.
@pytest.mark.parametrize("prepared", [True, False])
@pytest.mark.parametrize("S,B,T,D", [(2, 70, 100, 64), (1, 64, 32, 128)])
def test_l1_fused_forward_fills_its_parts(S, B, T, D, prepared):
    import torch

    rng = np.random.default_rng(3)
    rows = rng.normal(0, 0.3, (S * (B + T), D)).astype(np.float32)
    rel = rng.normal(0, 0.3, (5, D)).astype(np.float32)
    crel, label = rng.integers(0, 5, S * B).astype(np.int32), rng.integers(0, T, S * B).astype(np.int32)
    head = rows[:S * B].astype(np.float64) + (0 if prepared else rel[crel])
    dist = np.abs(head.reshape(S, B, 1, D) - rows[S * B:].reshape(S, 1, T, D)).sum(-1)
    score, positive = 4.0 - dist, label.reshape(S, B, 1) == np.arange(T)
    weight = np.where(positive, 0.5 * T, 0.5 * T / (T - 1))
    loss = np.mean(weight * np.logaddexp(0, np.where(positive, -score, score)))
    coef = np.where(positive, 1 / (1 + np.exp(score)), -1 / (1 + np.exp(-score))) * weight / (S * B * T)

    lib, dev = H.lib(), lambda a: torch.from_numpy(a).cuda()
    shape = _ScoreShape(S=S, B=B, T=T, Dp=D, score_fn=0, dist_fn=0, loss_fn=0, gamma=4.0, loss_scale=1.0, use_mfma=1,
                        operands_dense=int(prepared), tpad=64)
    table, drel, dcrel, dlabel = dev(rows), dev(rel), dev(crel), dev(label)
    source = _RowSource(base=table.data_ptr(), pitch=4 * D, etype=0, index=None, count=D, vec=1)
    n_part = lib._ZN3kge15score_fwd_partsERKNS_10ScoreShapeERKNS_9RowSourceE(C.byref(shape), C.byref(source))
    out, parts = torch.zeros(S, B, T, device="cuda"), torch.full((S * n_part + 256,), float("nan"), device="cuda")
    lib._ZN3kge16launch_score_fwdERKNS_10ScoreShapeERKNS_9RowSourceEPKfPKjS9_PfSA_PjSA_bP12ihipStream_t(
        C.byref(shape), C.byref(source), H.dptr(drel), H.dptr(dcrel), H.dptr(dlabel), H.dptr(out), None, None, H.dptr(parts),
        C.c_bool(True), None)
    torch.cuda.synchronize()
    parts = parts.cpu().numpy()
    assert np.isnan(parts[S * n_part:]).all()
    np.testing.assert_allclose(parts[:S * n_part].sum(dtype=np.float64), loss, rtol=1e-5)
    assert K.rel_l2(out.cpu().numpy(), coef) < 1e-5
