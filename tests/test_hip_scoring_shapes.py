"""The scoring kernels away from whole tiles, against the float64 oracle through the training step:
sizes around the edges of tiles and groups, one row, splits of a side over several workgroups."""

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


# L2 and dot on three-piece operands: tiles of 64 x 64 over slabs of 32, matrices filled up to 32
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
